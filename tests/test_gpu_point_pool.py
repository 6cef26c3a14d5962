"""The fused pool at the edges of its groups of 64 points and of the workgroups'
shares, against the same layers one product at a time: the sums run in the same
order, so values and first argmax are equal bit for bit.  Inputs with equal
points (ties go to the first), all-negative channels (maximum 0 at point 0) and
NaN coordinates (ReLU makes them 0).
"""
import pytest
import torch

from partgs_amd import proposal as SP

pytestmark = pytest.mark.gpu


def _layers(net, pts):
    p, pb = net.p, net.pb
    X = pts.reshape(-1, 3)
    h1 = ((X[:, 0:1] * p["W1"][:, 0] + X[:, 1:2] * p["W1"][:, 1]) + X[:, 2:3] * p["W1"][:, 2]) + p["b1"]
    h1 = torch.where(h1 > 0, h1, torch.zeros_like(h1))
    _, h2 = SP.linear(SP.to_bf16(h1), pb["W2"], p["b2"], relu=True, want_bf16=True)
    h3 = SP.linear(h2, pb["W3"], p["b3"], relu=True).view(*pts.shape[:2], -1)
    best = h3.max(1).values
    return best, (h3 == best[:, None]).int().argmax(1)


@pytest.mark.parametrize("B,N", [(1, 1), (2, 15), (1, 64), (3, 65), (1, 127), (5, 130), (1, 33_000), (700, 70), (40, 900)])
@pytest.mark.parametrize("kind", ["random", "ties", "negative", "nan", "offset"])
def test_pool(B, N, kind):
    net = SP.ProposalNet(seed=3)
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + N)
    for b in ("b1", "b2", "b3"):
        net.p[b] = torch.randn(net.p[b].shape, generator=g, device="cuda") * 0.1
    pts = torch.randn(B, N, 3, generator=g, device="cuda")
    if kind == "ties":
        pts = pts[:, torch.randint(0, (N + 3) // 4, (N,), generator=g, device="cuda")].contiguous()
    if kind == "negative":
        net.p["b3"] = torch.where(torch.arange(256, device="cuda") % 3 == 0, -1e4, net.p["b3"])
    if kind == "nan":
        pts[:, ::3] = float("nan")
    if kind == "offset":  # weights at a 2-byte aligned place
        for k in ("W2", "W3"):
            w = torch.zeros(net.pb[k].numel() + 1, dtype=torch.int16, device="cuda")[1:].view(net.pb[k].shape)
            net.pb[k] = w.copy_(net.pb[k])
    val, idx = net.pool(pts)
    want, first = _layers(net, pts)
    assert torch.equal(val, want)
    assert torch.equal(idx.long(), first.long())
