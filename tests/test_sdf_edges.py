"""The superquadric distance and its adjoint at the sizes where the split of
points over lanes changes (one workgroup is 256 points; a lane takes
B ceil(N / 256) / 2048 points, between 1 and 8), against FP64 torch.

Bars.  The distance: every power is within 1 ulp, and the three nested ones
and the final subtraction leave |error| <= 1e-6 (1 + |sdf| + 1); the
existing bar of 1e-5 covers it.  A parameter's gradient is an FP32 sum of N
terms in chains of at most 8 + 8 + ceil(chunks / 15) + 15 additions, each
term good to about 2e-6 relative through its ten powers: 2e-5 of the sum of
the terms' magnitudes bounds both.
"""
import pytest
import torch

from partgs_amd.block_fit import random_block_params

pytestmark = pytest.mark.gpu


def _sdf64(params, pts):
    S = torch.exp(params[:, 0:3]) + 0.2
    q = params[:, 3:7] / params[:, 3:7].norm(dim=1, keepdim=True)
    w, x, y, z = q.unbind(-1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).view(-1, 3, 3)
    e = torch.sigmoid(params[:, 10:12]) * 1.8 + 0.1
    e1, e2 = e[:, 0:1], e[:, 1:2]
    p = torch.einsum("bnj,bkj->bnk", pts[None] - params[:, None, 7:10], R) / (S[:, None] * 0.25)
    p = p.clamp(-5.0, 5.0)
    power = lambda t, a: t.clamp_min(1e-6).pow(a)  # noqa: E731
    a, b, c = power(p[..., 0] ** 2, 1 / e2), power(p[..., 1] ** 2, 1 / e1), power(p[..., 2] ** 2, 1 / e2)
    return power(power(a + c, e2 / e1) + b, e1 / 2) - 1.0


@pytest.mark.parametrize("B,N", [(1, 1), (3, 255), (1, 256), (2, 257), (16, 65_535), (16, 65_537), (24, 180_001)])
def test_sdf_sizes(B, N):
    import numpy as np

    from partgs_amd.block_losses import superquadric_sdf

    params = torch.from_numpy(random_block_params(np.random.default_rng(B * 7 + N), B)).cuda().requires_grad_(True)
    gen = torch.Generator(device="cuda").manual_seed(N)
    pts = torch.rand(N, 3, device="cuda", generator=gen) * 2 - 1
    g = torch.randn(B, N, device="cuda", generator=gen)
    sdf = superquadric_sdf(params, pts)
    sdf.backward(g)
    p64, x64 = params.detach().double(), pts.double()
    want = _sdf64(p64, x64)
    assert ((sdf.detach().double() - want).abs() <= 1e-5 * (1 + want.abs())).all()
    for k in range(12):
        d = torch.zeros_like(p64)
        d[:, k] = 1.0
        terms = torch.func.jvp(lambda p: _sdf64(p, x64), (p64,), (d,))[1] * g.double()
        err = (params.grad[:, k].double() - terms.sum(1)).abs()
        assert (err <= 2e-5 * terms.abs().sum(1)).all(), (k, err, terms.abs().sum(1))
