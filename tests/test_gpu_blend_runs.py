"""Runs of every pixel through the blend kernels at the lengths where their
batches (8 pairs), lanes (16, 32, 64 pairs) and segments (16 pairs, 257 pairs
and more) change, ending in the open, in the middle of a batch or after a few
pairs, against the oracle; and the path of quadrants that missed the pair
store, which must return the same bits.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from partgs_amd.camera import look_at
from partgs_amd.scenes import SurfelScene
from tests.helpers import gpu_backward, gpu_forward, oracle_run
from tests.test_gpu_parity import GRAD_TOL, _check_forward, upstream_grads

pytestmark = pytest.mark.gpu


def _stack(P, opacity, W=19, H=13):
    """P surfels behind each other, each over most of a 19 x 13 view."""
    rng = np.random.default_rng(P)
    cam = look_at((0.0, 0.0, 0.0), target=(0.0, 0.0, 1.0), width=W, height=H)
    z = rng.uniform(1.5, 4.0, P)
    means = np.concatenate([rng.uniform(-0.1, 0.1, (P, 2)) * z[:, None], z[:, None]], 1)
    q = np.tile([1.0, 0.0, 0.0, 0.0], (P, 1)) + rng.normal(size=(P, 4)) * 0.1
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).float()  # noqa: E731
    return SurfelScene(f(means), f(rng.uniform(0.8, 1.6, (P, 2)) * z[:, None]), f(q), f(np.full((P, 1), opacity)),
                       f(rng.normal(size=(P, 1, 3))), 0, cam, torch.ones(3))


@pytest.mark.parametrize("opacity", [0.006, 0.3, 0.95])
@pytest.mark.parametrize("P", [1, 7, 8, 9, 15, 16, 17, 31, 33, 63, 65, 128, 129, 255, 256, 257, 300, 513])
def test_run_lengths(P, opacity):
    O.set_threads(8)
    scene = _stack(P, opacity)
    o, rc = oracle_run(scene)
    assert rc == 0
    res = gpu_forward(scene)
    _check_forward(scene, res, o)
    H, W = scene.camera.image_height, scene.camera.image_width
    gc, go = upstream_grads(4, H, W)
    want = gpu_backward(res, gc, go)
    o64, _ = oracle_run(scene, f64=True)
    for x in (o, o64):
        x.backward(gc.numpy(), go.numpy())
    for k in want:
        exact = np.asarray(o64.get(k), np.float64)
        off = lambda a: np.abs(a.reshape(exact.shape) - exact) / (np.abs(exact) + np.abs(exact).max() + 1e-300)  # noqa: E731
        assert off(want[k]).max() <= off(np.asarray(o.get(k))).max() + GRAD_TOL, k
    missed = gpu_forward(scene, capacity=res["L"] + 64, pair_capacity=1)
    for k in ("color", "others", "radii"):
        assert torch.equal(missed[k], res[k]), k
    got = gpu_backward(missed, gc, go)
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)


def test_values_behind_a_saturated_pixel_do_not_reach_it():
    scene = _stack(20, 0.95)
    back = scene.means3D[:, 2].argsort()[10:]
    scene.shs[back[0]] = float("nan")
    scene.shs[back[1:]] = float("inf")
    res = gpu_forward(scene)
    missed = gpu_forward(scene, capacity=res["L"] + 64, pair_capacity=1)
    for k in ("color", "others"):
        assert torch.equal(missed[k], res[k]) and bool(torch.isfinite(res[k]).all()), k
