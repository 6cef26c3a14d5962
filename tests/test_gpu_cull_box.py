"""Cull boxes: no accepted pixel may fall outside a surfel's box, or the image
would differ from the oracle, which looks at every pixel.  Scenes on both
sides of the rule that picks the tight margin (planes of a pixel parallel to
within 1%, depth varying by a quarter over the level set), at coordinates
from a small image to a strip thousands of pixels wide, with surfels from a
fraction of a pixel to hundreds of pixels; images, counts and gradients as in
test_gpu_parity.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from partgs_amd.camera import look_at
from partgs_amd.scenes import SurfelScene
from tests.helpers import gpu_forward, oracle_run
from tests.test_gpu_parity import _check_backward, _check_forward

pytestmark = pytest.mark.gpu


def _scene(W, H, grazing, close, size, P=4000, seed=0):
    rng = np.random.default_rng(seed)
    cam = look_at((0.0, 0.0, -3.0), width=W, height=H)
    means = rng.uniform(-1, 1, (P, 3)) * [1.5, 1.5, 1.0]
    if close:
        means[:, 2] = -3.0 + rng.uniform(0.25, 0.8, P)
        means[:, :2] *= 0.2
    view = means - np.array([0.0, 0.0, -3.0])
    view /= np.linalg.norm(view, axis=1, keepdims=True)
    side = np.cross(view, rng.normal(size=(P, 3)))
    side /= np.linalg.norm(side, axis=1, keepdims=True)
    lift = 10.0 ** rng.uniform(-4, 0, (P, 1)) if grazing else rng.uniform(0.2, 1.0, (P, 1))
    n = side + lift * view
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    q = np.concatenate([1 + n[:, 2:], -n[:, 1:2], n[:, 0:1], np.zeros((P, 1))], 1)
    q /= np.maximum(np.linalg.norm(q, axis=1, keepdims=True), 1e-9)
    scales = np.exp(rng.uniform(np.log(size[0]), np.log(size[1]), (P, 2)))
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).float()  # noqa: E731
    return SurfelScene(f(means), f(scales), f(q), f(rng.uniform(0.002, 1, (P, 1))), f(rng.normal(size=(P, 1, 3))), 0,
                       cam, torch.ones(3))


@pytest.mark.parametrize("W,H", [(97, 61), (4801, 33)])
@pytest.mark.parametrize("grazing,close,size", [(False, False, (1e-3, 1e-2)), (True, False, (1e-3, 5e-2)),
                                                (False, True, (1e-3, 0.3)), (True, True, (1e-4, 0.3))])
def test_no_accepted_pixel_outside(W, H, grazing, close, size):
    O.set_threads(8)
    scene = _scene(W, H, grazing, close, size)
    o, rc = oracle_run(scene)
    assert rc == 0
    res = gpu_forward(scene)
    _check_forward(scene, res, o)
    _check_backward(scene, res, o, seed=1)


@pytest.mark.parametrize("P", [1, 300, 2000])
def test_faint_surfels_whose_three_sigma_conic_nearly_reaches_the_camera(P):
    """mean2D, the centre of the 3 sigma conic's box, then lies anywhere; the
    level set of a faint surfel is a small ellipse about its own centre."""
    O.set_threads(8)
    W, H = 53, 37
    rng = np.random.default_rng(P)
    cam = look_at((0.0, 0.0, 0.0), target=(0.0, 0.0, 1.0), width=W, height=H)
    z = rng.uniform(0.5, 5.0, P)
    means = np.concatenate([rng.uniform(-0.3, 0.3, (P, 2)) * z[:, None], z[:, None]], 1)
    tilt, turn = rng.uniform(0.2, 1.2, P), rng.uniform(0, 2 * np.pi, P)
    # about an axis of the image plane by tilt: the depths of the tangents are
    # sin(tilt) times their scales across the axis, so 9 (Tw.x^2 + Tw.y^2) is
    # near Tw.z^2 for scales of z / (3 sin(tilt))
    q = np.stack([np.cos(tilt / 2), np.sin(tilt / 2) * np.cos(turn), np.sin(tilt / 2) * np.sin(turn), np.zeros(P)], 1)
    s = z / (3 * np.sin(tilt)) * np.sqrt(1 + rng.choice([-1.0, 1.0], P) * 10.0 ** rng.uniform(-5, -1, P))
    opacity = np.exp(rng.uniform(0, 0.5, (P, 1))) / 255
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).float()  # noqa: E731
    scene = SurfelScene(f(means), f(np.stack([s, s], 1)), f(q), f(opacity), f(rng.normal(size=(P, 1, 3))), 0, cam,
                        torch.ones(3))
    o, rc = oracle_run(scene)
    assert rc == 0
    _check_forward(scene, gpu_forward(scene), o)
