"""Tile sorts where they can go wrong, bit for bit against the oracle: tiles
just within and above one workgroup's 2,048 instances, many segments, and
depths that defeat equal-width bins (all equal, a few values, one far surfel
stretching the range), at every tile size.
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


def _scene(P, depths, W=24, H=17, seed=0):
    """P small surfels facing the camera inside a 24 x 17 view, at given view depths."""
    rng = np.random.default_rng(seed)
    cam = look_at((0.0, 0.0, 0.0), target=(0.0, 0.0, 1.0), width=W, height=H)
    z = {"spread": rng.uniform(1, 3, P), "equal": np.full(P, 2.0), "few": rng.choice([1.5, 2.0, 2.5], P),
         "stretched": np.where(np.arange(P) == 0, 90.0, 2.0 + rng.uniform(0, 1e-4, P))}[depths]
    xy = rng.uniform(-0.5, 0.5, (P, 2)) * z[:, None]
    # the camera looks along +z with x mirrored or not; either way the depth is z
    means = np.concatenate([xy, z[:, None]], 1)
    q = np.tile([1.0, 0.0, 0.0, 0.0], (P, 1)) + rng.normal(size=(P, 4)) * 0.1
    scales = np.exp(rng.uniform(np.log(5e-3), np.log(3e-2), (P, 2)))
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).float()  # noqa: E731
    return SurfelScene(f(means), f(scales), f(q), f(rng.uniform(0.005, 0.05, (P, 1))), f(rng.normal(size=(P, 1, 3))),
                       0, cam, torch.ones(3))


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("P,depths", [(1300, "equal"), (2048, "spread"), (2049, "spread"), (2600, "few"),
                                      (7000, "equal"), (9000, "stretched"), (30_000, "spread"), (21_000, "few")])
def test_tile_sort(P, depths, tile):
    O.set_threads(8)
    scene = _scene(P, depths)
    o, rc = oracle_run(scene, tile=tile)
    assert rc == 0 and o.num_rendered >= P // 2
    res = gpu_forward(scene, tile=tile)
    _check_forward(scene, res, o)
    _check_backward(scene, res, o, seed=2)
