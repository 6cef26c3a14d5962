"""Bucket scatter at the edges of its surfel groups (256) and workgroups
(1,024), with the tiles counted in LDS and, above 4,096 tiles, by global
atomics: forward bit for bit and gradients against the oracle.
"""
import pytest

from oracle import oracle as O
from tests.helpers import gpu_forward, oracle_run
from tests.test_gpu_parity import _check_backward, _check_forward
from tests.test_gpu_tile_sort import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,tile", [(24, 17, 16), (605, 499, 8), (131, 67, 32)])
@pytest.mark.parametrize("P", [1, 255, 257, 1024, 1025, 2305])
def test_scatter(P, W, H, tile):
    O.set_threads(8)
    scene = _scene(P, "spread", W, H, seed=P)
    o, rc = oracle_run(scene, tile=tile)
    assert rc == 0
    res = gpu_forward(scene, tile=tile)
    _check_forward(scene, res, o)
    _check_backward(scene, res, o, seed=3)
