"""Pair offsets of long lists: one wave's eight chunks and one more, one step of
the four waves and one more, several steps; pixels that never saturate and
pixels that do in the first chunks, in another wave's or between two steps.
Images bit for bit the oracle's; the quadrants' recomputing path, which does not
use the offsets, returns the same bits.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import gpu_backward, gpu_forward, oracle_run
from tests.test_gpu_blend_runs import _stack
from tests.test_gpu_parity import _check_forward, upstream_grads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opacity", [0.0045, 0.012, 0.3])
@pytest.mark.parametrize("P", [512, 513, 600, 2048, 2049, 2113, 4500])
def test_long_lists(P, opacity):
    O.set_threads(8)
    scene = _stack(P, opacity, 11, 9)
    o, rc = oracle_run(scene)
    assert rc == 0
    res = gpu_forward(scene)
    _check_forward(scene, res, o)
    missed = gpu_forward(scene, capacity=res["L"] + 64, pair_capacity=1)
    for k in ("color", "others"):
        assert torch.equal(missed[k], res[k]), k
    gc, go = upstream_grads(6, 9, 11)
    want, got = gpu_backward(res, gc, go), gpu_backward(missed, gc, go)
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
