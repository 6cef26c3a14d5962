"""The _part variant through the accepted-pair store: semantic channel counts
at the edges of the kernels' widths (1, 4 | 5, 8 | 9, 16), ragged images and
every tile size, against the oracle; and the path that recomputes a
quadrant's pairs when they miss the store, which must return the same bits.

Bars as in test_gpu_part: images bit-exact, gradients within 1e-5.
"""
import pytest
import torch

from oracle import oracle as O
from partgs_amd import rasterizer_part as RP
from partgs_amd.scenes import superquadric_surfels, surfel_cloud
from tests.test_gpu_part import GRAD_NAMES, _check, _gpu_forward, _semantics, _upstream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,W,H,tile", [(1, 61, 47, 16), (4, 64, 33, 8), (8, 33, 64, 32), (9, 57, 40, 16)])
def test_part_channel_widths(S, W, H, tile):
    O.set_threads(8)
    scene = surfel_cloud(3, P=3000, width=W, height=H)
    _check(scene, _semantics(3000, S), tile=tile)


def _backward(res, S, H, W, **caps):
    a = res["args"]
    up = [t.cuda() for t in _upstream(S, H, W)]
    out = RP.rasterize_gaussians_bwd(
        a["bg"], a["means3D"], res["radii"], a["colors"], a["semantics"], a["scales"], a["rotations"],
        a["scale_modifier"], a["transMat_precomp"], a["viewmatrix"], a["projmatrix"], a["tan_fovx"], a["tan_fovy"],
        *up, a["sh"], a["degree"], a["campos"], res["geom"], res["L"], res["bin"], res["img"], False, 16, **caps)
    return dict(zip(GRAD_NAMES, out))


@pytest.mark.parametrize("S", [0, 1, 8, 16])
def test_part_recomputed_pairs_same_bits(S):
    W, H = 123, 77
    scene = superquadric_surfels(1, P=20_000, width=W, height=H, sh_degree=1)
    res = _gpu_forward(scene, _semantics(scene.P, S))
    want = _backward(res, S, H, W)
    # no pair fits; about half of them fit
    for pairs in (1, 4 * res["L"]):
        caps = dict(capacity=res["L"] + 64, pair_capacity=pairs)
        out = RP.rasterize_gaussians_fwd(**res["args"], **caps)
        got = dict(zip(("L", "color", "semantic", "others", "radii", "geom", "bin", "img"), out), args=res["args"])
        for k in ("color", "semantic", "others", "radii"):
            assert torch.equal(got[k], res[k]), (pairs, k)
        grads = _backward(got, S, H, W, **caps)
        for k, g in want.items():
            assert torch.equal(grads[k], g), (pairs, k)
