"""distCUDA2 at the sizes and inputs where its sort and box hierarchy can go
wrong, bit for bit against the brute-force oracle: around one leaf (16), one
wave (64), one node (1,024), one sorting workgroup (4,096) and one top box
(65,536 points); isolated points far from a dense cluster, equal points, and
coordinates that are not finite.
"""
import numpy as np
import pytest
import torch

from oracle import knn_oracle as K

pytestmark = pytest.mark.gpu


def _gpu(pts):
    from partgs_amd.knn import distCUDA2

    return distCUDA2(torch.from_numpy(np.ascontiguousarray(pts, np.float32)).cuda()).cpu().numpy()


@pytest.mark.parametrize("P", [2, 4, 15, 16, 17, 63, 64, 65, 129, 1023, 1024, 1025, 4095, 4096, 4097, 8193])
def test_sizes(P):
    pts = np.random.default_rng(P).normal(size=(P, 3)).astype(np.float32)
    np.testing.assert_array_equal(_gpu(pts), K.dist2_brute(pts))


@pytest.mark.parametrize("P", [65_535, 65_536, 65_537, 70_001])
def test_top_box_boundary(P):
    pts = np.random.default_rng(P).uniform(-1, 1, (P, 3)).astype(np.float32)
    np.testing.assert_array_equal(_gpu(pts), K.dist2_kdtree(pts))


def test_isolated_points_and_equal_points():
    rng = np.random.default_rng(5)
    dense = rng.normal(size=(6000, 3)) * 1e-3 + 0.25
    far = rng.normal(size=(40, 3)) * 50
    pts = np.concatenate([dense, far, np.full((200, 3), 0.125)]).astype(np.float32)
    np.testing.assert_array_equal(_gpu(pts), K.dist2_brute(pts))


def test_not_finite():
    pts = np.random.default_rng(6).normal(size=(700, 3)).astype(np.float32)
    pts[3, 0] = np.nan
    pts[77] = np.nan
    pts[130, 1] = np.inf
    pts[131, 2] = -np.inf
    with np.errstate(invalid="ignore", over="ignore"):
        want = K.dist2_brute(pts)
    np.testing.assert_array_equal(_gpu(pts), want)
