"""Backward preprocess of several views at the edges of its waves and of its
SH layouts (rows through LDS or not, inactive coefficients, no SHs), one view
seeing nothing: the gradients equal the single views' sums.

Tolerance: the sums differ in order only, at most three views and a handful of
terms each, (n + 1) 2^-24 of the sum of magnitudes: 1e-5 of the largest, as the
other batch tests.
"""
import math

import pytest
import torch

from helpers import assert_close_scaled
from partgs_amd.batch import BatchRasterizer
from partgs_amd.camera import look_at, random_sphere_camera
from partgs_amd.rasterizer import rasterize_gaussians_bwd, rasterize_gaussians_fwd
from partgs_amd.scenes import surfel_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coeffs,degree,layout", [(16, 3, "rows"), (16, 1, "rows"), (16, 3, "offset"), (16, 2, "offset"),
                                                  (9, 2, "plain"), (4, 0, "plain"), (0, 0, "colours")])
@pytest.mark.parametrize("P", [1, 63, 65, 257])
def test_sums_of_single_views(P, coeffs, degree, layout):
    s = surfel_cloud(P, P=P, width=40, height=30).to("cuda")
    s.scales = s.scales * 8
    cams = [random_sphere_camera(k, 3.0, w, h).to("cuda") for k, (w, h) in enumerate([(40, 30), (33, 47)])]
    cams.insert(1, look_at((0.0, 0.0, 9.0), target=(0.0, 0.0, 20.0), width=24, height=16).to("cuda"))
    g = torch.Generator().manual_seed(P)
    e = torch.empty(0, device="cuda")
    sh, col = e, torch.rand(P, 3, generator=g).cuda()
    if coeffs:
        flat = torch.randn(P * coeffs * 3 + 1, generator=g).cuda()
        sh, col = flat[int(layout == "offset"):][:P * coeffs * 3].view(P, coeffs, 3), e
    br = BatchRasterizer(cams, s.bg, degree)
    opt = lambda t: t if t.numel() else None  # noqa: E731
    args = (s.means3D, opt(sh), opt(col), s.opacities, s.scales, s.rotations)
    _, _, radii = br.forward_checked(*args)
    gcs = [torch.randn(3, c.image_height, c.image_width, generator=g).cuda() for c in cams]
    gos = [torch.randn(7, c.image_height, c.image_width, generator=g).cuda() for c in cams]
    grads = br.new_grads(P, coeffs)
    for t in grads.values():
        if t is not None:
            t.fill_(float("nan"))  # every entry is written
    br.backward_raw(*args, radii, br.pack(gcs, 3), br.pack(gos, 7), grads)
    acc = {}
    for v, cam in enumerate(cams):
        view = (cam.world_view_transform, cam.full_proj_transform, math.tan(cam.FoVx / 2), math.tan(cam.FoVy / 2))
        size = (cam.image_height, cam.image_width)
        L, _, _, rad, geom, binb, img = rasterize_gaussians_fwd(
            s.bg, s.means3D, col, s.opacities, s.scales, s.rotations, 1.0, e, *view, *size, sh, degree,
            cam.camera_center, False, False)
        assert torch.equal(rad, radii[v])
        assert v != 1 or L == 0
        o = rasterize_gaussians_bwd(s.bg, s.means3D, rad, col, s.scales, s.rotations, 1.0, e, *view, gcs[v], gos[v],
                                    sh, degree, cam.camera_center, geom, L, binb, img, False)
        assert_close_scaled(grads["means2D"][v].cpu().numpy(), o[0].cpu().numpy(), 1e-5, f"means2D {v}")
        for k, i in (("colors", 1), ("opacities", 2), ("means3D", 3), ("shs", 5), ("scales", 6), ("rotations", 7)):
            acc[k] = acc.get(k, 0) + o[i].double()
    for k, t in acc.items():
        if k != "shs" or coeffs:
            assert_close_scaled(grads[k].cpu().numpy().reshape(t.shape), t.cpu().numpy(), 1e-5, k)
