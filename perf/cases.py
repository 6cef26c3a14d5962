"""The workloads this framework's speed is judged by, as calls a user's program makes.

Each case is a dict of plain values; ``prepare`` builds the inputs (on the
GPU, from the seed alone), ``run`` makes one pass through the public entry
points, ``work`` says what the pass cannot do without and ``exact`` gives the
same outputs in 64 bits from plain torch.

Kinds:

* ``raster``   GaussianRasterizer, forward and backward: a training step's view.
  ``shape`` "cloud" is the uniform cloud of the 16,384-surfel configuration,
  "surface" surfels on 8 random superquadrics (300,000 and 1,000,000 in the
  configurations).  ``coeffs`` SH coefficients are stored, ``degree`` is the
  active degree (training starts at 0 and raises it).
* ``render``   render() under no_grad: an evaluation view with its maps.
* ``part``     the part-aware rasteriser (semantic channels), forward and backward.
* ``batch``    a captured training step over many views (capture_grouped_step).
* ``blocks``   block parameters -> surfels -> one view -> block gradients.
* ``fit``      one iteration of the block fitter's image term over all views.
* ``sdf``      superquadric distances and their adjoint (the ray losses).
* ``knn``      distCUDA2 of an initial point cloud.
* ``proposal`` the block-proposal network, forward and backward.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

DEV = "cuda"
SH_C0 = 0.28209479177387814


def listed():
    return [
        # the smallest training view: launches and host time count
        dict(name="raster_16k_256", kind="raster", shape="cloud", P=16384, W=256, H=256, coeffs=1, degree=0),
        # half-resolution training view, image smaller than the surfel count
        dict(name="raster_300k_400x300", kind="raster", shape="surface", P=300_000, W=400, H=300, coeffs=16,
             degree=3),
        # the headline training view
        dict(name="raster_300k_800x600", kind="raster", shape="surface", P=300_000, W=800, H=600, coeffs=16,
             degree=3),
        # a large scene at an odd, larger resolution
        dict(name="raster_1m_1237x823", kind="raster", shape="surface", P=1_000_000, W=1237, H=823, coeffs=16,
             degree=3),
        # evaluation: forward only, with the depth and normal maps render() derives
        dict(name="render_300k_799x601", kind="render", shape="surface", P=300_000, W=799, H=601, coeffs=16,
             degree=3),
        # part-aware training view with 8 semantic channels
        dict(name="part_300k_800x600", kind="part", shape="surface", P=300_000, W=800, H=600, coeffs=16, degree=3,
             channels=8),
        # 32 ragged views of a million surfels in one captured step
        dict(name="batch_1m_32views", kind="batch", P=1_000_000, views=32, groups=2),
        # block stage at full sampling: 65,536 surfels attached to 16 blocks
        dict(name="blocks_16x64x64", kind="blocks", B=16, n=64, W=400, H=300),
        # an iteration of the block fitter: small images, small launches
        dict(name="fit_16x24x24_6views", kind="fit", B=16, n=24, views=6, W=128, H=96),
        # the ray losses' samples against every block
        dict(name="sdf_16x262144", kind="sdf", B=16, N=2048 * 128),
        # scales of a large initial point cloud
        dict(name="knn_1m", kind="knn", P=1_000_000),
        # a training batch of the proposal network
        dict(name="proposal_32x20000", kind="proposal", scenes=32, N=20_000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["raster"] * 6 + ["render", "part", "part", "batch", "blocks", "fit", "sdf", "knn", "knn",
                       "proposal"])
    if kind in ("raster", "render", "part"):
        W = _log_int(rng, 160, 1300)
        H = max(90, int(W * rng.uniform(0.6, 1.0)))
        case = dict(kind=kind, shape="surface", P=_log_int(rng, 5_000, 1_000_000), W=W, H=H)
        if rng.random() < 0.25:  # fewer, larger surfels filling the frame
            case.update(shape="cloud", P=min(case["P"], _log_int(rng, 2_000, 40_000)))
        case["coeffs"], case["degree"] = rng.choice([(16, 3), (16, 3), (16, 0), (16, 1), (16, 2), (1, 0), (4, 1),
                                                     (9, 2)])
        if kind == "part":
            case["channels"] = rng.randint(1, 16)
        return case
    if kind == "batch":
        views = rng.randint(2, 12)
        return dict(kind=kind, P=_log_int(rng, 30_000, 400_000), views=views, groups=rng.randint(1, 2))
    if kind == "blocks":
        W = _log_int(rng, 160, 800)
        return dict(kind=kind, B=rng.randint(2, 24), n=_log_int(rng, 12, 80), W=W, H=int(W * rng.uniform(0.6, 1.0)))
    if kind == "fit":
        W = _log_int(rng, 80, 320)
        return dict(kind=kind, B=rng.randint(4, 16), n=_log_int(rng, 12, 48), views=rng.randint(2, 8), W=W,
                    H=int(W * rng.uniform(0.6, 1.0)))
    if kind == "sdf":
        return dict(kind=kind, B=rng.randint(1, 24), N=_log_int(rng, 2_000, 400_000))
    if kind == "knn":
        return dict(kind=kind, P=_log_int(rng, 1_000, 1_000_000))
    return dict(kind=kind, scenes=_log_int(rng, 1, 48), N=_log_int(rng, 1_000, 20_000))


# ---- inputs ---------------------------------------------------------------------------
def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 16 + salt)


def _quat(g, n):
    q = _randn(g, n, 4)
    return q / q.norm(dim=1, keepdim=True)


def _rotation(q):
    """Columns-as-axes rotation matrices of (w, x, y, z) quaternions, N x 3 x 3."""
    w, x, y, z = q.unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).view(-1, 3, 3)


def _spow(t, e):
    return torch.sign(t) * t.abs().pow(e)


def _surface_points(g, P, blocks=8):
    """Points and unit normals on the surfaces of random superquadrics."""
    k = torch.arange(P, device=DEV) % blocks
    e = (0.1 + 1.8 * _rand(g, blocks, 2))[k]
    ax = (0.1 + 0.4 * _rand(g, blocks, 3))[k]
    R = _rotation(_quat(g, blocks))[k]
    c = _randn(g, blocks, 3)
    c = (c / c.norm(dim=1, keepdim=True) * _rand(g, blocks, 1).pow(1 / 3))[k]
    eta = (_rand(g, P) - 0.5) * math.pi
    om = (_rand(g, P) - 0.5) * 2 * math.pi
    ce, se, co, so = eta.cos(), eta.sin(), om.cos(), om.sin()
    p = torch.stack([_spow(ce, e[:, 0]) * _spow(so, e[:, 1]), _spow(se, e[:, 0]),
                     _spow(ce, e[:, 0]) * _spow(co, e[:, 1])], 1) * ax
    n = torch.stack([_spow(ce, 2 - e[:, 0]) * _spow(so, 2 - e[:, 1]), _spow(se, 2 - e[:, 0]),
                     _spow(ce, 2 - e[:, 0]) * _spow(co, 2 - e[:, 1])], 1) / ax
    n = (R @ n[:, :, None])[:, :, 0]
    return (R @ p[:, :, None])[:, :, 0] + c, n / n.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _normal_quat(n, spin):
    """Quaternions whose rotation takes z to n, after a spin about z."""
    w = 1 + n[:, 2:3]
    q = torch.cat([w, -n[:, 1:2], n[:, 0:1], torch.zeros_like(w)], 1)
    q = torch.where(w > 1e-6, q, torch.tensor([0.0, 1.0, 0.0, 0.0], device=DEV, dtype=q.dtype))
    q = q / q.norm(dim=1, keepdim=True)
    c, s = spin.cos(), spin.sin()
    a, b, cc, d = q.unbind(1)
    return torch.stack([a * c - d * s, b * c + cc * s, cc * c - b * s, a * s + d * c], 1)


def _camera(seed, W, H):
    """Camera on the radius-3 sphere looking at the origin, 60 degrees."""
    rng = np.random.default_rng(seed)
    pos = rng.normal(size=3)
    pos *= 3.0 / np.linalg.norm(pos)
    f = -pos / np.linalg.norm(pos)
    up = np.array([0.0, 1.0, 0.0]) if abs(f[1]) < 0.99 else np.array([0.0, 0.0, 1.0])
    r = np.cross(f, up)
    r /= np.linalg.norm(r)
    rot = np.stack([r, np.cross(f, r), f])
    w2c = np.eye(4)
    w2c[:3, :3], w2c[:3, 3] = rot, -rot @ pos
    fov, near, far = math.radians(60.0), 0.01, 100.0
    proj = np.zeros((4, 4))
    proj[0, 0] = proj[1, 1] = 1.0 / math.tan(fov / 2)
    proj[2, 2], proj[2, 3], proj[3, 2] = far / (far - near), -far * near / (far - near), 1.0
    t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float32, device=DEV)  # noqa: E731
    return SimpleNamespace(image_width=W, image_height=H, FoVx=fov, FoVy=fov, znear=near, zfar=far,
                           world_view_transform=t(w2c.T), projection_matrix=t(proj.T),
                           full_proj_transform=t(w2c.T @ proj.T), camera_center=t(pos))


def _scene(case, seed):
    """Surfels as the rasteriser takes them (FP32)."""
    g = _gen(seed)
    P = case["P"]
    if case.get("shape") == "cloud":
        means, q = _rand(g, P, 3) * 2 - 1, _quat(g, P)
        lo, hi = 1e-3, 5e-2
    else:
        means, n = _surface_points(g, P)
        q = _normal_quat(n, _rand(g, P) * math.pi)
        lo, hi = 1e-3, 1e-2
    scales = torch.exp(_rand(g, P, 2) * math.log(hi / lo) + math.log(lo))
    opac = torch.sigmoid(_randn(g, P, 1))
    M = case.get("coeffs", 16)
    shs = torch.randn(P, M, 3, generator=g, device=DEV) * 0.05
    shs[:, 0] = ((_rand(g, P, 3) - 0.5) / SH_C0).float()
    return dict(means3D=means.float(), shs=shs, opacities=opac.float(), scales=scales.float(), rotations=q.float())


def _upstream(seed, *shape):
    return torch.randn(*shape, generator=_gen(seed, 1), device=DEV)


def _settings(cls, cam, bg, degree):
    return cls(image_height=cam.image_height, image_width=cam.image_width, tanfovx=math.tan(cam.FoVx * 0.5),
               tanfovy=math.tan(cam.FoVy * 0.5), bg=bg, scale_modifier=1.0, viewmatrix=cam.world_view_transform,
               projmatrix=cam.full_proj_transform, sh_degree=degree, campos=cam.camera_center, prefiltered=False,
               debug=False)


def _batch_cameras(case, seed):
    sizes = ((640, 480), (400, 300), (800, 600))
    return [_camera(seed * 64 + v, *sizes[v % 3]) for v in range(case["views"])]


def _blocks(g, B):
    """B x 12 block parameters (log scales, quaternion, translation, epsilon logits), logits, colours."""
    s = torch.log(0.1 + 0.4 * _rand(g, B, 3))
    t = _randn(g, B, 3)
    t = t / t.norm(dim=1, keepdim=True) * _rand(g, B, 1).pow(1 / 3)
    u = (0.1 + 1.6 * _rand(g, B, 2)) / 1.8
    params = torch.cat([s, _quat(g, B), t, torch.log(u / (1 - u))], 1).float()
    return params, _randn(g, B).float(), (0.15 + 0.8 * _rand(g, B, 3)).float()


PIPE = SimpleNamespace(compute_cov3D_python=False, depth_ratio=1.0)


def prepare(case, seed):
    kind = case["kind"]
    st = SimpleNamespace(kind=kind)
    if kind in ("raster", "render", "part"):
        sc = _scene(case, seed)
        st.bg = torch.ones(3, device=DEV)
        st.cam = _camera(seed, case["W"], case["H"])
        H, W = case["H"], case["W"]
        if kind == "render":
            st.pc = SimpleNamespace(get_xyz=sc["means3D"], get_opacity=sc["opacities"], get_scaling=sc["scales"],
                                    get_rotation=sc["rotations"], get_features=sc["shs"],
                                    active_sh_degree=case["degree"])
            return st
        st.leaves = {k: v.requires_grad_(True) for k, v in sc.items()}
        st.means2D = torch.zeros_like(sc["means3D"], requires_grad=True)
        if kind == "raster":
            from partgs_amd.rasterizer import GaussianRasterizationSettings, GaussianRasterizer
            st.grads = (_upstream(seed, 3, H, W), _upstream(seed + 1, 7, H, W))
        else:
            from partgs_amd.rasterizer_part import GaussianRasterizationSettings, GaussianRasterizer
            S = case["channels"]
            st.leaves["semantics"] = torch.rand(case["P"], S, generator=_gen(seed, 2),
                                                device=DEV).requires_grad_(True)
            st.grads = (_upstream(seed, 3, H, W), _upstream(seed + 1, S, H, W), _upstream(seed + 2, 8, H, W))
        st.rast = GaussianRasterizer(_settings(GaussianRasterizationSettings, st.cam, st.bg, case["degree"]))
    elif kind == "batch":
        from partgs_amd.batch import ViewGroups, capture_grouped_step
        sc = _scene(case, seed)
        st.vg = ViewGroups(_batch_cameras(case, seed), torch.ones(3, device=DEV), 3, groups=case["groups"])
        st.step = capture_grouped_step(st.vg, sc["means3D"], sc["shs"], None, sc["opacities"], sc["scales"],
                                       sc["rotations"], _upstream(seed, 3 * st.vg.N), _upstream(seed + 1, 7 * st.vg.N))
        st.inputs = sc
    elif kind in ("blocks", "fit"):
        from partgs_amd.blocks import make_grid
        st.leaves = [t.requires_grad_(True) for t in _blocks(_gen(seed), case["B"])]
        st.grid = make_grid(case["n"], case["n"], device=DEV)
        st.bg = torch.ones(3, device=DEV)
        W, H = case["W"], case["H"]
        if kind == "blocks":
            from partgs_amd.rasterizer import GaussianRasterizationSettings, GaussianRasterizer
            st.cam = _camera(seed, W, H)
            st.rast = GaussianRasterizer(_settings(GaussianRasterizationSettings, st.cam, st.bg, 0))
            st.grads = (_upstream(seed, 3, H, W), _upstream(seed + 1, 7, H, W))
        else:
            from partgs_amd.batch import BatchConfig, BatchRasterizer
            cams = [_camera(seed * 64 + v, W, H) for v in range(case["views"])]
            st.br = BatchRasterizer(cams, st.bg, 0, BatchConfig(tile=16))
            st.grads = _upstream(seed, case["views"] * 3 * H * W)
    elif kind == "sdf":
        st.params = _blocks(_gen(seed), case["B"])[0].requires_grad_(True)
        st.points = (_rand(_gen(seed, 3), case["N"], 3) * 2 - 1).float()
        st.grads = _upstream(seed, case["B"], case["N"])
    elif kind == "knn":
        st.points = _surface_points(_gen(seed), case["P"])[0].float()
    else:
        from partgs_amd.proposal import ProposalNet
        st.net = ProposalNet(seed=seed & 0xFFFF, device=DEV)
        st.points = _proposal_points(case, seed)
        st.grads = _upstream(seed, case["scenes"], 16, 12)
    return st


def _proposal_points(case, seed):
    g = _gen(seed)
    pts = torch.stack([_surface_points(g, case["N"])[0] for _ in range(case["scenes"])])
    return (pts + 0.005 * _randn(g, *pts.shape)).float()


def _fresh(leaves):
    for t in leaves:
        t.grad = None


def run(st):
    if st.kind == "raster":
        _fresh([st.means2D, *st.leaves.values()])
        color, radii, allmap = st.rast(means2D=st.means2D, **st.leaves)
        torch.autograd.backward((color, allmap), st.grads)
        return dict(color=color.detach(), allmap=allmap.detach(), radii=radii, means2D=st.means2D.grad,
                    **{"d_" + k: t.grad for k, t in st.leaves.items()})
    if st.kind == "render":
        from partgs_amd.renderer import render
        with torch.no_grad():
            out = render(st.cam, st.pc, PIPE, st.bg)
        return {k: out[k] for k in ("render", "radii", "rend_alpha", "rend_normal", "rend_dist", "surf_depth",
                                    "surf_normal")}
    if st.kind == "part":
        _fresh([st.means2D, *st.leaves.values()])
        color, semantic, radii, allmap = st.rast(means2D=st.means2D, **st.leaves)
        torch.autograd.backward((color, semantic, allmap), st.grads)
        return dict(color=color.detach(), semantic=semantic.detach(), allmap=allmap.detach(), radii=radii,
                    means2D=st.means2D.grad, **{"d_" + k: t.grad for k, t in st.leaves.items()})
    if st.kind == "batch":
        st.step.replay()
        color, others, radii = st.step.outputs
        return dict(color=color, others=others, radii=radii,
                    **{"d_" + k: v for k, v in st.step.grads.items() if k != "colors"})
    if st.kind == "blocks":
        from partgs_amd.blocks import generate_surfels
        _fresh(st.leaves)
        params, occ, colors = st.leaves
        means, scales, rots, opac = generate_surfels(params, occ, st.grid)
        col = colors.repeat_interleave(st.grid.surfels_per_block(), dim=0)
        color, radii, allmap = st.rast(means3D=means, means2D=torch.zeros_like(means), opacities=opac,
                                       colors_precomp=col, scales=scales, rotations=rots)
        torch.autograd.backward((color, allmap), st.grads)
        return dict(color=color.detach(), allmap=allmap.detach(), radii=radii, d_params=params.grad, d_occ=occ.grad,
                    d_colors=colors.grad)
    if st.kind == "fit":
        from partgs_amd.block_fit import render_blocks
        _fresh(st.leaves)
        image = render_blocks(st.br, *st.leaves, st.grid)
        image.backward(st.grads)
        return dict(image=image.detach(), **dict(zip(("d_params", "d_occ", "d_colors"), [t.grad for t in st.leaves])))
    if st.kind == "sdf":
        from partgs_amd.block_losses import superquadric_sdf
        st.params.grad = None
        sdf = superquadric_sdf(st.params, st.points)
        sdf.backward(st.grads)
        return dict(sdf=sdf.detach(), d_params=st.params.grad)
    if st.kind == "knn":
        from partgs_amd.knn import distCUDA2
        return distCUDA2(st.points)
    out, cache = st.net.forward(st.points)
    return dict(out=out, **{"d_" + k: v for k, v in st.net.backward(st.grads, cache).items()})


# ---- what a pass cannot do without -------------------------------------------------------
def work(case):
    """Inputs read once and outputs written once; operations only where the path is a fixed count of them."""
    kind = case["kind"]
    if kind in ("raster", "render", "part"):
        P, N, M, S = case["P"], case["W"] * case["H"], case["coeffs"], case.get("channels", 0)
        surfel, maps = 10 + 3 * M + S, (18 if kind == "part" else 10) + S
        if kind == "render":
            return dict(bytes=4.0 * (P * (surfel + 1) + N * 13), flops=0.0)
        return dict(bytes=4.0 * (P * (2 * surfel + 4) + N * 2 * maps), flops=0.0)
    if kind == "batch":
        P, V, N = case["P"], case["views"], case["views"] * 297_000
        return dict(bytes=4.0 * (P * (2 * 58 + 4 * V) + N * 20), flops=0.0)
    if kind in ("blocks", "fit"):
        # the surfels between the block layer and the rasteriser pass through memory both ways
        P, N = case["B"] * case["n"] ** 2, case["W"] * case["H"] * case.get("views", 1)
        return dict(bytes=4.0 * (4 * P * 13 + N * (20 if kind == "blocks" else 6)), flops=0.0)
    if kind == "sdf":
        B, N = case["B"], case["N"]
        return dict(bytes=4.0 * (2 * B * N + 6 * N), flops=150.0 * B * N)
    if kind == "knn":
        return dict(bytes=16.0 * case["P"], flops=0.0)
    B, N = case["scenes"], case["N"]
    per_point = 2.0 * (3 * 64 + 64 * 128 + 128 * 256)
    return dict(bytes=12.0 * B * N + 4.0 * 3 * 90_000, flops=B * N * per_point + 3 * B * 256 * per_point)


# ---- the same outputs in 64 bits -----------------------------------------------------------
def _sh_color(sh, degree, d):
    """View-dependent colour of SH coefficients (P x M x 3) along unit directions d."""
    x, y, z = (d[:, i:i + 1] for i in range(3))
    xx, yy, zz = x * x, y * y, z * z
    basis = [torch.full_like(x, SH_C0)]
    if degree > 0:
        c1 = 0.4886025119029199
        basis += [-c1 * y, c1 * z, -c1 * x]
    if degree > 1:
        basis += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.31539156525252005 * (2 * zz - xx - yy),
                  -1.0925484305920792 * x * z, 0.5462742152960396 * (xx - yy)]
    if degree > 2:
        basis += [-0.5900435899266435 * y * (3 * xx - yy), 2.890611442640554 * x * y * z,
                  -0.4570457994644658 * y * (4 * zz - xx - yy), 0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
                  -0.4570457994644658 * x * (4 * zz - xx - yy), 1.445305721320277 * z * (xx - yy),
                  -0.5900435899266435 * x * (xx - 3 * yy)]
    return (torch.stack(basis, 1) * sh[:, :len(basis)]).sum(1) + 0.5


def _truncated(size, tan):
    """The image size as the backward pass recomputes it from the focal length, in FP32."""
    f, t = np.float32, np.float32(tan)
    return int(f(f(f(size) / f(f(2) * t)) * t) * f(2))


def _as(value, path):
    """value, with the gradient of path."""
    return path + (value - path).detach()


def _centre(T, t):
    """Centre and squared half extents of the screen box of splats T (P x 3 x 3, rows Tu, Tv, Tw)."""
    Tu, Tv, Tw = T.unbind(1)
    f = t / (t * Tw * Tw).sum(1, keepdim=True)
    c = torch.stack([(f * Tu * Tw).sum(1), (f * Tv * Tw).sum(1)], 1)
    return c, c * c - torch.stack([(f * Tu * Tu).sum(1), (f * Tv * Tv).sum(1)], 1)


def _pair(pix, T, centre, opac):
    """Alpha and depth of splats at pixels, with the low-pass floor of the footprint."""
    Tu, Tv, Tw = T.unbind(1)
    k, l = pix[:, 0:1] * Tw - Tu, pix[:, 1:2] * Tw - Tv
    p = torch.linalg.cross(k, l)
    s = p[:, :2] / p[:, 2:3]
    rho3, rho2 = (s * s).sum(1), 2.0 * ((centre - pix) ** 2).sum(1)
    near = rho3 <= rho2
    depth = torch.where(near, (s * Tw[:, :2]).sum(1) + Tw[:, 2], Tw[:, 2])
    rho = torch.where(near, rho3, rho2)
    raw = opac[:, 0] * torch.exp(-0.5 * rho)
    return _as(raw.clamp_max(0.99), raw), depth, torch.isfinite(rho) & (depth >= 0.2)


def _raster64(s, cam, degree, bg, part=False):
    """Forward of the surfel rasteriser in 64 bits.  s: the surfel tensors (float64; shs or colors).
    Returns colour, maps, semantic, radii and what the screen-space statistic needs."""
    W, H, tan = cam.image_width, cam.image_height, math.tan(cam.FoVx * 0.5)
    view, proj = cam.world_view_transform.double(), cam.full_proj_transform.double()
    mean, R = s["means3D"], _rotation(s["rotations"])
    P = mean.shape[0]
    L = R[:, :, :2] * s["scales"][:, None, :]
    pv = mean @ view[:3, :3] + view[3, :3]
    if part:
        fx = 0.5 * W / tan, 0.5 * H / tan
        rows = torch.cat([L.transpose(1, 2) @ view[:3, :3], pv[:, None]], 1)  # tangents and centre in camera space
        T = torch.stack([fx[0] * rows[..., 0] + 0.5 * W * rows[..., 2], fx[1] * rows[..., 1] + 0.5 * H * rows[..., 2],
                         rows[..., 2]], 1)
        t, shift, Wb, Hb, T_c = torch.tensor([1.0, 1.0, -1.0], device=DEV, dtype=T.dtype), 0.5, W, H, T
        centre, h2 = _centre(T, t)
    else:
        rows = torch.cat([torch.cat([L.transpose(1, 2), mean[:, None]], 1),
                          torch.tensor([0.0, 0.0, 1.0], device=DEV, dtype=mean.dtype).expand(P, 3)[:, :, None]], 2)
        A = rows @ proj

        def homography(w, h):
            return torch.stack([A[..., 0] * (w / 2) + A[..., 3] * ((w - 1) / 2),
                                A[..., 1] * (h / 2) + A[..., 3] * ((h - 1) / 2), A[..., 3]], 1)

        t, shift, Wb, Hb = torch.tensor([9.0, 9.0, -1.0], device=DEV, dtype=A.dtype), 0.0, _truncated(W, tan), \
            _truncated(H, tan)
        T_b = homography(Wb, Hb)
        T = T_c = _as(homography(W, H), T_b)
        centre, h2 = _centre(homography(W, H), t)
        centre = _as(centre, _centre(T_b, t)[0])
    T = T * 1.0  # the blend's own use of T, whose gradient the screen-space statistic reads
    if T.requires_grad:
        T.retain_grad()
        T_c.retain_grad()
    n = R[:, :, 2] @ view[:3, :3]
    facing = -(pv * n).sum(1, keepdim=True)
    normal = torch.where(facing > 0, n, -n)
    if "colors" in s:
        rgb = s["colors"]
    else:
        d = mean - cam.camera_center.double()
        rgb = _sh_color(s["shs"], degree, d / d.norm(dim=1, keepdim=True)).clamp_min(0.0)
    with torch.no_grad():
        if part:
            ext = h2.clamp_min(0.0).sqrt().amax(1).clamp_min(math.sqrt(0.5))
            radius = torch.ceil(3.0 * ext)
        else:
            radius = torch.ceil(h2.clamp_min(1e-4).sqrt().amax(1).clamp_min(3.0 * 0.707106))
        gx, gy = (W + 15) // 16, (H + 15) // 16
        lo = torch.trunc((centre - radius[:, None]) / 16)
        hi = torch.trunc((centre + radius[:, None] + 15) / 16)
        lim = torch.tensor([gx, gy], device=DEV, dtype=lo.dtype)
        lo, hi = torch.minimum(lo.clamp_min(0), lim).long(), torch.minimum(hi.clamp_min(0), lim).long()
        size = hi - lo
        area = size[:, 0] * size[:, 1]
        seen = (pv[:, 2] > 0.2) & (area > 0) & (facing[:, 0] != 0) & torch.isfinite(centre).all(1)
        area = torch.where(seen, area, torch.zeros_like(area))
        radii = torch.where(seen, radius, torch.zeros_like(radius)).int()
        who = torch.repeat_interleave(torch.arange(P, device=DEV), area)
        k = torch.arange(who.numel(), device=DEV) - (torch.cumsum(area, 0) - area)[who]
        tx, ty = lo[who, 0] + k % size[who, 0], lo[who, 1] + k // size[who, 0]
        cell = torch.arange(256, device=DEV)
        found = []
        for c in range(0, who.numel(), 16384):
            w = who[c:c + 16384]
            px = (tx[c:c + 16384, None] * 16 + cell % 16).reshape(-1)
            py = (ty[c:c + 16384, None] * 16 + cell // 16).reshape(-1)
            ws = w.repeat_interleave(256)
            ok = (px < W) & (py < H)
            px, py, ws = px[ok], py[ok], ws[ok]
            pix = torch.stack([px, py], 1).double() + shift
            alpha, _, hit = _pair(pix, T[ws], centre[ws], s["opacities"][ws])
            hit &= alpha >= 1.0 / 255.0
            found.append(torch.stack([py[hit] * W + px[hit], ws[hit]]))
        at, sid = torch.cat(found, 1) if found else torch.zeros(2, 0, dtype=torch.long, device=DEV)
        rank = torch.empty(P, dtype=torch.long, device=DEV)
        rank[torch.argsort(pv[:, 2], stable=True)] = torch.arange(P, device=DEV)
        order = torch.argsort(at * P + rank[sid])
        at, sid = at[order], sid[order]
        pix = torch.stack([at % W, at // W], 1).double() + shift
        start = torch.searchsorted(at, at)  # first pair of each pair's pixel
        # the blended pairs of a pixel end where the transmittance would fall below 1e-4
        alpha = _pair(pix, T[sid], centre[sid], s["opacities"][sid])[0]
        logs = torch.log1p(-alpha)
        after = torch.cumsum(logs, 0)
        keep = after - (after - logs)[start] >= math.log(1e-4)
        at, sid, pix = at[keep], sid[keep], pix[keep]
        start = torch.searchsorted(at, at)
    alpha, depth, _ = _pair(pix, T[sid], centre[sid], s["opacities"][sid])

    def before(x):  # sum of x over the pixel's earlier pairs
        e = torch.cumsum(x, 0) - x
        return e - e[start]

    trans = torch.exp(before(torch.log1p(-alpha)))
    w = alpha * trans
    m = 100.0 / 99.8 * (1.0 - 0.2 / depth)
    dist = (m * m * (1 - trans) + before(m * m * w) - 2 * m * before(m * w)) * w
    cols = torch.cat([rgb[sid] * w[:, None], (depth * w)[:, None], w[:, None], normal[sid] * w[:, None],
                      dist[:, None]], 1)
    flat = torch.zeros(H * W, 9, device=DEV, dtype=w.dtype).index_add(0, at, cols)
    left = 1.0 - flat[:, 4:5]
    # median: the last pair met with more than half the light left
    half = trans.detach() > 0.5
    last = torch.full((H * W,), -1, dtype=torch.long, device=DEV)
    last = last.scatter_reduce(0, at[half], torch.nonzero(half)[:, 0], "amax")
    some = last >= 0
    zero = torch.zeros(H * W, device=DEV, dtype=w.dtype)
    median = zero.index_put((torch.nonzero(some)[:, 0],), depth[last[some]])
    maps = [flat[:, 3], flat[:, 4], flat[:, 5], flat[:, 6], flat[:, 7], median, flat[:, 8]]
    semantic = None
    if part:
        maps.append(zero.index_put((torch.nonzero(some)[:, 0],), w[last[some]]))
        S = s["semantics"].shape[1]
        semantic = torch.zeros(H * W, S, device=DEV, dtype=w.dtype).index_add(0, at, s["semantics"][sid] *
                                                                             w.detach()[:, None])
        semantic = semantic.t().reshape(S, H, W)
    color = (flat[:, :3] + left * bg.double()).t().reshape(3, H, W)
    return dict(color=color, allmap=torch.stack(maps).reshape(-1, H, W), semantic=semantic, radii=radii, T=T, T_c=T_c,
                sizes=(Wb, Hb), tan=tan)


def _screen_stat(r, part):
    """The densification statistic: the gradient of T's centre column, scaled to the screen."""
    g = r["T_c"].grad if part else r["T"].grad
    z = r["T"].detach()[:, 2, 2]
    scale = [0.5 * v for v in r["sizes"]]
    return torch.stack([g[:, 0, 2] * z * scale[0], g[:, 1, 2] * z * scale[1], torch.zeros_like(z)], 1)


def _surfels64(params, occ, grid):
    """Surfels attached to the blocks' faces, one per face, in 64 bits."""
    S = torch.exp(params[:, 0:3]) + 0.2
    q = params[:, 3:7] / params[:, 3:7].norm(dim=1, keepdim=True)
    R = _rotation(q)
    eps = torch.sigmoid(params[:, 10:12]) * 1.8 + 0.1
    e1, e2 = eps[:, 0, None, None], eps[:, 1, None, None]
    E, Om = torch.meshgrid(grid.eta.double(), grid.omega.double(), indexing="ij")
    ce, se, co, so = (_spow(f(x)[None], e) for f, x, e in
                      ((torch.cos, E, e1), (torch.sin, E, e1), (torch.cos, Om, e2), (torch.sin, Om, e2)))
    local = torch.stack([ce * so, se.expand_as(ce * so), ce * co], -1) * 0.25 * S[:, None, None]
    V = torch.einsum("bijc,bcd->bijd", local, R) + params[:, None, None, 7:10]
    V0, V1 = V[:, :-1], V[:, 1:]
    V2 = torch.roll(V, -1, 2)[:, :-1]
    V0, V1, V2 = (v.reshape(-1, 3) for v in (V0, V1, V2))
    unit = lambda v: v / (v.norm(dim=1, keepdim=True) + 1e-8)  # noqa: E731
    n = unit(torch.linalg.cross(V1 - V0, V2 - V0))
    c = (V0 + V1 + V2) / 3
    len1 = (V1 - c).norm(dim=1, keepdim=True) + 1e-8
    a = (V1 - c) / len1
    b0 = V2 - c
    b = unit(b0 - (b0 * n).sum(1, keepdim=True) * n - (b0 * a).sum(1, keepdim=True) * a)
    scales = torch.cat([len1 / 2, (b0 * b).sum(1, keepdim=True) / 2], 1).clamp_min(0.0) + 1e-8
    m = torch.stack([a, b, n], -1)
    d = torch.diagonal(m, dim1=1, dim2=2)
    lead = torch.stack([1 + d[:, 0] + d[:, 1] + d[:, 2], 1 + d[:, 0] - d[:, 1] - d[:, 2],
                        1 - d[:, 0] + d[:, 1] - d[:, 2], 1 - d[:, 0] - d[:, 1] + d[:, 2]], 1)
    s = lambda i, j: m[:, i, j] + m[:, j, i]  # noqa: E731
    k = lambda i, j: m[:, i, j] - m[:, j, i]  # noqa: E731
    rows = torch.stack([torch.stack([lead[:, 0], k(2, 1), k(0, 2), k(1, 0)], 1),
                        torch.stack([k(2, 1), lead[:, 1], s(1, 0), s(0, 2)], 1),
                        torch.stack([k(0, 2), s(1, 0), lead[:, 2], s(1, 2)], 1),
                        torch.stack([k(1, 0), s(2, 0), s(2, 1), lead[:, 3]], 1)], 1)
    q = rows[torch.arange(len(rows), device=DEV), lead.argmax(1)]
    q = torch.where(q[:, :1] < 0, -q, q)
    q = q / q.norm(dim=1, keepdim=True)
    opac = torch.sigmoid(occ).repeat_interleave(E[:-1].numel())[:, None]
    return dict(means3D=c, scales=scales, rotations=q, opacities=opac)


def _sdf64(params, points):
    S = torch.exp(params[:, 0:3]) + 0.2
    R = _rotation(params[:, 3:7] / params[:, 3:7].norm(dim=1, keepdim=True))
    eps = torch.sigmoid(params[:, 10:12]) * 1.8 + 0.1
    e1, e2 = eps[:, 0:1], eps[:, 1:2]
    q = torch.einsum("bnj,bkj->bnk", points[None] - params[:, None, 7:10], R) / (S[:, None] * 0.25)
    q = q.clamp(-5.0, 5.0)
    power = lambda t, e: t.clamp_min(1e-6).pow(e)  # noqa: E731
    x, y, z = (power(q[..., i] ** 2, 1.0 / e) for i, e in ((0, e2), (1, e1), (2, e2)))
    return power(power(x + z, e2 / e1) + y, e1 / 2) - 1.0


def _knn64(pts):
    """Mean of the three smallest squared distances to other points, by looking at all of them."""
    out = []
    for c in range(0, len(pts), 4096):
        q = pts[c:c + 4096]
        d = sum((q[:, None, i] - pts[None, :, i]) ** 2 for i in range(3))
        d[torch.arange(len(q), device=DEV), torch.arange(c, c + len(q), device=DEV)] = math.inf
        total = 0.0
        for _ in range(3):
            v, i = d.min(1)
            total = total + v
            d.scatter_(1, i[:, None], math.inf)
        out.append(total / 3)
    return torch.cat(out)


def _maps64(cam, allmap):
    """render()'s maps from the rasteriser's, in 64 bits."""
    W, H = cam.image_width, cam.image_height
    view, full = cam.world_view_transform.double(), cam.full_proj_transform.double()
    c2w = view.T.inverse()
    ndc = torch.tensor([[W / 2, 0, 0, W / 2], [0, H / 2, 0, H / 2], [0, 0, 0, 1]], dtype=torch.float64, device=DEV).T
    intr = (c2w.T @ full @ ndc)[:3, :3].T
    alpha, depth = allmap[1:2], torch.nan_to_num(allmap[5:6], 0, 0)
    gx, gy = torch.meshgrid(torch.arange(W, device=DEV).double(), torch.arange(H, device=DEV).double(), indexing="xy")
    rays = torch.stack([gx, gy, torch.ones_like(gx)], -1).reshape(-1, 3) @ intr.inverse().T @ c2w[:3, :3].T
    pts = (depth.reshape(-1, 1) * rays + c2w[:3, 3]).reshape(H, W, 3)
    n = torch.zeros_like(pts)
    n[1:-1, 1:-1] = torch.nn.functional.normalize(
        torch.linalg.cross(pts[2:, 1:-1] - pts[:-2, 1:-1], pts[1:-1, 2:] - pts[1:-1, :-2]), dim=-1)
    return dict(rend_alpha=alpha, rend_normal=(allmap[2:5].permute(1, 2, 0) @ view[:3, :3].T).permute(2, 0, 1),
                rend_dist=allmap[6:7], surf_depth=depth, surf_normal=n.permute(2, 0, 1) * alpha)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("raster", "render", "part"):
        cam, bg = _camera(seed, case["W"], case["H"]), torch.ones(3, device=DEV)
        s = {k: v.double() for k, v in _scene(case, seed).items()}
        H, W = case["H"], case["W"]
        if kind == "render":
            with torch.no_grad():
                r = _raster64(s, cam, case["degree"], bg)
                return dict(render=r["color"], radii=r["radii"], **_maps64(cam, r["allmap"]))
        part = kind == "part"
        if part:
            s["semantics"] = torch.rand(case["P"], case["channels"], generator=_gen(seed, 2), device=DEV).double()
        s = {k: v.requires_grad_(True) for k, v in s.items()}
        r = _raster64(s, cam, case["degree"], bg, part)
        outs = [r["color"], r["allmap"]]
        grads = [_upstream(seed, 3, H, W).double(), _upstream(seed + 2 if part else seed + 1, 8 if part else 7, H,
                                                              W).double()]
        if part:
            outs.append(r["semantic"])
            grads.append(_upstream(seed + 1, case["channels"], H, W).double())
        torch.autograd.backward(outs, grads)
        res = dict(color=r["color"].detach(), allmap=r["allmap"].detach(), radii=r["radii"],
                   means2D=_screen_stat(r, part), **{"d_" + k: t.grad for k, t in s.items()})
        if part:
            res["semantic"] = r["semantic"].detach()
        return res
    if kind == "batch":
        return None  # 32 views of a million surfels: over 20 seconds
    if kind in ("blocks", "fit"):
        from partgs_amd.blocks import make_grid
        leaves = [t.double().requires_grad_(True) for t in _blocks(_gen(seed), case["B"])]
        params, occ, colors = leaves
        grid, bg = make_grid(case["n"], case["n"], device=DEV), torch.ones(3, device=DEV)
        W, H = case["W"], case["H"]
        s = _surfels64(params, occ, grid)
        s["colors"] = colors.repeat_interleave(case["n"] ** 2, dim=0)
        if kind == "blocks":
            r = _raster64(s, _camera(seed, W, H), 0, bg)
            torch.autograd.backward((r["color"], r["allmap"]), (_upstream(seed, 3, H, W).double(),
                                                                _upstream(seed + 1, 7, H, W).double()))
            res = dict(color=r["color"].detach(), allmap=r["allmap"].detach(), radii=r["radii"])
        else:
            image = torch.cat([_raster64(s, _camera(seed * 64 + v, W, H), 0, bg)["color"].reshape(-1)
                               for v in range(case["views"])])
            image.backward(_upstream(seed, case["views"] * 3 * H * W).double())
            res = dict(image=image.detach())
        return dict(res, d_params=params.grad, d_occ=occ.grad, d_colors=colors.grad)
    if kind == "sdf":
        params = _blocks(_gen(seed), case["B"])[0].double().requires_grad_(True)
        sdf = _sdf64(params, (_rand(_gen(seed, 3), case["N"], 3) * 2 - 1).float().double())
        sdf.backward(_upstream(seed, case["B"], case["N"]).double())
        return dict(sdf=sdf.detach(), d_params=params.grad)
    if kind == "knn":
        # a million points against a million others: over 20 seconds
        return _knn64(_surface_points(_gen(seed), case["P"])[0].float().double()) if case["P"] <= 300_000 else None
    # the network on its FP32 weights without the 16-bit roundings; those choose among near ties the point a
    # channel's maximum falls on and switch ReLUs near zero, so the gradients behind them have no such value
    from partgs_amd.proposal import ProposalNet
    w = {k: v.double() for k, v in ProposalNet(seed=seed & 0xFFFF, device=DEV).p.items()}
    pts = _proposal_points(case, seed).double()
    pooled = []
    for scene in pts:
        h = scene
        for k in "123":
            h = torch.relu(h @ w["W" + k].T + w["b" + k])
        pooled.append(h.amax(0))
    g = torch.stack(pooled)
    head = {k: w[k].clone().requires_grad_(True) for k in ("W5", "b5")}
    out = torch.relu(g @ w["W4"].T + w["b4"]) @ head["W5"].T + head["b5"]
    out.backward(_upstream(seed, case["scenes"], 16, 12).double().reshape(case["scenes"], -1))
    return dict(out=out.detach().view(-1, 16, 12), **{"d_" + k: t.grad for k, t in head.items()},
                **{"d_" + k + i: None for k in "Wb" for i in "1234"})
