"""The cell-list route of the drop-in renderer (rasterizer.view_forward) against
the per-tile-list route (forward_raw / backward_raw) on the same inputs.

Radii and images equal bit for bit, with activations in the kernels (exp,
normalisation, sigmoid, as torch rounds them) or before them, SH in one tensor
or two, every SH size that has its own kernel and one that has none, given
colours and covariances, and row counts around a work-group's 256.  Gradients
agree within 1e-5 (two orders of the same sums)."""
import pytest
import torch

from dmgs_amd import cameras as C
from dmgs_amd import gaussian_renderer as GR
from dmgs_amd import rasterizer as RZ
from dmgs_amd import scenes as S
from dmgs_amd.gaussian_renderer import PipelineParams, render
from helpers import grad_rel_err, settings_from_cam

pytestmark = pytest.mark.gpu


class _Plain(S.FreeGaussians):
    """A subclass: read through its getters."""


@pytest.mark.parametrize("P,deg,active,mod", [(1, 3, 3, 1.0), (255, 0, 0, 1.0), (256, 1, 1, 0.7), (257, 2, 2, 1.0),
                                              (1000, 3, 1, 1.0), (5001, 3, 3, 0.8)])
def test_model_tensors_equal_getters(P, deg, active, mod):
    print(f"case: view route P={P} degree={deg} active={active} modifier={mod}", flush=True)
    m = S.free_scene(P, seed=P, sh_degree=deg).to("cuda")
    m._rotation[0] = 0.0  # a quaternion whose norm is clamped
    parts = [p.clone() for p in m.parameters()]
    cam = C.camera_at((0.4, 0.3, -3.5), 173, 119)
    bg = torch.tensor([0.1, 0.6, 0.3], device="cuda")
    g = torch.randn(3, 119, 173, generator=torch.Generator().manual_seed(1)).cuda()
    got = {}
    for name, cls, pipe in (("model", S.FreeGaussians, PipelineParams()), ("getters", _Plain, PipelineParams()),
                            ("tiles", _Plain, PipelineParams(debug=True))):  # debug: the per-tile lists
        mm = cls(*[p.clone() for p in parts], sh_degree=deg).requires_grad_(True)
        mm.active_sh_degree = active
        out = render(cam, mm, pipe, bg, mod)
        (out["render"] * g).sum().backward()
        with torch.no_grad():
            eager = render(cam, mm, pipe, bg, mod)
        assert torch.equal(eager["render"], out["render"]) and torch.equal(eager["radii"], out["radii"])
        got[name] = (out["render"].detach(), out["radii"], out["viewspace_points"].grad,
                     [p.grad for p in mm.parameters()])
    for name in ("model", "getters"):
        assert torch.equal(got[name][1], got["tiles"][1]), name
        assert torch.equal(got[name][0], got["tiles"][0]), name
        assert grad_rel_err(got[name][2], got["tiles"][2]) < 1e-5, name
        for a, b in zip(got[name][3], got["tiles"][3]):
            assert (a is None) == (b is None)
            if a is not None and a.numel():
                assert grad_rel_err(a, b) < 1e-5, name


@pytest.mark.parametrize("P,M,colors,cov", [(300, 5, False, False), (257, 0, True, False), (300, 16, False, True),
                                            (513, 0, True, True)])
def test_rasterizer_inputs(P, M, colors, cov):
    """An SH size without a kernel of its own, given colours and covariances, through GaussianRasterizer."""
    print(f"case: view route inputs P={P} M={M} colors={colors} cov={cov}", flush=True)
    gen = torch.Generator().manual_seed(P)
    base = S.free_scene(P, seed=P).to("cuda")
    cam = C.camera_at((0.4, 0.3, -3.5), 90, 70)
    col = torch.rand(P, 3, generator=gen).cuda() if colors else None
    sh = None if colors else (torch.randn(P, M, 3, generator=gen) * 0.3).cuda()
    g = torch.randn(3, 70, 90, generator=gen).cuda()
    got = []
    for debug in (False, True):
        rs = settings_from_cam(cam, torch.ones(3), 1 if M == 5 else 3, debug=debug)
        leaf = lambda t: None if t is None else t.detach().clone().requires_grad_(True)
        x = dict(means3D=leaf(base._xyz), means2D=leaf(torch.zeros_like(base._xyz)), opacities=leaf(base.get_opacity),
                 shs=leaf(sh), colors_precomp=leaf(col), scales=None if cov else leaf(base.get_scaling),
                 rotations=None if cov else leaf(base.get_rotation),
                 cov3D_precomp=leaf(base.get_covariance()) if cov else None)
        color, radii = RZ.GaussianRasterizer(rs)(**x)
        (color * g).sum().backward()
        got.append((color.detach(), radii, {k: v.grad for k, v in x.items() if v is not None}))
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][0], got[1][0])
    for k, v in got[1][2].items():
        assert grad_rel_err(got[0][2][k], v) < 1e-5, k


@pytest.mark.parametrize("n", [1, 255, 257, 1000])
@pytest.mark.parametrize("M,deg", [(1, 0), (4, 1), (9, 1), (9, 2), (16, 0), (16, 3)])
def test_sh_sigmoid_kernel_equals_torch(n, M, deg):
    """sigmoid(SH) of both feature layouts against float64 torch ops.

    The sum has up to 16 products of factors below 3 in magnitude (|sh| < 5): its float32 error stays below
    16 * 15 * 2^-23 = 3e-5, and a quarter of that after the sigmoid."""
    print(f"case: sh sigmoid n={n} M={M} degree={deg}", flush=True)
    gen = torch.Generator().manual_seed(n * 31 + M + deg)
    cam = C.camera_at((0.4, 0.3, -3.5), 64, 64)
    xyz = (torch.rand(n, 3, generator=gen) * 2 - 1).cuda()
    g = torch.randn(n, 3, generator=gen).cuda()
    base = torch.randn(n, 3 * M, generator=gen).cuda()
    for color_major in (True, False):
        view = (lambda t: t.view(-1, 3, M)) if color_major else (lambda t: t.view(-1, M, 3).transpose(1, 2))
        f32, x32 = base.clone().requires_grad_(True), xyz.clone().requires_grad_(True)
        f64, x64 = base.double().requires_grad_(True), xyz.double().requires_grad_(True)
        assert GR._sh_kernel_fits(view(f32), x32, deg)
        assert not GR._sh_kernel_fits(view(f64), x64, deg)
        out, ref = GR._python_colors(view(f32), x32, cam, deg), GR._python_colors(view(f64), x64, cam, deg)
        assert (out.double() - ref).abs().max() < 8e-6
        (out * g).sum().backward()
        (ref * g.double()).sum().backward()
        assert grad_rel_err(f32.grad.double(), f64.grad) < 1e-5
        if deg:
            assert grad_rel_err(x32.grad.double(), x64.grad) < 1e-5
        else:
            assert not x32.grad.any()


def test_sh_sigmoid_second_order():
    """A graph of the backward (create_graph) goes through the torch ops."""
    gen = torch.Generator().manual_seed(3)
    cam = C.camera_at((0.4, 0.3, -3.5), 64, 64)
    xyz = (torch.rand(7, 3, generator=gen) * 2 - 1).cuda().requires_grad_(True)
    f = torch.randn(7, 3, 16, generator=gen).cuda().requires_grad_(True)
    second = []
    for ff, xx in ((f, xyz), (f.detach().double().requires_grad_(True), xyz.detach().double().requires_grad_(True))):
        a, b = torch.autograd.grad(GR._python_colors(ff, xx, cam, 3).sum(), (ff, xx), create_graph=True)
        second.append(torch.autograd.grad((a ** 2).sum() + (b ** 2).sum(), (ff, xx)))
    for s, r in zip(*second):
        assert grad_rel_err(s.double(), r) < 1e-4


def test_counts_in_plain_and_pinned_memory():
    """The geometry call writes pinned counts from its kernel and copies to plain host memory: the same numbers."""
    import ctypes
    from dmgs_amd import _native as N
    from dmgs_amd.gaussian_renderer import _settings
    lib, P = N.load(), 3000
    m = S.free_scene(P, seed=4).to("cuda")
    rs = _settings(C.camera_at((0.4, 0.3, -3.5), 173, 119), torch.zeros(3, device="cuda"), 3, 1.0, False)
    fr = RZ._Frame(rs, m._xyz.device, 16)
    g = RZ._gaussians(P, dict(means3D=m._xyz, opacities=m._opacity, shs=m._features_dc, shs_rest=m._features_rest,
                              scales=m._scaling, rotations=m._rotation),
                      RZ.RAW_SCALES | RZ.RAW_ROTATIONS | RZ.RAW_OPACITIES)
    state = torch.empty(lib.dmgs_view_state_size(P, 173, 119, 0), dtype=torch.uint8, device="cuda")
    radii = torch.empty(P, dtype=torch.int32, device="cuda")
    stream = N.stream_handle(m._xyz.device)
    got = []
    for counts in (torch.zeros(4, dtype=torch.int32, pin_memory=True)[1:3], torch.zeros(4, dtype=torch.int32)[1:3]):
        N.check(lib.dmgs_view_geometry(ctypes.byref(fr.c), ctypes.byref(g), 0, N.ptr(radii), N.ptr(state),
                                       N.ptr(counts), stream), "dmgs_view_geometry")
        N.check(lib.dmgs_view_counts(stream), "dmgs_view_counts")
        got.append(counts.tolist())
    assert got[0] == got[1] and min(got[0]) > 0
