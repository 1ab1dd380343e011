"""The rounding sequences of the backward, bit for bit: the blend's, and the per-Gaussian one over a model's tensors.

Gradients of scales and rotations are small differences of the blend's
per-splat sums, so single elements show any change in the order of its
roundings, however accurate; a norm over all elements does not.  One pixel
that looks along a row of splats centred on it makes every quantity of the
walk exact but the ones in question: alpha is the opacity 1/2, transmittances
are powers of two, and reciprocals of powers of two are exact.  What is left,

    S <- fma(1 - alpha, S, alpha <c, g>),   dL/dalpha = fma(-T_end <bg, g>, 1 / (1 - alpha), (<c, g> - S) T),

is restated here with one rounding each and compared with no tolerance.

The per-Gaussian backward of the cell-list route is compared on the same
accumulator, with no tolerance either, with the per-tile-list route's kernel
followed by torch's own gradients of exp, normalize and sigmoid."""
import ctypes

import numpy as np
import pytest
import torch

from dmgs_amd import _native as N
from dmgs_amd import cameras as C
from dmgs_amd import rasterizer as RZ
from helpers import settings_from_cam

pytestmark = pytest.mark.gpu

f32 = np.float32


def _fma(a, b, c):
    """a b + c rounded once: the product of two 24-bit numbers is exact in 64 bits."""
    return f32(np.float64(a) * np.float64(b) + np.float64(c))


def _walk(colors, g, bg):
    T = f32(0.5 ** len(colors))
    bg_term = f32(-T * f32(bg[0] * g[0] + bg[1] * g[1] + bg[2] * g[2]))  # exact: powers of two
    S, out = f32(0), []
    for c in colors[::-1]:
        T = f32(2 * T)
        cg = _fma(c[2], g[2], _fma(c[1], g[1], f32(c[0] * g[0])))
        out.append(_fma(bg_term, f32(2), f32(f32(cg - S) * T)))
        S = _fma(f32(0.5), S, f32(f32(0.5) * cg))
    return np.array(out[::-1], dtype=f32)


@pytest.mark.parametrize("tile_lists", [False, True])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_blend_backward_sequence(seed, tile_lists):
    print(f"case: gradient rounding seed={seed} tile_lists={tile_lists}", flush=True)
    n = 13  # transmittance 2^-13 is the last above 1e-4
    r = np.random.default_rng(seed)
    colors = r.random((n, 3), dtype=f32)
    g, bg = np.array([1.0, -0.25, 0.5], dtype=f32), np.array([1.0, 1.0, 0.5], dtype=f32)
    t = lambda a: torch.tensor(a, dtype=torch.float32, device="cuda")
    proj = torch.zeros(4, 4, device="cuda")
    proj[0, 0] = proj[1, 1] = proj[2, 2] = proj[2, 3] = 1.0  # w = z
    rs = RZ.GaussianRasterizationSettings(
        image_height=1, image_width=1, tanfovx=0.5, tanfovy=0.5, bg=t(bg), scale_modifier=1.0,
        viewmatrix=torch.eye(4, device="cuda"), projmatrix=proj, sh_degree=0, campos=torch.zeros(3, device="cuda"),
        prefiltered=False, debug=tile_lists)
    means = t([[0.0, 0.0, 1.0 + 0.1 * i] for i in range(n)])
    cov = t([[0.01, 0.0, 0.0, 0.01, 0.0, 0.01]] * n)
    opacity = torch.full((n, 1), 0.5, device="cuda", requires_grad=True)
    image, radii = RZ.GaussianRasterizer(rs)(means3D=means, means2D=torch.zeros_like(means), opacities=opacity,
                                             colors_precomp=t(colors), cov3D_precomp=cov)
    assert (radii > 0).all()
    (image * t(g).reshape(3, 1, 1)).sum().backward()
    got, want = opacity.grad.cpu().numpy().reshape(-1), _walk(colors, g, bg)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (got, want)


@pytest.mark.parametrize("P,M,deg,cov,raw", [
    (1, 16, 3, False, 7), (255, 1, 0, False, 7), (256, 4, 1, False, 7), (257, 9, 2, False, 7), (20011, 16, 3, False, 7),
    (20011, 16, 1, False, 4), (20011, 5, 1, False, 0), (20011, 0, 0, True, 0), (20011, 16, 3, True, 4),
    (20011, 0, 0, False, 3)])
def test_view_geometry_backward(P, M, deg, cov, raw):
    """M: SH coefficients (0: given colours); two SH tensors where the kernel takes them."""
    print(f"case: view geometry backward P={P} M={M} degree={deg} cov={cov} raw={raw}", flush=True)
    lib, g = N.load(), torch.Generator().manual_seed(P + M)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()
    xyz, log_scale, quat, logit = rnd(P, 3), rnd(P, 3) * 0.8 - 3.0, rnd(P, 4), rnd(P, 1)
    quat[0] = 0.0  # a norm that is clamped
    quat[P // 2:] *= torch.exp(rnd(P - P // 2, 1))
    A = rnd(P, 3, 3) * 0.05
    S = A @ A.transpose(1, 2)
    cov6 = torch.stack([S[:, 0, 0], S[:, 0, 1], S[:, 0, 2], S[:, 1, 1], S[:, 1, 2], S[:, 2, 2]], 1).contiguous()
    leaves = dict(scales=log_scale, rotations=quat, opacities=logit)
    leaves = {k: v.clone().requires_grad_(True) for k, v in leaves.items()}
    act = dict(scales=torch.exp(leaves["scales"]) if raw & 1 else leaves["scales"],
               rotations=torch.nn.functional.normalize(leaves["rotations"]) if raw & 2 else leaves["rotations"],
               opacities=torch.sigmoid(leaves["opacities"]) if raw & 4 else leaves["opacities"])
    shs, colors = (rnd(P, M, 3) * 0.4 if M else None), (None if M else torch.rand(P, 3, generator=g).cuda())
    cam = C.camera_at((0.7, 0.5, -2.5), 801, 603)
    fr = RZ._Frame(settings_from_cam(cam, torch.ones(3), deg, scale_modifier=0.7), xyz.device, M)
    radii = (torch.rand(P, generator=g) > 0.05).int().cuda() * 7
    acc = rnd(9 * P + 64)
    new = lambda *s: torch.full(s, 7.0, device="cuda")
    s, ptr = N.stream_handle(xyz.device), N.ptr
    shape = None if cov else (act["scales"].detach(), act["rotations"].detach())
    want = dict(means2D=new(P, 3), colors=new(P, 3), opacities=new(P, 1), conic=new(P, 4), means3D=new(P, 3),
                cov3D=new(P, 6), shs=new(P, M, 3) if M else None, scales=None if cov else new(P, 3),
                rotations=None if cov else new(P, 4))
    N.check(lib.dmgs_geometry_backward(
        ctypes.byref(fr.c), P, ptr(xyz), ptr(shs), ptr(colors), ptr(shape and shape[0]), ptr(shape and shape[1]),
        ptr(cov6) if cov else None, ptr(radii), ptr(acc), *(ptr(want[k]) for k in (
            "means2D", "colors", "opacities", "conic", "means3D", "cov3D", "shs", "scales", "rotations")), s), "tiles")
    for k in ("opacities",) if cov else ("scales", "rotations", "opacities"):
        if act[k] is not leaves[k]:
            want[k] = torch.autograd.grad(act[k], leaves[k], want[k])[0]
    for split in (False, True) if M in (4, 9, 16) else (False,):
        t = dict(means3D=xyz, colors_precomp=colors, shs=shs, cov3D_precomp=cov6 if cov else None,
                 **{k: v.detach() for k, v in leaves.items() if k == "opacities" or not cov})
        got = dict(means2D=new(P, 3), colors=new(P, 3), opacities=new(P, 1), means3D=new(P, 3), cov3D=new(P, 6))
        if not cov:
            got.update(scales=new(P, 3), rotations=new(P, 4))
        if M:
            got["shs"] = new(P, M, 3)
        if split:
            t["shs"], t["shs_rest"] = shs[:, :1].clone(), shs[:, 1:].clone()
            got["shs"], got["shs_rest"] = new(P, 1, 3), new(P, M - 1, 3)
        d = N.DmgsGaussianGrads()
        for k, v in got.items():
            setattr(d, k, v.data_ptr())
        N.check(lib.dmgs_view_geometry_backward(ctypes.byref(fr.c), ctypes.byref(RZ._gaussians(P, t, raw)), ptr(radii),
                                                ptr(acc), ctypes.byref(d), s), "view")
        if split:
            got["shs"] = torch.cat((got["shs"], got.pop("shs_rest")), 1)
        for k, v in got.items():
            assert torch.equal(v, want[k]), (k, split, (v != want[k]).sum().item())
