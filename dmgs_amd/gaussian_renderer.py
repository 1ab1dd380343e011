"""Drop-in ``render`` / ``render_dyn`` (gaussian_renderer/__init__.py:18-101,
104-193), same signatures and return dicts, backed by the gfx950 rasterizer.

``pipe`` only needs the attributes ``PipelineParams`` defines
(arguments/__init__.py:64-69): ``convert_SHs_python``, ``compute_cov3D_python``
and ``debug``.  The model protocol is the reference's (get_xyz, get_opacity,
get_scaling, get_rotation, get_features, get_covariance, active_sh_degree,
max_sh_degree, scene/gaussian_model.py:95-118).  The Python SH path applies
``sigmoid`` to the SH value, as the reference adapter does
(gaussian_renderer/__init__.py:74-78); the kernel path adds 0.5 and clamps.
"""
import math

import torch

from . import _native as N
from .binding import FaceBoundGaussians
from .rasterizer import (RAW_OPACITIES, RAW_ROTATIONS, RAW_SCALES, GaussianRasterizationSettings, GaussianRasterizer,
                         _cells_route, _f32, model_inputs_fit, rasterize_model)
from .scenes import FreeGaussians
from .sh_utils import eval_sh


class PipelineParams:
    """Defaults of the reference's PipelineParams (arguments/__init__.py:64-69)."""

    def __init__(self, convert_SHs_python=False, compute_cov3D_python=False, debug=False):
        self.convert_SHs_python = convert_SHs_python
        self.compute_cov3D_python = compute_cov3D_python
        self.debug = debug


def _settings(cam, bg_color, sh_degree, scaling_modifier, debug):
    dev = bg_color.device
    return GaussianRasterizationSettings(
        image_height=int(cam.image_height), image_width=int(cam.image_width),
        tanfovx=math.tan(cam.FoVx * 0.5), tanfovy=math.tan(cam.FoVy * 0.5), bg=bg_color,
        scale_modifier=scaling_modifier, viewmatrix=cam.world_view_transform.to(dev),
        projmatrix=cam.full_proj_transform.to(dev), sh_degree=sh_degree,
        campos=cam.camera_center.to(dev), prefiltered=False, debug=debug)


def _screenspace(xyz):
    pts = torch.zeros_like(xyz, dtype=xyz.dtype, requires_grad=True, device=xyz.device)
    try:
        pts.retain_grad()
    except Exception:
        pass
    return pts


def _torch_colors(features_view, xyz, campos, active_sh_degree):
    dirs = xyz - campos.repeat(features_view.shape[0], 1)
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    return torch.sigmoid(eval_sh(active_sh_degree, features_view, dirs))


# The Python SH path as one kernel each way (352 launches per training iteration of 122 880 Gaussians before).
class _ShSigmoid(torch.autograd.Function):
    @staticmethod
    def forward(ctx, feats, xyz, campos, degree):
        n, _, M = feats.shape
        colors = torch.empty(n, 3, dtype=torch.float32, device=xyz.device)
        N.check(N.load().dmgs_sh_sigmoid(n, M, degree, int(feats.stride(2) == 1), N.ptr(feats), N.ptr(xyz),
                                         N.ptr(campos), N.ptr(colors), None, None, None, N.stream_handle(xyz.device)),
                "dmgs_sh_sigmoid")
        ctx.save_for_backward(feats, xyz, campos, colors)
        ctx.degree = degree
        return colors

    @staticmethod
    def backward(ctx, grad):
        feats, xyz, campos, colors = ctx.saved_tensors
        n, _, M = feats.shape
        if torch.is_grad_enabled():  # create_graph: the derivative of the torch ops, itself differentiable
            asked = [t for t, need in zip((feats, xyz), ctx.needs_input_grad) if need]
            out = _torch_colors(feats, xyz, campos, ctx.degree)
            grads = iter(torch.autograd.grad(out, asked, grad, create_graph=True, allow_unused=True)
                         if out.requires_grad else [None] * len(asked))
            return tuple(next(grads) if need else None for need in ctx.needs_input_grad[:2]) + (None, None)
        # saved-tensor hooks may give the tensors back in another layout or type
        xyz, campos, colors, g = (_f32(t, xyz.device) for t in (xyz, campos, colors, grad))
        if not _sh_kernel_fits(feats, xyz, ctx.degree):
            feats = _f32(feats, xyz.device)
        dfeats = torch.empty_strided(feats.shape, feats.stride(), dtype=torch.float32, device=feats.device)
        dxyz = torch.empty_like(xyz)
        N.check(N.load().dmgs_sh_sigmoid(n, M, ctx.degree, int(feats.stride(2) == 1), N.ptr(feats), N.ptr(xyz),
                                         N.ptr(campos), N.ptr(colors), N.ptr(g), N.ptr(dfeats), N.ptr(dxyz),
                                         N.stream_handle(xyz.device)), "dmgs_sh_sigmoid")
        return dfeats, dxyz, None, None


def _sh_kernel_fits(feats, xyz, degree):
    """Whether (n, 3, M) features are rows the SH kernel reads in place."""
    if feats.dim() != 3 or feats.shape[1] != 3 or xyz.dim() != 2 or tuple(xyz.shape) != (feats.shape[0], 3):
        return False
    n, _, M = feats.shape
    return (n > 0 and M in (1, 4, 9, 16) and 0 <= degree <= 3 and (degree + 1) ** 2 <= M and
            feats.device.type == "cuda" and feats.device == xyz.device and
            feats.dtype == torch.float32 and xyz.dtype == torch.float32 and xyz.is_contiguous() and
            feats.stride() in ((3 * M, M, 1), (3 * M, 1, 3)) and feats.data_ptr() % 16 == 0)


def _python_colors(features_view, xyz, cam, active_sh_degree):
    if _sh_kernel_fits(features_view, xyz, active_sh_degree):
        campos = cam.camera_center.to(device=xyz.device, dtype=torch.float32).contiguous()
        if campos.numel() == 3 and not campos.requires_grad:
            return _ShSigmoid.apply(features_view, xyz, campos, active_sh_degree)
    return _torch_colors(features_view, xyz, cam.camera_center.to(xyz.device), active_sh_degree)


def _model_tensors(pc):
    """(xyz, dc, rest, opacity, scales, rotations, raw mask) of this package's
    own models, whose getters the rasterizer's kernels evaluate themselves, or
    None (any other model, a subclass included, is read through its getters)."""
    if type(pc) is FreeGaussians:
        return (pc._xyz, pc._features_dc, pc._features_rest, pc._opacity, pc._scaling, pc._rotation,
                RAW_SCALES | RAW_ROTATIONS | RAW_OPACITIES)
    if type(pc) is FaceBoundGaussians:
        return (pc._xyz, pc._masked(pc._features_dc), pc._masked(pc._features_rest), pc._masked(pc._opacity),
                pc._scale, pc._rot, RAW_OPACITIES)
    return None


def render(viewpoint_camera, pc, pipe, bg_color: torch.Tensor, scaling_modifier=1.0, override_color=None):
    """Render the scene (gaussian_renderer/__init__.py:18-101)."""
    screenspace_points = _screenspace(pc.get_xyz)
    rs = _settings(viewpoint_camera, bg_color, pc.active_sh_degree, scaling_modifier, pipe.debug)
    if not pipe.compute_cov3D_python and not pipe.convert_SHs_python and override_color is None and _cells_route(rs):
        m = _model_tensors(pc)
        if m is not None and model_inputs_fit(*m[:-1]):
            xyz, dc, rest, opacity, scales, rotations, raw = m
            rendered_image, radii = rasterize_model(xyz, screenspace_points, dc, rest, opacity, scales, rotations,
                                                    raw, rs)
            return {"render": rendered_image, "viewspace_points": screenspace_points,
                    "visibility_filter": radii > 0, "radii": radii}
    rasterizer = GaussianRasterizer(raster_settings=rs)
    means3D = pc.get_xyz
    opacity = pc.get_opacity
    scales = rotations = cov3D_precomp = None
    if pipe.compute_cov3D_python:
        cov3D_precomp = pc.get_covariance(scaling_modifier)
    else:
        scales = pc.get_scaling
        rotations = pc.get_rotation
    shs = colors_precomp = None
    if override_color is None:
        if pipe.convert_SHs_python:
            feats = pc.get_features
            shs_view = feats.transpose(1, 2).view(-1, 3, (pc.max_sh_degree + 1) ** 2)
            colors_precomp = _python_colors(shs_view, pc.get_xyz, viewpoint_camera, pc.active_sh_degree)
        else:
            shs = pc.get_features
    else:
        colors_precomp = override_color
    rendered_image, radii = rasterizer(means3D=means3D, means2D=screenspace_points, shs=shs,
                                       colors_precomp=colors_precomp, opacities=opacity, scales=scales,
                                       rotations=rotations, cov3D_precomp=cov3D_precomp)
    return {"render": rendered_image, "viewspace_points": screenspace_points, "visibility_filter": radii > 0,
            "radii": radii}


def render_dyn(viewpoint_camera, gs_info: dict, pipe, bg_color: torch.Tensor, scaling_modifier=1.0,
               override_color=None):
    """Render dynamically generated Gaussians (gaussian_renderer/__init__.py:104-193).
    Requires ``pipe.compute_cov3D_python`` like the reference (NotImplementedError otherwise)."""
    xyz = gs_info['xyz']
    opacity = gs_info['opacity']
    covariance = gs_info['covariance']
    features = gs_info['features']
    active_sh_degree = gs_info['active_sh_degree']
    max_sh_degree = gs_info['max_sh_degree']
    screenspace_points = _screenspace(xyz)
    rs = _settings(viewpoint_camera, bg_color, active_sh_degree, scaling_modifier, pipe.debug)
    rasterizer = GaussianRasterizer(raster_settings=rs)
    if not pipe.compute_cov3D_python:
        raise NotImplementedError
    cov3D_precomp = covariance
    shs = colors_precomp = None
    if override_color is None:
        if pipe.convert_SHs_python:
            shs_view = features.view(-1, 3, (max_sh_degree + 1) ** 2)
            colors_precomp = _python_colors(shs_view, xyz, viewpoint_camera, active_sh_degree)
        else:
            shs = features
    else:
        colors_precomp = override_color
    rendered_image, radii = rasterizer(means3D=xyz, means2D=screenspace_points, shs=shs,
                                       colors_precomp=colors_precomp, opacities=opacity, scales=None,
                                       rotations=None, cov3D_precomp=cov3D_precomp)
    return {"render": rendered_image, "viewspace_points": screenspace_points, "visibility_filter": radii > 0,
            "radii": radii}
