"""Drop-in replacement for the ``diff_gaussian_rasterization`` Python module.

Same names and argument meaning as the reference's rasterizer API, as called
from gaussian_renderer/__init__.py:14,36-51,86-94 (the module itself is the
un-vendored submodule named in .gitmodules:4-6):

* ``GaussianRasterizationSettings`` — 12 fields, NamedTuple;
* ``GaussianRasterizer(settings)(means3D, means2D, opacities, shs=None,
  colors_precomp=None, scales=None, rotations=None, cov3D_precomp=None)``
  -> ``(color (3,H,W) float32, radii (P,) int32)``, plus ``markVisible``;
* ``rasterize_gaussians`` / ``_RasterizeGaussians`` (torch.autograd.Function)
  whose backward returns gradients in input order, ``means2D.grad`` in NDC
  units with z = 0.

Errors follow the reference: an ``Exception`` unless exactly one of {shs,
colors_precomp} and exactly one of {(scales, rotations), cov3D_precomp} is
given; P == 0 returns an all-zero image.  With ``debug`` every kernel is
synchronised and checked, and a failing call saves its CPU-copied arguments to
``snapshot_fw.dump`` / ``snapshot_bw.dump`` before re-raising.

All compute runs in the gfx950 HIP library through ``dmgs_amd._native``.  An
image takes the cell-list route (``view_forward``: the batched engine's lists
and blend with one view); ``forward_raw`` / ``backward_raw`` are the route of
the reference's per-tile lists, taken with ``debug`` (every kernel
synchronised), for images of more than 65536 cells of 64x64 pixels or 65535
tiles a side, and by callers that want those lists.  Both give the same image bit for bit.
"""
import ctypes
from typing import NamedTuple

import torch
import torch.nn as nn

from . import _native as N


class GaussianRasterizationSettings(NamedTuple):
    image_height: int
    image_width: int
    tanfovx: float
    tanfovy: float
    bg: torch.Tensor
    scale_modifier: float
    viewmatrix: torch.Tensor
    projmatrix: torch.Tensor
    sh_degree: int
    campos: torch.Tensor
    prefiltered: bool
    debug: bool


def _f32(t, device):
    t = t.to(device=device, dtype=torch.float32).contiguous()
    if t.data_ptr() % 16:  # the kernels use 16-byte vector loads
        t = t.clone()
    return t


def _present(t):
    return t is not None and t.numel() > 0


class _Frame:
    """Device-side copies of the per-view constants and the C settings struct."""

    def __init__(self, rs, device, sh_coeffs):
        self.view = _f32(rs.viewmatrix, device)
        self.proj = _f32(rs.projmatrix, device)
        self.campos = _f32(rs.campos, device).reshape(-1)
        self.bg = _f32(rs.bg, device).reshape(-1)
        if self.bg.numel() != 3:
            raise ValueError("bg must have 3 channels")
        s = N.DmgsSettings()
        s.image_width = int(rs.image_width)
        s.image_height = int(rs.image_height)
        s.tanfovx = float(rs.tanfovx)
        s.tanfovy = float(rs.tanfovy)
        s.scale_modifier = float(rs.scale_modifier)
        s.sh_degree = int(rs.sh_degree)
        s.sh_coeffs = int(sh_coeffs)
        s.prefiltered = int(bool(rs.prefiltered))
        s.debug = int(bool(rs.debug))
        s.viewmatrix = self.view.data_ptr()
        s.projmatrix = self.proj.data_ptr()
        s.campos = self.campos.data_ptr()
        s.bg = self.bg.data_ptr()
        self.c = s


class _NullStage:
    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


_NULL_STAGE = _NullStage()
_stage_hook = None


def set_stage_hook(hook):
    """Install ``hook(name)`` returning a context manager entered around every
    C-ABI stage call on the launching stream (used by the benchmark to time
    stages with device events).  ``None`` removes it."""
    global _stage_hook
    _stage_hook = hook


def _stage(name):
    return _NULL_STAGE if _stage_hook is None else _stage_hook(name)


def _cpu_copy(args):
    return tuple(a.detach().cpu() if isinstance(a, torch.Tensor) else a for a in args)


def rasterize_gaussians(means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                        raster_settings):
    fn = _RasterizeGaussians if torch.is_grad_enabled() else _RasterizeGaussiansNoGrad
    return fn.apply(means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                    raster_settings)


def _check_color_and_shape(sh, colors_precomp, scales, rotations, cov3Ds_precomp):
    if _present(sh) == _present(colors_precomp):
        raise Exception("Please provide excatly one of either SHs or precomputed colors!")
    if (_present(scales) or _present(rotations)) == _present(cov3Ds_precomp) or \
            (_present(scales) != _present(rotations)):
        raise Exception("Please provide exactly one of either scale/rotation pair or precomputed 3D covariance!")


def forward_raw(means3D, opacities, sh, colors_precomp, scales, rotations, cov3Ds_precomp, rs):
    """Run the forward pipeline; returns (color, radii, state) where state holds
    everything the backward needs (the reference's three byte buffers)."""
    dev = means3D.device
    if dev.type != "cuda":
        raise RuntimeError("dmgs_amd rasterizer needs CUDA/HIP tensors")
    N.load()
    P = means3D.shape[0]
    if means3D.dim() != 2 or means3D.shape[1] != 3:
        raise RuntimeError("means3D must have dimensions (num_points, 3)")
    H, W = int(rs.image_height), int(rs.image_width)
    M = sh.shape[1] if _present(sh) else 0
    radii = torch.zeros(P, dtype=torch.int32, device=dev)
    if P == 0:
        return torch.zeros(3, H, W, dtype=torch.float32, device=dev), radii, None
    _check_color_and_shape(sh, colors_precomp, scales, rotations, cov3Ds_precomp)
    fr = _Frame(rs, dev, M)
    t = dict(
        means3D=_f32(means3D, dev), opacities=_f32(opacities, dev),
        shs=_f32(sh, dev) if _present(sh) else None,
        colors=_f32(colors_precomp, dev) if _present(colors_precomp) else None,
        scales=_f32(scales, dev) if _present(scales) else None,
        rotations=_f32(rotations, dev) if _present(rotations) else None,
        cov3D=_f32(cov3Ds_precomp, dev) if _present(cov3Ds_precomp) else None,
    )
    lib = N.load()
    stream = N.stream_handle(dev)
    geom = torch.empty(lib.dmgs_geometry_workspace_size(P), dtype=torch.uint8, device=dev)
    count = torch.zeros(1, dtype=torch.int32, device=dev)
    with _stage("geometry"):
        N.check(lib.dmgs_forward_geometry(ctypes_ref(fr.c), P, N.ptr(t["means3D"]), N.ptr(t["opacities"]),
                                          N.ptr(t["shs"]), N.ptr(t["colors"]), N.ptr(t["scales"]),
                                          N.ptr(t["rotations"]), N.ptr(t["cov3D"]), N.ptr(radii), N.ptr(geom),
                                          N.ptr(count), stream), "dmgs_forward_geometry")
    K = int(count.item())  # the one host synchronisation of the plain path (as in the reference)
    binning = torch.empty(max(1, lib.dmgs_binning_workspace_size(K)), dtype=torch.uint8, device=dev)
    image = torch.empty(lib.dmgs_image_workspace_size(W, H), dtype=torch.uint8, device=dev)
    color = torch.empty(3, H, W, dtype=torch.float32, device=dev)
    with _stage("binning"):
        N.check(lib.dmgs_forward_binning(ctypes_ref(fr.c), P, K, N.ptr(geom), N.ptr(binning), N.ptr(image),
                                         stream), "dmgs_forward_binning")
    with _stage("render_forward"):
        N.check(lib.dmgs_render_forward(ctypes_ref(fr.c), P, K, N.ptr(geom), N.ptr(binning), N.ptr(image),
                                        N.ptr(color), stream), "dmgs_render_forward")
    state = dict(frame=fr, tensors=t, geom=geom, binning=binning, image=image, K=K, P=P, M=M)
    return color, radii, state


def backward_raw(state, radii, grad_color):
    """Run the backward pipeline for a forward ``state``; returns a dict of gradients."""
    fr, t = state["frame"], state["tensors"]
    P, K, M = state["P"], state["K"], state["M"]
    dev = t["means3D"].device
    lib = N.load()
    f = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=dev)
    out = dict(means2D=f(P, 3), colors=f(P, 3), opacity=f(P, 1), conic=f(P, 2, 2), means3D=f(P, 3),
               cov3D=f(P, 6), sh=f(P, M, 3) if t["shs"] is not None else None,
               scales=f(P, 3) if t["scales"] is not None else None,
               rotations=f(P, 4) if t["rotations"] is not None else None)
    bws = torch.empty(lib.dmgs_backward_workspace_size(P), dtype=torch.uint8, device=dev)
    g = grad_color.to(dtype=torch.float32).contiguous()
    stream = N.stream_handle(dev)
    with _stage("render_backward"):
        N.check(lib.dmgs_render_backward(ctypes_ref(fr.c), P, K, N.ptr(state["geom"]), N.ptr(state["binning"]),
                                         N.ptr(state["image"]), N.ptr(bws), N.ptr(g), stream), "dmgs_render_backward")
    with _stage("geometry_backward"):
        N.check(lib.dmgs_geometry_backward(ctypes_ref(fr.c), P, N.ptr(t["means3D"]), N.ptr(t["shs"]),
                                           N.ptr(t["colors"]), N.ptr(t["scales"]), N.ptr(t["rotations"]),
                                           N.ptr(t["cov3D"]), N.ptr(radii), N.ptr(bws), N.ptr(out["means2D"]),
                                           N.ptr(out["colors"]), N.ptr(out["opacity"]), N.ptr(out["conic"]),
                                           N.ptr(out["means3D"]), N.ptr(out["cov3D"]), N.ptr(out["sh"]),
                                           N.ptr(out["scales"]), N.ptr(out["rotations"]), stream),
                "dmgs_geometry_backward")
    return out


def ctypes_ref(struct):
    return ctypes.byref(struct)


# ---- the cell-list route -------------------------------------------------
RAW_SCALES, RAW_ROTATIONS, RAW_OPACITIES = 1, 2, 4
_INPUTS = ("means3D", "opacities", "shs", "shs_rest", "colors_precomp", "scales", "rotations", "cov3D_precomp")


def _gaussians(P, t, raw):
    g = N.DmgsGaussians()
    g.count, g.raw = P, raw
    for name in _INPUTS:
        x = t.get(name)
        if x is not None:
            setattr(g, name, x.data_ptr())
    return g


def view_forward(t, sh_coeffs, raw, rs, keep):
    """One image from a model's tensors: ``t`` maps the names of ``_INPUTS``
    to contiguous float32, 16-byte aligned device tensors, ``raw`` marks what
    the kernels activate, ``keep`` says that a backward will follow.  Returns
    (color, radii, state); state holds what ``view_backward`` needs beside
    the inputs."""
    means = t["means3D"]
    dev, P = means.device, means.shape[0]
    H, W = int(rs.image_height), int(rs.image_width)
    fr = _Frame(rs, dev, sh_coeffs)
    lib = N.load()
    stream = N.stream_handle(dev)
    byte = dict(dtype=torch.uint8, device=dev)
    nbytes = lib.dmgs_view_state_size(P, W, H, int(keep))
    ws = torch.empty(nbytes, **byte)
    radii = torch.empty(P, dtype=torch.int32, device=dev)
    counts = torch.empty(2, dtype=torch.int32, pin_memory=True)
    s = ctypes_ref(fr.c)
    g = _gaussians(P, t, raw)
    with _stage("geometry"):  # ends with the one host synchronisation of the path (as in the reference)
        N.check(lib.dmgs_view_geometry(s, ctypes_ref(g), int(keep), N.ptr(radii), N.ptr(ws), N.ptr(counts), stream),
                "dmgs_view_geometry")
        try:  # what does not depend on the counts is allocated while they are on their way
            bws = torch.empty(lib.dmgs_batched_backward_size(1, P), **byte) if keep else None
            color = torch.empty(3, H, W, dtype=torch.float32, device=dev)
        finally:  # also on an error: the copy writes into counts
            rc = lib.dmgs_view_counts(stream)
        N.check(rc, "dmgs_view_counts")
    cells, tiles = (int(c) & 0xFFFFFFFF for c in counts.tolist())
    K = max(1, cells)
    lists = torch.empty(lib.dmgs_batched_lists_size(K), **byte)
    with _stage("binning"):
        N.check(lib.dmgs_view_binning(s, P, int(keep), K, N.ptr(ws), N.ptr(lists), stream), "dmgs_view_binning")
    with _stage("render_forward"):
        N.check(lib.dmgs_view_blend(s, P, int(keep), K, N.ptr(ws), N.ptr(lists), N.ptr(bws), N.ptr(color), stream),
                "dmgs_view_blend")
    return color, radii, dict(frame=fr, ws=ws, lists=lists, bws=bws, cells=K, K=tiles, P=P, M=sh_coeffs, raw=raw,
                              walked=False)


def view_backward(t, state, radii, grad_color, colors=False, cov3D=False):
    """Gradients of ``view_forward`` (dict by input name, and ``means2D``);
    colour and covariance gradients where asked for."""
    fr, P = state["frame"], state["P"]
    dev = radii.device
    lib = N.load()
    f = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=dev)
    like = lambda name: None if t.get(name) is None else torch.empty_like(t[name])
    out = dict(means2D=f(P, 3), means3D=f(P, 3), opacities=f(P, 1), shs=like("shs"), shs_rest=like("shs_rest"),
               scales=like("scales"), rotations=like("rotations"), colors_precomp=f(P, 3) if colors else None,
               cov3D_precomp=f(P, 6) if cov3D else None)
    d = N.DmgsGaussianGrads()
    for field, name in (("means2D", "means2D"), ("means3D", "means3D"), ("opacities", "opacities"), ("shs", "shs"),
                        ("shs_rest", "shs_rest"), ("colors", "colors_precomp"), ("cov3D", "cov3D_precomp"),
                        ("scales", "scales"), ("rotations", "rotations")):
        if out[name] is not None:
            setattr(d, field, out[name].data_ptr())
    gc = grad_color.to(dtype=torch.float32).contiguous()
    stream = N.stream_handle(dev)
    s = ctypes_ref(fr.c)
    with _stage("render_backward"):
        if state["walked"]:  # the forward left the accumulator cleared for one backward
            state["bws"][:lib.dmgs_backward_workspace_size(P)].zero_()
        state["walked"] = True
        N.check(lib.dmgs_view_blend_backward(s, P, state["cells"], N.ptr(state["ws"]), N.ptr(state["lists"]),
                                             N.ptr(state["bws"]), N.ptr(gc), stream), "dmgs_view_blend_backward")
    with _stage("geometry_backward"):
        N.check(lib.dmgs_view_geometry_backward(s, ctypes_ref(_gaussians(P, t, state["raw"])), N.ptr(radii),
                                                N.ptr(state["bws"]), ctypes_ref(d), stream),
                "dmgs_view_geometry_backward")
    return out


def _cells_route(rs):
    return not rs.debug and N.load().dmgs_view_supported(int(rs.image_width), int(rs.image_height)) == 1


def _take_state(ctx):
    """The forward's state, for one backward: kept for another one while the graph is (``retain_graph``), released
    with it otherwise, so that the workspaces do not live as long as the image does."""
    if ctx.state is _RELEASED:
        raise RuntimeError("Trying to backward through a rendered image a second time: specify retain_graph=True for "
                           "the first")
    state = ctx.state
    if not _graph_is_kept():
        ctx.state = _RELEASED
    return state


_RELEASED = object()
# torch's own test, as its compiled functions use it; without it nothing is released early
_graph_is_kept = getattr(torch._C._autograd, "_get_current_graph_task_keep_graph", lambda: True)


def _rasterize(ctx, args, keep):
    """Shared forward of the two autograd functions below."""
    means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp, rs = args
    raw_args = (means3D, opacities, sh, colors_precomp, scales, rotations, cov3Ds_precomp, rs)
    if rs.debug:
        try:
            color, radii, state = forward_raw(*raw_args)
        except Exception:
            torch.save(_cpu_copy(raw_args[:-1]), "snapshot_fw.dump")
            print("\nAn error occured in forward. Please forward snapshot_fw.dump for debugging.")
            raise
    elif means3D.device.type != "cuda" or means3D.dim() != 2 or means3D.shape[1] != 3 or means3D.shape[0] == 0 or \
            not _cells_route(rs):
        color, radii, state = forward_raw(*raw_args)
    else:
        _check_color_and_shape(sh, colors_precomp, scales, rotations, cov3Ds_precomp)
        dev = means3D.device
        opt = lambda x: _f32(x, dev) if _present(x) else None
        t = dict(means3D=_f32(means3D, dev), opacities=_f32(opacities, dev), shs=opt(sh), colors_precomp=opt(colors_precomp),
                 scales=opt(scales), rotations=opt(rotations), cov3D_precomp=opt(cov3Ds_precomp))
        color, radii, state = view_forward(t, sh.shape[1] if _present(sh) else 0, 0, rs, keep)
        state["tensors"] = t
    ctx.state = state if keep else None
    ctx.raster_settings = rs
    ctx.num_rendered = 0 if state is None else state["K"]
    ctx.shapes = [None if x is None else x.shape for x in args[:-1]]
    ctx.mark_non_differentiable(radii)
    return color, radii


class _RasterizeGaussians(torch.autograd.Function):
    @staticmethod
    def forward(ctx, means3D, means2D, sh, colors_precomp, opacities, scales, rotations, cov3Ds_precomp,
                raster_settings):
        color, radii = _rasterize(ctx, (means3D, means2D, sh, colors_precomp, opacities, scales, rotations,
                                        cov3Ds_precomp, raster_settings), True)
        ctx.save_for_backward(radii)
        return color, radii

    @staticmethod
    def backward(ctx, grad_out_color, _grad_radii):
        (radii,) = ctx.saved_tensors
        state = _take_state(ctx)
        shapes = ctx.shapes
        needs = ctx.needs_input_grad
        if state is None:  # no Gaussians
            z = [None if (s is None or not needs[i]) else torch.zeros(s, device=grad_out_color.device)
                 for i, s in enumerate(shapes)]
            return tuple(z) + (None,)
        if "ws" in state:
            g = view_backward(state["tensors"], state, radii, grad_out_color, colors=needs[3], cov3D=needs[7])
            ordered = [g["means3D"], g["means2D"], g["shs"], g["colors_precomp"], g["opacities"], g["scales"],
                       g["rotations"], g["cov3D_precomp"]]
        else:
            if ctx.raster_settings.debug:
                try:
                    g = backward_raw(state, radii, grad_out_color)
                except Exception:
                    torch.save(_cpu_copy((grad_out_color,) + tuple(state["tensors"].values())), "snapshot_bw.dump")
                    print("\nAn error occured in backward. Writing snapshot_bw.dump for debugging.\n")
                    raise
            else:
                g = backward_raw(state, radii, grad_out_color)
            ordered = [g["means3D"], g["means2D"], g["sh"], g["colors"], g["opacity"], g["scales"], g["rotations"],
                       g["cov3D"]]
        grads = []
        for i, (gr, s) in enumerate(zip(ordered, shapes)):
            if not needs[i] or s is None or gr is None or s.numel() == 0:
                grads.append(None)
            else:
                grads.append(gr.reshape(s))
        return tuple(grads) + (None,)


class _RasterizeGaussiansNoGrad(torch.autograd.Function):
    """The forward with autograd off: nothing is kept for a backward."""

    @staticmethod
    def forward(ctx, *args):
        return _rasterize(ctx, args, False)


def _through_activations(t, state, radii, grad_color):
    """``view_backward`` of a model's tensors with a graph of its own (create_graph): the rasterizer's gradients,
    which have none, through torch's activations, which do."""
    raw = state["raw"]
    acts = dict(t)
    if raw & RAW_SCALES:
        acts["scales"] = torch.exp(t["scales"])
    if raw & RAW_ROTATIONS:
        acts["rotations"] = nn.functional.normalize(t["rotations"])
    if raw & RAW_OPACITIES:
        acts["opacities"] = torch.sigmoid(t["opacities"])
    with torch.no_grad():
        g = view_backward({k: x.detach() for k, x in acts.items()}, dict(state, raw=0), radii, grad_color)
    state["walked"] = True
    for k in ("scales", "rotations", "opacities"):
        if acts[k] is not t[k] and acts[k].requires_grad:
            g[k], = torch.autograd.grad(acts[k], t[k], g[k], create_graph=True)
    return g


class _RasterizeModel(torch.autograd.Function):
    """A model's own tensors (``raw`` as in ``view_forward``), SH in two
    tensors; gradients reach those tensors directly."""

    @staticmethod
    def forward(ctx, xyz, means2D, dc, rest, opacity, scales, rotations, raw, rs, keep):
        t = dict(means3D=xyz, opacities=opacity, shs=dc, scales=scales, rotations=rotations)
        if rest.numel():
            t["shs_rest"] = rest
        color, radii, state = view_forward(t, 1 + rest.shape[1], raw, rs, keep)
        if keep:
            ctx.save_for_backward(radii, xyz, dc, rest, opacity, scales, rotations)
            ctx.state = state
        ctx.num_rendered = state["K"]
        ctx.mark_non_differentiable(radii)
        return color, radii

    @staticmethod
    def backward(ctx, grad_out_color, _grad_radii):
        radii, *saved = ctx.saved_tensors
        xyz, dc, rest, opacity, scales, rotations = (_f32(x, radii.device) for x in saved)  # hooks may change them
        needs = ctx.needs_input_grad
        state = _take_state(ctx)
        t = dict(means3D=xyz, opacities=opacity, shs=dc, scales=scales, rotations=rotations)
        if rest.numel():
            t["shs_rest"] = rest
        if torch.is_grad_enabled():
            g = _through_activations(t, state, radii, grad_out_color)
        else:
            g = view_backward(t, state, radii, grad_out_color)
        out = (g["means3D"], g["means2D"], g["shs"], rest.new_zeros(rest.shape) if g["shs_rest"] is None else g["shs_rest"],
               g["opacities"], g["scales"], g["rotations"])
        return tuple(x if n else None for x, n in zip(out, needs)) + (None, None, None)


def model_inputs_fit(xyz, dc, rest, opacity, scales, rotations):
    """Whether a model's tensors have the form ``rasterize_model`` reads in
    place: contiguous float32 on one GPU, 16-byte aligned, at least one row,
    and 1, 4, 9 or 16 SH coefficients."""
    P = xyz.shape[0]
    if xyz.dim() != 2 or P == 0 or dc.dim() != 3 or rest.dim() != 3:
        return False
    M = 1 + rest.shape[1]
    want = ((xyz, (P, 3)), (dc, (P, 1, 3)), (rest, (P, M - 1, 3)), (opacity, (P, 1)), (scales, (P, 3)),
            (rotations, (P, 4)))
    dev = xyz.device
    return dev.type == "cuda" and M in (1, 4, 9, 16) and all(
        tuple(x.shape) == s and x.dtype == torch.float32 and x.device == dev and x.is_contiguous() and
        x.data_ptr() % 16 == 0 for x, s in want)


def rasterize_model(xyz, means2D, dc, rest, opacity, scales, rotations, raw, raster_settings):
    """``rasterize_gaussians`` on a model's own tensors (see ``model_inputs_fit``)."""
    return _RasterizeModel.apply(xyz, means2D, dc, rest, opacity, scales, rotations, raw, raster_settings,
                                 torch.is_grad_enabled())


class GaussianRasterizer(nn.Module):
    def __init__(self, raster_settings):
        super().__init__()
        self.raster_settings = raster_settings

    def markVisible(self, positions):
        with torch.no_grad():
            rs = self.raster_settings
            pos = _f32(positions, positions.device)
            P = pos.shape[0]
            present = torch.zeros(P, dtype=torch.uint8, device=pos.device)
            view = _f32(rs.viewmatrix, pos.device)
            N.check(N.load().dmgs_mark_visible(P, N.ptr(pos), N.ptr(view), N.ptr(present),
                                               N.stream_handle(pos.device)), "dmgs_mark_visible")
            return present.bool()

    def forward(self, means3D, means2D, opacities, shs=None, colors_precomp=None, scales=None, rotations=None,
                cov3D_precomp=None):
        raster_settings = self.raster_settings
        if (shs is None and colors_precomp is None) or (shs is not None and colors_precomp is not None):
            raise Exception('Please provide excatly one of either SHs or precomputed colors!')
        if ((scales is None or rotations is None) and cov3D_precomp is None) or \
                ((scales is not None or rotations is not None) and cov3D_precomp is not None):
            raise Exception('Please provide exactly one of either scale/rotation pair or precomputed 3D covariance!')
        empty = lambda: torch.Tensor([])
        shs = empty() if shs is None else shs
        colors_precomp = empty() if colors_precomp is None else colors_precomp
        scales = empty() if scales is None else scales
        rotations = empty() if rotations is None else rotations
        cov3D_precomp = empty() if cov3D_precomp is None else cov3D_precomp
        return rasterize_gaussians(means3D, means2D, shs, colors_precomp, opacities, scales, rotations,
                                   cov3D_precomp, raster_settings)
