"""The cell-list engine against the per-tile lists, which share neither its lists nor their sorts.

``render`` and the batched engine run the same duplicate, cell sort and blend
kernels, so one checked against the other would not show a fault of both.
``debug`` renders with the reference's per-tile lists: the comparisons of the
batched engine's tests are repeated with those, and single views with the
forms that only large images or long lists take."""
import functools

import pytest
import torch

import test_gpu_batched as TB
from dmgs_amd import cameras as C
from dmgs_amd import rasterizer as RZ
from dmgs_amd import scenes as S
from dmgs_amd.gaussian_renderer import PipelineParams, render
from helpers import grad_rel_err, settings_from_cam

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("test", [
    functools.partial(TB.test_batched_matches_single_view, 20000, [(128, 96), (200, 200), (160, 90)]),
    functools.partial(TB.test_batched_matches_single_view, 8000, [(48, 40), (40, 48), (64, 32)] * 6 + [(24, 24), (56, 40)]),
    functools.partial(TB.test_batched_lower_sh_degrees, 1), TB.test_batched_active_degree_below_model_degree,
    TB.test_batched_scale_modifier, TB.test_huge_splats_cover_every_cell,
    TB.test_batched_matches_single_view_at_large_sort_size, TB.test_densification_stats_match_per_view_consumer,
    TB.test_65536_cells_keep_one_run_per_cell], ids=lambda t: getattr(t, "func", t).__name__[5:])
def test_batched_against_tile_lists(test, monkeypatch):
    monkeypatch.setattr(TB, "PipelineParams", lambda: PipelineParams(debug=True))
    test()


@pytest.mark.parametrize("P,size,scale,logit,least", [
    (30000, (1040, 1025), 0.0, 0.0, 0),           # 4225 tiles: nothing kept, two launches for their order
    (13000, (1600, 900), 3.5, -3.0, 4 << 20),     # 375 cells and long lists: one sort pass of 512 digits
    (4000, (4224, 4160), 0.5, 0.0, 0)])           # 4290 cells: global cell lists
def test_view_against_tile_lists(P, size, scale, logit, least):
    """Radii and images bit for bit; gradients within 1e-5, two orders of the same sums."""
    print(f"case: view against tile lists P={P} size={size}", flush=True)
    parts = [p.cuda() for p in S.free_scene(P, seed=6, sh_degree=1).parameters()]
    parts[3] += scale
    parts[5] += logit
    cam, bg = C.camera_at((0.4, 0.3, -4.0), *size), torch.tensor([0.1, 0.6, 0.3])
    g = torch.randn(3, size[1], size[0], generator=torch.Generator().manual_seed(1)).cuda()
    got = []
    for debug in (False, True):
        m = S.FreeGaussians(*[p.clone() for p in parts], sh_degree=1).requires_grad_(True)
        out = render(cam, m, PipelineParams(debug=debug), bg.cuda())
        out["render"].backward(g)
        got.append((out["render"].detach(), out["radii"], [out["viewspace_points"].grad] + [p.grad for p in m.parameters()]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    for a, b in zip(got[0][2], got[1][2]):
        assert b.any() and grad_rel_err(a, b) < 1e-5
    if least:
        t = dict(means3D=m._xyz.detach(), shs=m.get_features.detach(), opacities=m.get_opacity.detach(),
                 scales=m.get_scaling.detach(), rotations=m.get_rotation.detach())
        assert RZ.view_forward(t, 4, 0, settings_from_cam(cam, bg, 1), True)[2]["cells"] >= least
