"""Colours that are not finite reach only the pixels that their splats contribute to.

A splat that a pixel skips (alpha below 1/255, or behind the point where the
pixel is saturated) takes no part in it.  The pixels that some splats take
part in are found by changing their colours from 0 to 1e6 (the smallest weight,
1e-4 / 255, moves a pixel by 0.4); with colours that are not finite exactly
those pixels may change."""
import pytest
import torch

from dmgs_amd import cameras as C
from dmgs_amd import rasterizer as RZ
from dmgs_amd import scenes as S
from helpers import settings_from_cam

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,size", [("tile_lists", (150, 130)), ("kept", (150, 130)), ("halves", (150, 130)),
                                       ("whole", (400, 390))])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_only_touched_pixels(form, size, value):
    """The forms of the blend: per-tile lists; cell lists with segments kept; two work-groups a tile; one."""
    print(f"case: odd colours {form} {value}", flush=True)
    m = S.free_scene(3000, seed=5).to("cuda")
    m._opacity += 1.5  # saturated pixels in the middle
    cam = C.camera_at((0.3, 0.4, -3.2), *size)
    rs = settings_from_cam(cam, torch.tensor([0.2, 0.4, 0.6]), 0, debug=form == "tile_lists")
    odd = torch.arange(7, 3000, 211, device="cuda")
    base = torch.rand(3000, 3, generator=torch.Generator().manual_seed(1)).cuda()

    def image(x):
        colors = base.clone()
        colors[odd, :] = x
        with torch.set_grad_enabled(form in ("kept", "tile_lists")):
            return RZ.GaussianRasterizer(rs)(
                means3D=m._xyz.clone().requires_grad_(True), means2D=torch.zeros_like(m._xyz), opacities=m.get_opacity,
                colors_precomp=colors, scales=m.get_scaling, rotations=m.get_rotation)[0].detach()

    zero, large, got = image(0.0), image(1e6), image(value)
    touched = (large - zero).abs() > 0.1
    assert touched.any() and not touched.all()
    assert torch.equal(got[~touched], zero[~touched])
    assert not torch.isfinite(got[touched]).any()
