"""The blend kernels at the edges of their list handling, against the FP64 oracle.

The forward takes a cell's list in chunks of 1024 positions, stages 256
members at a time and keeps a segment for the backward every 64 members:
lists of no entry, one entry, around 64 and 256, and longer than a chunk; a
list cut off by saturation; more segments than the workspace has slots for.  Tolerances are those of the other parity tests
(images 1e-4, gradients 1e-3 norm-relative; 1e-5 between two groupings of the
same sums)."""
import math

import pytest
import torch

from dmgs_amd import batched as BT
from dmgs_amd import cameras as C
from dmgs_amd import scenes as S
from helpers import grad_rel_err
from oracle import raster as OR

pytestmark = pytest.mark.gpu


def _covering(n, logit, scale, seed=0):
    """n splats; of log-scale 0.5 each covers the whole view."""
    g = torch.Generator().manual_seed(seed)
    xyz = torch.rand(n, 3, generator=g) - 0.5
    dc = torch.randn(n, 1, 3, generator=g) * 0.5
    scale = torch.randn(n, 3, generator=g) * 0.1 + scale
    return S.FreeGaussians(xyz, dc, torch.randn(n, 3, 3, generator=g) * 0.1, scale, torch.randn(n, 4, generator=g),
                           logit + 0.3 * torch.randn(n, 1, generator=g), 1)


@pytest.mark.parametrize("n,logit,size,scale", [
    (1, -2.0, (16, 16), 0.5), (63, -4.0, (17, 16), 0.5), (64, -4.0, (16, 33), 0.5), (65, -4.0, (33, 17), 0.5), (128, -4.0, (16, 16), 0.5),
    (255, -4.5, (20, 20), 0.5), (256, -4.5, (20, 20), 0.5), (257, -4.5, (20, 20), 0.5), (700, -4.5, (48, 40), 0.5),
    (300, 1.0, (40, 40), 0.5),       # saturates within the first chunk
    (600, -4.5, (320, 320), 0.5),  # 400 tiles of nine segments, 1024 slots
    (1100, -4.5, (16, 16), 0.5),   # more than one chunk of a cell list
    (40, 0.0, (300, 180), -3.0)])  # most tiles, and whole cells, are empty
def test_list_edges(n, logit, size, scale):
    print(f"case: list edges n={n} logit={logit} size={size} scale={scale}", flush=True)
    m = _covering(n, logit, scale)
    cam = C.camera_at((0.3, -0.2, -4.0), *size, device="cpu")
    bg = torch.tensor([0.2, 0.5, 0.8])
    st = OR.settings_for(cam, bg.double(), 1)
    kw = dict(shs=m.get_features, scales=m.get_scaling, rotations=m.get_rotation)
    col, _, state = OR.rasterize(m.get_xyz, m.get_opacity, st, **kw)
    dL = torch.randn(col.shape, generator=torch.Generator().manual_seed(1))
    dL[:, state["ambiguous"]] = 0.0
    want = OR.rasterize_backward(state, st, m.get_xyz, dL.double(), **kw)
    params = BT.pack_model(m.to("cuda"))
    r = BT.BatchedRenderer([cam], bg, n, sh_degree=1)
    r.plan(params)
    images = r.forward(params)
    grads = r.backward(params, dL.cuda().reshape(-1).contiguous()).clone()
    ok = ~state["ambiguous"]
    err = (r.image(images, 0).cpu().double() - col).abs()[:, ok].max().item()
    assert err < 1e-4, f"image error {err}"
    got = BT.unpack_grads(grads, 4)
    o = torch.sigmoid(m._opacity.double())
    for name, ref in (("_xyz", want[0]), ("_opacity", want[4] * o * (1 - o)),
                      ("_features_dc", want[2][:, :1])):
        assert grad_rel_err(got[name], ref) < 1e-3, name
    # a second backward, and one after a forward that kept no segments
    twice = r.backward(params, dL.cuda().reshape(-1).contiguous()).clone()
    ws, r.bwd_ws = r.bwd_ws, None
    again = r.forward(params)
    assert torch.equal(again, images)
    r.bwd_ws, r._acc_clear = ws, False
    whole = r.backward(params, dL.cuda().reshape(-1).contiguous())
    assert grad_rel_err(whole, grads) < 1e-5
    assert grad_rel_err(twice, grads) < 1e-5


@pytest.mark.parametrize("n,logit,size,scale", [(1, 0.0, (17, 9), 0.5), (2, 0.0, (16, 24), 0.5), (3, 0.0, (31, 8), 0.5),
                                                (257, -4.5, (40, 40), 0.5), (300, 1.0, (33, 41), 0.5),
                                                (3000, 0.0, (352, 368), -2.5), (40, 0.0, (300, 180), -3.0)])
def test_two_work_groups_per_tile(n, logit, size, scale):
    """A forward without a backward to follow blends up to 512 tiles with two work-groups each: the same operations
    on every value as the one that keeps segments, so images, transmittances and counts are equal bit for bit."""
    print(f"case: split tiles n={n} logit={logit} size={size} scale={scale}", flush=True)
    model = _covering(n, logit, scale)
    cams = [C.camera_at((0.2, 0.1, -3.0), *size)]
    r = BT.BatchedRenderer(cams, [torch.tensor([0.1, 0.5, 0.9], device="cuda")], n, sh_degree=1)
    params = BT.pack_model(model.to("cuda"))
    r.plan(params)
    assert r.total_tiles <= 512
    got = []
    for keep in (True, False):
        if not keep:
            r.bwd_ws = None
        img = r.forward(params).clone()
        X = r.total_pixels
        T = r.state[r._offsets[3]:r._offsets[3] + 4 * X].view(torch.float32).clone()
        cnt = r.state[r._offsets[4]:r._offsets[4] + 4 * X].view(torch.int32).clone()
        got.append((img, T, cnt))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    # and twice: the halves' largest counts do not depend on an earlier forward
    assert torch.equal(r.forward(params), got[0][0])


@pytest.mark.parametrize("n,logit,size,long", [(60, 1.0, (16, 16), -1.0), (200, 0.0, (33, 41), -1.0),
                                               (400, -1.0, (120, 70), -0.5), (300, -5.4, (48, 48), -1.0),
                                               (2000, 0.0, (300, 200), -2.5)])
def test_needles_across_quadrants_and_strips(n, logit, size, long):
    """Thin splats in any direction, centres inside and outside the image: which quadrants and strips they reach
    decides what is evaluated, so a rectangle wrongly left out is missing from the image or the gradients.  Opacities
    around 1/255 included.  Tolerances of the other parity tests."""
    print(f"case: needles n={n} logit={logit} size={size} long={long}", flush=True)
    g = torch.Generator().manual_seed(3)
    xyz = (torch.rand(n, 3, generator=g) - 0.5) * 4.0
    scale = torch.tensor([long, -4.5, -4.5]) + 0.2 * torch.randn(n, 3, generator=g)
    m = S.FreeGaussians(xyz, torch.randn(n, 1, 3, generator=g) * 0.5, torch.randn(n, 3, 3, generator=g) * 0.1, scale,
                        torch.randn(n, 4, generator=g), logit + 0.3 * torch.randn(n, 1, generator=g), 1)
    cam = C.camera_at((0.3, -0.2, -4.0), *size, device="cpu")
    bg = torch.tensor([0.2, 0.5, 0.8])
    st = OR.settings_for(cam, bg.double(), 1)
    kw = dict(shs=m.get_features, scales=m.get_scaling, rotations=m.get_rotation)
    col, _, state = OR.rasterize(m.get_xyz, m.get_opacity, st, **kw)
    dL = torch.randn(col.shape, generator=torch.Generator().manual_seed(1))
    dL[:, state["ambiguous"]] = 0.0
    want = OR.rasterize_backward(state, st, m.get_xyz, dL.double(), **kw)
    params = BT.pack_model(m.to("cuda"))
    r = BT.BatchedRenderer([cam], bg, n, sh_degree=1)
    r.plan(params)
    images = r.forward(params).clone()
    grads = r.backward(params, dL.cuda().reshape(-1).contiguous())
    ok = ~state["ambiguous"]
    assert (r.image(images, 0).cpu().double() - col).abs()[:, ok].max().item() < 1e-4
    got = BT.unpack_grads(grads, 4)
    o = torch.sigmoid(m._opacity.double())
    for name, ref in (("_xyz", want[0]), ("_opacity", want[4] * o * (1 - o)), ("_features_dc", want[2][:, :1])):
        assert grad_rel_err(got[name], ref) < 1e-3, name
    r.bwd_ws = None  # without a backward to follow: two work-groups a tile
    assert torch.equal(r.forward(params), images)
