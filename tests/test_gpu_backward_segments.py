"""The blend backward in list segments against the walk of whole lists, bit for bit.

A batch of at most 4096 tiles walks each tile's list in segments of 64
members, each from the state that a pass over the list from the back leaves
for it; a larger batch walks the lists whole.  A view's gradient is the same
number either way, not only to rounding: scales and rotations magnify the last
bits.  The large batch is the small one with a larger second view, whose image
gradient is zero, so that nothing else differs.  One tile has an image
gradient, so that the tiles' atomic additions have no order to differ in.  The
two forwards (two work-groups a tile, and one) are compared in passing."""
import pytest
import torch

from dmgs_amd import batched as BT
from dmgs_amd import cameras as C
from dmgs_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,logit,dist,size,scale,tile", [
    (64, -4.0, 4.0, (16, 16), 0.5, (0, 0)), (65, -4.0, 4.0, (16, 16), 0.5, (0, 0)), (129, -4.0, 4.0, (15, 13), 0.5, (0, 0)),
    (700, -4.5, 4.0, (16, 16), 0.5, (0, 0)),
    (1025, -4.5, 4.0, (16, 16), 0.5, (0, 0)),       # more than one chunk of a list
    (400, 1.0, 4.0, (16, 16), 0.5, (0, 0)),         # saturates
    (3000, -1.0, 1.2, (16, 16), -4.0, (0, 0)),      # small splats: quadrants and pixels skip most of them
    (17500, -4.6, 1.2, (16, 16), -4.0, (0, 0)),     # more boundaries than a tile keeps
    (9000, -1.0, 1.2, (70, 64), -4.5, (1, 2)),      # a few members in each chunk
    (9000, -1.0, 1.2, (70, 64), -4.5, (4, 1)),      # partly outside the image
    (2000, -5.2, 4.0, (320, 320), 0.5, (3, 7)),     # 400 tiles share 4096 slots: longer segments
    (2000, -5.2, 4.0, (320, 320), 0.5, (10, 10))])
def test_segments_equal_whole_lists(n, logit, dist, size, scale, tile):
    print(f"case: segments n={n} logit={logit} dist={dist} size={size} scale={scale} tile={tile}", flush=True)
    g = torch.Generator().manual_seed(n)
    m = S.FreeGaussians(torch.rand(n, 3, generator=g) - 0.5, torch.randn(n, 1, 3, generator=g) * 0.5,
                        torch.randn(n, 3, 3, generator=g) * 0.1, torch.randn(n, 3, generator=g) * 0.1 + scale,
                        torch.randn(n, 4, generator=g), logit + 0.3 * torch.randn(n, 1, generator=g), 1)
    params = BT.pack_model(m.to("cuda"))
    bg = torch.tensor([0.2, 0.5, 0.8])
    eye = (0.05, -0.04, -dist)
    W, H = size
    dL = torch.zeros(3, H, W)
    x, y = 16 * tile[0], 16 * tile[1]
    dL[:, y:y + 16, x:x + 16] = torch.randn(dL[:, y:y + 16, x:x + 16].shape, generator=g)
    got = []
    for other in ((16, 16), (1040, 1040)):
        r = BT.BatchedRenderer([C.camera_at(eye, *size), C.camera_at(eye, *other)], bg, n, sh_degree=1)
        assert r.total_tiles <= 512 or r.total_tiles > 4096
        r.plan(params)
        images = r.forward(params)
        X = W * H
        state = [r.state[o:o + 4 * X].clone() for o in r._offsets[3:5]]  # transmittances, counts
        dL_all = torch.zeros_like(images)
        dL_all[:3 * X] = dL.reshape(-1).cuda()
        for _ in range(2):  # the second one from the states of the first
            grads = r.backward(params, dL_all).clone()
            got.append([images[:3 * X].clone(), *state, grads])
    if n == 17500:
        assert state[1].view(torch.int32).max() > 64 * 257
    assert got[0][3].abs().max() > 0
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert torch.equal(a, b), (a != b).sum().item()
