"""Batches that are never followed by a backward hold nothing for one."""
import pytest
import torch

from dmgs_amd import _native as N
from dmgs_amd import batched as BT
from dmgs_amd import cameras as C
from dmgs_amd import scenes as S
from dmgs_amd import serving as SV
from helpers import grad_rel_err


def test_forward_state_has_no_segments():
    lib = N.load()
    size = lambda T, P=1_000_000: lib.dmgs_batched_forward_state_size(2, P, T, 256 * T)
    # a tile's share of the state: its pixels' transmittance and count, its range, order, bucket and work
    per_tile = 256 * 8 + 8 + 4 + 4 + 4 + 1
    assert 0 <= size(4097) - size(4096) <= per_tile + 4 * 256
    assert 0 <= size(4096) - size(4095) <= per_tile + 4 * 256
    for P in (100, 1_000_000):
        slots = min(16384, max(1024, 2 * P // 16))
        assert lib.dmgs_batched_state_size(2, P, 4096, 256 * 4096) - size(4096, P) >= slots * 4096
    assert lib.dmgs_batched_forward_state_size(0, 10, 1, 256) == 0


@pytest.mark.gpu
def test_planned_forward_only_then_for_a_backward():
    print("case: forward-only state", flush=True)
    m = S.free_scene(2000, seed=2, sh_degree=1).to("cuda")
    params = BT.pack_model(m)
    cams = [C.camera_at((0.3, 0.2, -3.5), 130, 90), C.camera_at((2.0, 1.0, 2.5), 61, 77)]
    bg = torch.tensor([0.2, 0.5, 0.8])
    renderers = [BT.BatchedRenderer(cams, bg, 2000, sh_degree=1) for _ in range(3)]
    r, grown, counted = renderers
    r.plan(params)
    images = r.forward(params)
    dL = torch.randn(images.shape, generator=torch.Generator().manual_seed(1)).cuda()
    want = r.backward(params, dL)
    size = lambda x: x.lib.dmgs_batched_forward_state_size(x.B, x.P, x.total_tiles, x.total_pixels)
    grown.plan(params, backward=False)
    assert torch.equal(grown.forward(params), images) and grown.state.numel() == size(grown) < r.state.numel()
    grown.plan(params, K_cap=grown.K_cap)
    # the counting pass's results are still there after the state has grown
    counted.count_instances(params)
    assert counted.state.numel() == size(counted)
    counted.plan(params, K_cap=r.K_cap)
    got = counted.forward(params, stages=BT.STAGE_BINNING | BT.STAGE_BLEND)
    assert torch.equal(got, images)
    assert torch.equal(grown.forward(params), images)
    for x in (grown, counted):
        assert x.state.numel() == r.state.numel()
        assert grad_rel_err(x.backward(params, dL), want) < 1e-5
    srv = SV.RenderServer({"a": (params, 1)})
    lists = srv._lists_bytes(srv.ipp["a"] * r.total_pixels)
    assert srv.footprint("a", cams) == size(r) + 12 * r.total_pixels + lists
