"""The radix sort's scatter at the edges of its tiles (1024 and 4096 keys), of the runs of tiles that the XCDs take
(8 per round) and of its digit widths (6, 8 and 9 ballots a key): keys and values equal torch's stable sort."""
import pytest
import torch

from dmgs_amd import _native as N
from dmgs_amd import batched as BT
from dmgs_amd import cameras as C
from dmgs_amd import scenes as S

pytestmark = pytest.mark.gpu
LARGE = 4 << 20  # from here on a tile holds 4096 keys


@pytest.mark.parametrize("n,bits", [(1, 1), (63, 5), (65, 8), (1023, 12), (1024, 13), (1025, 16), (7 * 1024 + 1, 9),
                                    (8 * 1024 + 1, 17), (9 * 1024, 32), (100_003, 10), (LARGE - 1, 11),
                                    (LARGE, 12), (LARGE + 1, 13), (LARGE + 7 * 4096 + 65, 32)])
def test_sort_pairs_tile_edges(n, bits):
    print(f"case: sort n={n} bits={bits}", flush=True)
    g = torch.Generator().manual_seed(n + bits)
    k = torch.randint(0, 1 << bits, (n,), generator=g, dtype=torch.int64)
    if n > 100:
        k[n // 3:n // 2] = k[n // 3]  # a long run of one digit
    v = torch.randperm(n, generator=g).to(torch.int32)
    to32 = lambda t: torch.where(t >= 1 << 31, t - (1 << 32), t).to(torch.int32)
    k0, v0 = to32(k).cuda(), v.cuda()
    k1, v1 = torch.empty_like(k0), torch.empty_like(v0)
    lib = N.load()
    scratch = torch.empty(lib.dmgs_sort_scratch_size(n), dtype=torch.uint8, device="cuda")
    N.check(lib.dmgs_sort_pairs(N.ptr(k0), N.ptr(v0), N.ptr(k1), N.ptr(v1), n, bits, N.ptr(scratch),
                                N.stream_handle(k0.device)), "dmgs_sort_pairs")
    order = torch.sort(k, stable=True).indices
    assert torch.equal(k0.cpu(), to32(k[order])) and torch.equal(v0.cpu(), v[order])


@pytest.mark.parametrize("P,sizes", [(3000, [(1100, 1000), (64, 64)]), (20000, [(1920, 1080)]),
                                     (20000, [(1088, 960), (2048, 1024), (33, 17)]), (700_000, [(1600, 900)] * 3)])
def test_wide_digit_lists_equal_two_passes(P, sizes):
    """Cell lists of views of 257 to 512 cells: one pass of 512 digits (capacities from 4 Mi) equals two passes."""
    print(f"case: wide digit P={P} sizes={sizes}", flush=True)
    model = S.free_scene(P, seed=6, layout="mixture")
    cams = [C.camera_at((0.3 * k, 0.2, -4.0), w, h) for k, (w, h) in enumerate(sizes)]
    r = BT.BatchedRenderer(cams, [torch.zeros(3, device="cuda")] * len(cams), P, sh_degree=3, cell_mode=1)
    params = BT.pack_model(model.to("cuda"))
    K = r.count_instances(params)
    got = []
    for cap in (max(K, LARGE), min(K, LARGE - 1)):
        r.plan(params, K_cap=cap)
        images = r.forward(params)
        got.append([t.cpu() for t in r.cell_lists()] + [images.cpu()])
    if K >= LARGE:  # a truncated list cannot be compared; the order can
        assert P == 700_000
        ranges, keys, ids = got[0][:3]
        k = keys.long() & 0xFFFF
        cell, view = k & 0xFFF, k >> 12
        pos = torch.arange(k.numel())
        assert torch.all(cell[1:] >= cell[:-1]) and torch.all((cell[1:] > cell[:-1]) | (view[1:] >= view[:-1]))
        base = torch.tensor([r.views[v].cell_base for v in range(r.B)])
        same = (cell[1:] == cell[:-1]) & (view[1:] == view[:-1])
        first = torch.cat([torch.zeros(1, dtype=torch.long), pos[1:][~same]])
        assert torch.equal(ranges[base[view[first]] + cell[first], 0].long(), first)
    else:
        for a, b in zip(*got):
            assert torch.equal(a, b)


@pytest.mark.parametrize("P,scale,cap", [(1, -2.0, None), (300, -1.0, None), (5000, -3.5, 511), (5000, -3.5, 512),
                                         (5000, -3.5, 513), (5000, -3.5, (1 << 20) - 1), (5000, -3.5, 1 << 20),
                                         (5000, -3.5, LARGE - 1), (5000, -3.5, LARGE), (40, 1.5, None)])
def test_duplicate_chunk_sizes(P, scale, cap):
    """The instances of each output chunk size (512, 1024 and 4096 slots), full, cut off and mostly empty: for every
    capacity the lists are the first `capacity` instances in depth order, sorted by cell."""
    print(f"case: duplicate P={P} scale={scale} capacity={cap}", flush=True)
    model = S.free_scene(P, seed=P)
    model._scaling = model._scaling + 3.5 + scale
    r = BT.BatchedRenderer([C.camera_at((0.3, 0.2, -4.0), 640, 400)], [torch.zeros(3, device="cuda")], P, sh_degree=3,
                           cell_mode=1)
    params = BT.pack_model(model.to("cuda"))
    K = r.count_instances(params)
    assert K > 0
    r.plan(params, K_cap=8 * LARGE // 4)  # 4096-slot chunks, all instances
    r.forward(params)
    _, keys, ids = r.cell_lists()
    assert keys.numel() == K
    cap = cap or K
    r.plan(params, K_cap=cap)
    r.forward(params)
    ranges, k2, i2 = r.cell_lists()
    if cap >= K:
        assert torch.equal(keys, k2) and torch.equal(ids, i2)
    else:  # a prefix in depth order: a subset of every cell's list, in its order
        assert k2.numel() == cap
        full = list(zip((keys & 0xFFFF).tolist(), ids.tolist()))
        place = {e: n for n, e in enumerate(full)}
        at = [place[e] for e in zip((k2 & 0xFFFF).tolist(), i2.tolist())]
        assert at == sorted(at) and len(set(at)) == cap


@pytest.mark.parametrize("size", [(16, 16), (512, 512), (1024, 1024), (1040, 1008), (1025, 1024)])
def test_tile_order_is_a_permutation_by_length(size):
    """1, 1024, 4096 and 4095 tiles in one launch, 4160 in two: every tile once, longest lists first."""
    print(f"case: tile order {size}", flush=True)
    P = 4000
    r = BT.BatchedRenderer([C.camera_at((0.3, 0.2, -4.0), *size)], [torch.zeros(3, device="cuda")], P, sh_degree=0)
    params = BT.pack_model(S.free_scene(P, seed=2, sh_degree=0).to("cuda"))
    r.plan(params)
    images = r.forward(params).clone()
    T = r.total_tiles
    gx, cx = (size[0] + 15) // 16, ((size[0] + 15) // 16 + 3) // 4
    ranges = r.cell_lists()[0].long()
    length = ranges[:, 1] - ranges[:, 0]
    t = torch.arange(T)
    cost = length[(t // gx // 4) * cx + t % gx // 4].clamp(min=0).double()
    bucket = torch.where(cost > 0, 254 - (8 * torch.log2(cost.clamp(min=1))).floor().clamp(max=254), 255.0)
    # the order lies before the range table in the state: the one run of T words that is a permutation
    words = r.state[:r._offsets[2]].view(torch.int32).cpu()
    found = 0
    for at in range(0, words.numel() - T + 1, 64):  # sub-buffers are 256-byte aligned
        o = words[at:at + T].long()
        if int(o[0]) < T and torch.equal(torch.sort(o).values, t):
            b = bucket[o]
            if bool((b[1:] >= b[:-1] - 1).all()):  # log2 rounds either way at a bucket's edge
                found += 1
    assert found >= 1
    assert torch.isfinite(images).all()
