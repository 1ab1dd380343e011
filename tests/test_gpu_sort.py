"""The radix sort's scatter at the edges of its tiles (1024 and 4096 keys), of the runs of tiles that the XCDs take
(8 per round) and of its digit widths (6 and 8 ballots a key): keys and values equal torch's stable sort."""
import pytest
import torch

from dmgs_amd import _native as N

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
