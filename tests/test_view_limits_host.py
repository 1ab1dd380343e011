"""Limits of the cell-list route, on the host (nothing is launched)."""
import ctypes

import pytest

from dmgs_amd import _native as N

MAX_SIDE = 65535 * 16  # a splat's tile rectangle holds 16 bits per edge, the exclusive upper one included


@pytest.mark.parametrize("w,h,fits", [
    (MAX_SIDE, 16, True), (16, MAX_SIDE, True), (MAX_SIDE + 1, 16, False), (16, MAX_SIDE + 1, False),
    (2097152, 16, False),  # 32768 cells, but 131072 tiles in a row
    (16384, 16384, True), (16385, 16384, False), (1, 1, True), (0, 16, False), (16, -1, False)])
def test_sizes_with_cell_lists(w, h, fits):
    lib = N.load()
    assert lib.dmgs_view_supported(w, h) == int(fits)
    assert (lib.dmgs_view_state_size(10, w, h, 0) > 0) == fits


@pytest.mark.parametrize("w,h,ok", [(MAX_SIDE, 16, True), (MAX_SIDE + 1, 16, False), (16, MAX_SIDE + 1, False)])
def test_batched_views_refuse_what_a_rectangle_cannot_hold(w, h, ok):
    v = (N.DmgsView * 1)()
    v[0].width, v[0].height, v[0].tanfovx, v[0].tanfovy = w, h, 0.5, 0.5
    tt, tc, mc, tp = N.c_int32(0), N.c_int32(0), N.c_int32(0), N.c_int64(0)
    rc = N.load().dmgs_batched_prepare_views(v, 1, ctypes.byref(tt), ctypes.byref(tc), ctypes.byref(mc), ctypes.byref(tp))
    assert rc == (0 if ok else -1)
    assert ok or "tiles a side" in N.last_error()


def test_list_sizes_do_not_fall():
    """Memory sized for one capacity serves every smaller one, whose blocks and chunks may be smaller."""
    lib = N.load()
    at = sorted({e + d for e in (1, 1 << 10, 1 << 20, 4 << 20, 6 << 20, 16 << 20) for d in (-1, 0, 1, 300, 5000)} - {0})
    for size in (lib.dmgs_batched_lists_size, lib.dmgs_binning_workspace_size):
        sizes = [size(k) for k in at]
        assert sizes == sorted(sizes)
    states = [lib.dmgs_batched_forward_state_size(1, p, 16, 4096) for p in at]
    assert states == sorted(states)
