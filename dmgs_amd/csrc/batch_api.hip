// C-ABI of the batched multi-view pipeline (include/dmgs.h, "batched views").
//
// B views of one scene go through one launch sequence with no host
// synchronisation: fused-activation preprocess of all views, one depth sort
// over the B*P (view, Gaussian) entries, duplication into global tile ids
// (each view owns a contiguous tile range), one stable tile sort, ranges, and
// one blend launch over every tile of every view.  The instance count stays
// on the device; buffers are sized by a capacity fixed at plan time, and the
// count is exposed so the host can detect an overflow after the fact.  The
// sequence contains only kernels (no memset / memcpy nodes), so it can be
// captured in a HIP graph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstddef>
#include <cstdio>

#include "../../include/dmgs.h"
#include "dmgs_common.h"
#include "dmgs_kernels.h"

namespace dmgs {
void set_last_error(const char* msg);
int check_view(const dmgs_settings* s, int64_t P, const float* means3D, const float* opacities, const float* shs,
               const float* colors_precomp, const float* scales, const float* rotations, const float* cov3D_precomp);
}
static_assert(sizeof(dmgs_gaussians) == 80, "dmgs_gaussians layout");
static_assert(sizeof(dmgs_gaussian_grads) == 72, "dmgs_gaussian_grads layout");

static_assert(sizeof(dmgs_view) == sizeof(dmgs::ViewDesc), "dmgs_view / ViewDesc layout");
static_assert(offsetof(dmgs_view, tile_base) == offsetof(dmgs::ViewDesc, tile_base), "dmgs_view layout");
static_assert(offsetof(dmgs_view, pixel_base) == offsetof(dmgs::ViewDesc, pixel_base), "dmgs_view layout");
static_assert(offsetof(dmgs_view, tanfovx) == offsetof(dmgs::ViewDesc, tanfovx), "dmgs_view layout");
static_assert(offsetof(dmgs_view, width) == offsetof(dmgs::ViewDesc, W), "dmgs_view layout");
static_assert(offsetof(dmgs_view, bg) == offsetof(dmgs::ViewDesc, bg), "dmgs_view layout");
static_assert(sizeof(dmgs_batch) == 104 && offsetof(dmgs_batch, capacity) == 56 && offsetof(dmgs_batch, dens) == 96,
              "dmgs_batch layout");
static_assert(offsetof(dmgs_view, cell_base) == offsetof(dmgs::ViewDesc, cell_base), "dmgs_view layout");

namespace {

int bfail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int bfail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  dmgs::set_last_error(buf);
  return code;
}

int bcheck(const char* what, hipStream_t s) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return bfail(DMGS_EHIP, "%s: %s", what, hipGetErrorString(e));
  (void)s;
  return DMGS_OK;
}

constexpr size_t kAlign = 256;
inline size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }
template <typename T>
T* at(void* base, size_t off) { return reinterpret_cast<T*>(static_cast<char*>(base) + off); }

int bits_for(uint32_t n) {
  int b = 0;
  while (b < 32 && (n >> b) != 0) ++b;
  return b;
}

// K-independent state of a batch: per-entry splats / keys / order / radii /
// scan, the depth-sort scratch, per-tile ranges and per-pixel blend state.
struct StateLayout {
  size_t splats, keys_a, keys_b, order_a, order_b, rects, rects_sorted, radii, offsets, gscratch, visible,
      status, tile_order, tile_bucket, bucket_hist, tile_work, ranges, final_T, n_contrib, tile_last,
      seg_head, seg_rec, seg_state, total;
  int seg_cap;  // slots for the list segments of the blend's backward (0: too many tiles for any)
  StateLayout(size_t N, size_t T, size_t X, bool segments = true) {
    size_t o = 0;
    splats = o; o += align_up(N * DMGS_SPLAT_F4 * 16);
    keys_a = o; o += align_up(N * 4);
    keys_b = o; o += align_up(N * 4);
    order_a = o; o += align_up(N * 4);
    order_b = o; o += align_up(N * 4);
    rects = o; o += align_up(N * 8);
    rects_sorted = o; o += align_up(N * 8);
    radii = o; o += align_up(N * 4);
    offsets = o; o += align_up(N * 4);
    gscratch = o; o += align_up(std::max(dmgs::radix_scratch_words(N), dmgs::scan_scratch_words(N)) * 4);
    visible = o; o += align_up(4);  // visible entries of the last forward (the depth sort's length)
    status = o; o += align_up(4);
    tile_order = o; o += align_up(T * 4);
    tile_bucket = o; o += align_up(T);
    tile_work = o; o += align_up(T * 4);
    bucket_hist = o; o += 512 * 4;  // directly before the ranges: the duplicate zeroes both in one run
    ranges = o; o += align_up(T * 8);
    final_T = o; o += align_up(X * 4);
    n_contrib = o; o += align_up(X * 4);
    // all that a forward without a backward touches ends here, in either form
    // slots: with half of them 60k Gaussians at 800x800 take 98 us instead of 76, 1.5M 291 instead of 203
    const size_t slots = std::min<size_t>(32768, align_up(std::max<size_t>(4096, N / 4)));  // divisible by the parts
    seg_cap = segments && T <= (size_t)dmgs::kSegmentTiles ? (int)slots : 0;
    seg_head = o; o += align_up(seg_cap ? dmgs::kSegmentParts * dmgs::kSegmentHeadStride * 4 : 0);
    tile_last = o; o += align_up(seg_cap ? T * 4 : 0);
    seg_rec = o; o += align_up((size_t)seg_cap * 16);
    seg_state = o; o += (size_t)seg_cap * 256 * 8;
    total = o;
  }
};

// Per-instance lists (tile keys and entry ids, ping-pong) and their scratch.
struct ListLayout {
  size_t tkeys_a, tkeys_b, vals_a, vals_b, scratch, chunk, total;
  explicit ListLayout(size_t K) {
    size_t o = 0;
    tkeys_a = o; o += align_up(K * 4);
    tkeys_b = o; o += align_up(K * 4);
    vals_a = o; o += align_up(K * 4);
    vals_b = o; o += align_up(K * 4);
    scratch = o; o += align_up(dmgs::radix_list_scratch_words(K) * 4);  // sort histograms
    chunk = o; o += align_up(dmgs::duplicate_scratch_words(K) * 4);  // duplicate chunk starts
    total = o;
  }
};

// A splat's tile rectangle holds 16 bits per edge, the exclusive upper one included (pack_rect): 65535 tiles a side.
bool tiles_fit_rect(int32_t W, int32_t H) { return W <= 0xFFFF * DMGS_BLOCK_X && H <= 0xFFFF * DMGS_BLOCK_Y; }

int check_batch(const dmgs_batch* b) {
  if (!b) return bfail(DMGS_EINVAL, "batch is null");
  if (b->num_views <= 0 || b->num_gaussians <= 0 || (int64_t)b->num_views * b->num_gaussians > (int64_t)0x7fffffff)
    return bfail(DMGS_EINVAL, "invalid batch: %d views x %lld Gaussians", b->num_views,
                 (long long)b->num_gaussians);
  // cell ids share a key with the 16-bit tile mask of the cell lists
  if (b->total_cells <= 0 || b->total_cells > b->total_tiles || b->total_cells > (1 << DMGS_CELL_KEY_BITS))
    return bfail(DMGS_EINVAL, "invalid cell total (at most 65536 cells)");
  if (b->capacity < 0 || b->capacity > (int64_t)0xffffffff) return bfail(DMGS_EINVAL, "invalid instance capacity");
  if (b->total_tiles <= 0 || b->total_pixels <= 0) return bfail(DMGS_EINVAL, "invalid view totals");
  if (b->cell_mode != 0 && b->cell_mode != 1) return bfail(DMGS_EINVAL, "cell_mode must be 0 or 1");
  if (b->cell_mode == 1 && (b->num_views > 16 || b->max_view_cells <= 0 || b->max_view_cells > 4096 ||
                            b->max_view_cells > b->total_cells))
    return bfail(DMGS_EINVAL, "cell_mode 1 needs at most 16 views and 1..4096 cells per view");
  if (b->sh_degree < 0 || b->sh_degree > 3) return bfail(DMGS_EINVAL, "sh_degree must be in [0, 3]");
  if (!b->views || !b->state) return bfail(DMGS_EINVAL, "views and state are required");
  if (b->dens && (reinterpret_cast<uintptr_t>(b->dens) & 3u)) return bfail(DMGS_EINVAL, "dens must be 4-byte aligned");
  const auto misaligned = [](const void* p) { return p && (reinterpret_cast<uintptr_t>(p) & 255u) != 0; };
  if (misaligned(b->state) || misaligned(b->lists) || misaligned(b->bwd_ws))
    return bfail(DMGS_EINVAL, "workspaces must be 256-byte aligned");
  return DMGS_OK;
}

struct Ctx {
  size_t N;
  StateLayout S;
  ListLayout L;
  explicit Ctx(const dmgs_batch* b, bool segments = true)
      : N((size_t)b->num_views * b->num_gaussians),
        S(N, (size_t)b->total_tiles, (size_t)b->total_pixels, segments),
        L((size_t)b->capacity), capacity((size_t)b->capacity), mode(b->cell_mode),
        local_bits(b->cell_mode == 1 ? std::max(1, bits_for((uint32_t)(b->max_view_cells - 1))) : 0),
        global_bits(std::max(1, bits_for((uint32_t)(b->total_cells - 1)))) {}
  // the depth keys also order by view (with one view plain depth bits do, at any depth)
  bool view_keys(const dmgs_batch* b) const { return mode == 1 && b->num_views > 1; }
  uint32_t* count(const dmgs_batch* b) const { return at<uint32_t>(b->state, S.offsets) + (N - 1); }
  size_t capacity;
  int mode;
  // key bits of the cell sort: the cell within the view (mode 1) or the
  // global cell id (mode 0; cell ids 0 .. total_cells - 1, so 65536 cells
  // need 16 bits and bit 16, the first tile-mask bit, stays out of the sort)
  int local_bits;
  int global_bits;
  int cell_sort_bits() const { return mode == 1 ? local_bits : global_bits; }
  // a one-pass sort (view-major lists of at most 256 cells per view, or 512 on large ones) leaves the lists in the b buffers
  bool lists_in_b() const { return mode == 1 && dmgs::radix_one_pass(capacity, local_bits); }
};

dmgs::MVArgs mv_args(const dmgs_batch* b, const Ctx& c, const float* params) {
  dmgs::MVArgs a{};
  a.P = (int)b->num_gaussians;
  a.B = b->num_views;
  a.sh_degree = b->sh_degree;
  a.scale_modifier = b->scale_modifier;
  a.views = reinterpret_cast<const dmgs::ViewDesc*>(b->views);
  a.params = params;
  a.splats = at<float4>(b->state, c.S.splats);
  a.radii = at<int32_t>(b->state, c.S.radii);
  a.rects = at<uint2>(b->state, c.S.rects);
  a.depth_keys = at<uint32_t>(b->state, c.S.keys_a);  // sorted in place into keys_a / order_a
  a.order = at<uint32_t>(b->state, c.S.order_a);
  a.view_major = c.view_keys(b) ? 1 : 0;
  a.gacc = static_cast<float*>(b->bwd_ws);
  a.dens = b->dens;
  return a;
}

dmgs::RenderArgs render_args(const dmgs_batch* b, const Ctx& c) {
  dmgs::RenderArgs r{};
  r.num_tiles = b->total_tiles;
  r.P = (uint32_t)c.N;
  r.K = (uint32_t)b->capacity;
  r.K_dev = c.count(b);
  r.views = reinterpret_cast<const dmgs::ViewDesc*>(b->views);
  r.tile_view = b->tile_view;
  r.ranges = at<uint2>(b->state, c.S.ranges);
  r.point_list = at<uint32_t>(b->lists, c.lists_in_b() ? c.L.vals_b : c.L.vals_a);
  r.list_keys = at<uint32_t>(b->lists, c.lists_in_b() ? c.L.tkeys_b : c.L.tkeys_a);
  r.splats = at<float4>(b->state, c.S.splats);
  r.final_T = at<float>(b->state, c.S.final_T);
  r.n_contrib = at<uint32_t>(b->state, c.S.n_contrib);
  r.gacc = static_cast<float*>(b->bwd_ws);
  r.tile_order = at<uint32_t>(b->state, c.S.tile_order);
  // the forward measures each tile's backward list length, for the order of a backward of whole lists
  if (b->total_tiles > dmgs::kSegmentTiles) r.tile_work = at<uint32_t>(b->state, c.S.tile_work);
  if (b->bwd_ws && c.S.seg_cap) {
    r.seg.head = at<uint32_t>(b->state, c.S.seg_head);
    r.seg.cap = c.S.seg_cap;
    r.seg.rec = at<uint4>(b->state, c.S.seg_rec);
    r.seg.state = at<float2>(b->state, c.S.seg_state);
    r.seg.tile_last = at<uint32_t>(b->state, c.S.tile_last);
  }
  return r;
}

// The visible entries, in entry order, sorted by their keys (culled entries drop out in the first pass), and
// the scan of their cell counts; with_chunks: also the duplicate's chunk table.
void order_entries(const dmgs_batch* b, const Ctx& c, bool with_chunks, hipStream_t st) {
  uint32_t* keys = at<uint32_t>(b->state, c.S.keys_a);
  uint32_t* order = at<uint32_t>(b->state, c.S.order_a);
  uint32_t* offs = at<uint32_t>(b->state, c.S.offsets);
  uint32_t* gs = at<uint32_t>(b->state, c.S.gscratch);
  uint32_t* V_dev = at<uint32_t>(b->state, c.S.visible);
  dmgs::radix_sort_entry_keys(keys, order, at<uint32_t>(b->state, c.S.keys_b), at<uint32_t>(b->state, c.S.order_b),
                              c.N, gs, st, V_dev, c.view_keys(b) ? at<uint32_t>(b->state, c.S.status) : nullptr);
  dmgs::launch_gather_rects(at<uint2>(b->state, c.S.rects), order, at<uint2>(b->state, c.S.rects_sorted), offs, c.N,
                            st, V_dev);
  if (with_chunks)
    dmgs::launch_inclusive_scan_chunks(offs, offs, c.N, gs, at<uint32_t>(b->lists, c.L.chunk), (uint32_t)b->capacity,
                                       st);
  else
    dmgs::launch_inclusive_scan(offs, offs, c.N, gs, st);
}

// The cell lists, their ranges and the blend's dispatch order.
int bin_entries(const dmgs_batch* b, const Ctx& c, bool chunks_ready, hipStream_t st) {
  const uint32_t K = (uint32_t)b->capacity;
  dmgs::DupArgs d{};
  d.P = (int)c.N;
  d.order = at<uint32_t>(b->state, c.S.order_a);
  d.offsets = at<uint32_t>(b->state, c.S.offsets);
  d.splats = at<float4>(b->state, c.S.splats);
  d.rects = at<uint2>(b->state, c.S.rects_sorted);
  d.views = reinterpret_cast<const dmgs::ViewDesc*>(b->views);
  d.per_view = (uint32_t)b->num_gaussians;
  d.tile_keys = at<uint32_t>(b->lists, c.L.tkeys_a);
  d.values = at<uint32_t>(b->lists, c.L.vals_a);
  d.K = K;
  d.K_dev = c.count(b);
  d.chunk_first = at<uint32_t>(b->lists, c.L.chunk);
  d.chunk_ready = chunks_ready;
  d.view_major = b->cell_mode == 1;
  // the duplicate also zeroes the tile-order histogram and the cell ranges (adjacent)
  d.zero = at<uint32_t>(b->state, c.S.bucket_hist);
  d.zero_n = 512 + 2 * (size_t)b->total_cells;
  // view-major lists: the duplicate also counts the first sort pass's digits
  const bool wide = d.view_major && c.local_bits == 9 && c.lists_in_b();
  const int w0 = wide ? 9 : d.view_major ? dmgs::radix_min_passes_first_width(K, c.local_bits) : -1;
  if (w0 > 0) {
    d.hist = at<uint32_t>(b->lists, c.L.scratch);
    d.hist_bits = w0;
  }
  dmgs::launch_duplicate(d, st);
  uint32_t* kb = at<uint32_t>(b->lists, c.L.tkeys_b);
  uint32_t* vb = at<uint32_t>(b->lists, c.L.vals_b);
  if (d.view_major) {  // sort the cell-within-view bits only; the view order is already there
    uint32_t* scratch = at<uint32_t>(b->lists, c.L.scratch);
    if (wide) dmgs::radix_sort_pairs_wide_digit(d.tile_keys, d.values, kb, vb, K, scratch, st, d.K_dev);
    const bool in_b = wide || dmgs::radix_sort_pairs_min_passes(d.tile_keys, d.values, kb, vb, K, c.local_bits, scratch,
                                                                st, d.K_dev, w0 > 0);
    if (in_b != c.lists_in_b()) return bfail(DMGS_EHIP, "internal: sorted list buffer mismatch");
    dmgs::launch_view_cell_ranges(in_b ? kb : d.tile_keys, K, at<uint2>(b->state, c.S.ranges), b->total_cells,
                                  d.views, st, d.K_dev, true);
  } else {
    dmgs::radix_sort_pairs(d.tile_keys, d.values, kb, vb, K, c.global_bits, at<uint32_t>(b->lists, c.L.scratch), st,
                           d.K_dev);
    dmgs::launch_tile_ranges(d.tile_keys, K, at<uint2>(b->state, c.S.ranges), b->total_cells, st, d.K_dev,
                             DMGS_CELL_KEY_MASK);
  }
  // blend dispatch order: tiles with the longest lists first
  dmgs::launch_tile_order(render_args(b, c), at<uint32_t>(b->state, c.S.tile_order),
                          at<uint8_t>(b->state, c.S.tile_bucket), at<uint32_t>(b->state, c.S.bucket_hist), st, true);
  return bcheck("batch binning", st);
}

int blend_views(const dmgs_batch* b, const Ctx& c, float* images, hipStream_t st) {
  dmgs::RenderArgs r = render_args(b, c);
  r.out_color = images;
  if (b->bwd_ws) {  // the blend work-groups also clear the backward accumulator
    r.clear = static_cast<float4*>(b->bwd_ws);
    r.clear_n = (c.N * DMGS_GACC_STRIDE + 3) / 4;  // inside the 256-byte-aligned workspace
  }
  r.clear_words = at<uint32_t>(b->state, c.S.bucket_hist);  // for the backward's tile order
  r.clear_words_n = 512;
  dmgs::launch_render_fwd(r, st);
  return bcheck("batch render forward", st);
}

// Accumulates into bwd_ws, which holds zeros on entry.
int blend_views_backward(const dmgs_batch* b, const Ctx& c, const float* dL_dimages, hipStream_t st) {
  dmgs::RenderArgs r = render_args(b, c);
  r.dL_dpix = dL_dimages;
  // re-order the tiles by the list lengths, if the forward measured them (the
  // forward blend, and then each backward blend, zero the histogram)
  r.clear_words = at<uint32_t>(b->state, c.S.bucket_hist);
  r.clear_words_n = 512;
  dmgs::launch_tile_order_bwd(r, at<uint32_t>(b->state, c.S.tile_order), at<uint8_t>(b->state, c.S.tile_bucket),
                              at<uint32_t>(b->state, c.S.bucket_hist), st, true);
  dmgs::launch_render_bwd(r, st);
  return bcheck("batch render backward", st);
}

// ---- one view over a model's own tensors ----
// Its state: the batch state of one view, then the view's record and the tile sums.
struct ViewLayout {
  int grid_x, grid_y, cells;
  StateLayout S;
  size_t record, tile_sums, counts, total;
  ViewLayout(int64_t P, int W, int H, bool keep)
      : grid_x((W + DMGS_BLOCK_X - 1) / DMGS_BLOCK_X),
        grid_y((H + DMGS_BLOCK_Y - 1) / DMGS_BLOCK_Y),
        cells(cells_along(grid_x) * cells_along(grid_y)),
        S((size_t)P, (size_t)grid_x * grid_y, (size_t)W * H, keep) {
    record = S.total;
    tile_sums = record + align_up(sizeof(dmgs::ViewDesc));
    counts = tile_sums + align_up(dmgs::kTileSums * 4);
    total = counts + align_up(8);
  }
  static int cells_along(int tiles) { return (tiles + (1 << DMGS_CELL_SHIFT) - 1) >> DMGS_CELL_SHIFT; }
};
bool view_has_cells(int32_t W, int32_t H) {
  if (W <= 0 || H <= 0 || (int64_t)W * H > (int64_t)1 << 30 || !tiles_fit_rect(W, H)) return false;
  const int64_t cx = ViewLayout::cells_along((W + DMGS_BLOCK_X - 1) / DMGS_BLOCK_X);
  const int64_t cy = ViewLayout::cells_along((H + DMGS_BLOCK_Y - 1) / DMGS_BLOCK_Y);
  return cx * cy <= 1 << DMGS_CELL_KEY_BITS;
}

dmgs_batch view_batch(const dmgs_settings* s, int64_t P, const ViewLayout& V, void* state, int64_t K, void* lists,
                      void* bwd_ws) {
  dmgs_batch b{};
  b.views = at<dmgs_view>(state, V.record);
  b.num_views = 1;
  b.num_gaussians = P;
  b.total_tiles = V.grid_x * V.grid_y;
  b.total_cells = b.max_view_cells = V.cells;
  b.total_pixels = (int64_t)s->image_width * s->image_height;
  b.capacity = K;
  b.state = state;
  b.lists = lists;
  b.bwd_ws = bwd_ws;
  b.cell_mode = V.cells <= 4096 ? 1 : 0;
  return b;
}

dmgs::ViewArgs view_args(const dmgs_settings* s, const dmgs_gaussians* g, const ViewLayout& V) {
  dmgs::ViewArgs a{};
  a.P = (int)g->count;
  a.W = s->image_width;
  a.H = s->image_height;
  a.grid_x = V.grid_x;
  a.grid_y = V.grid_y;
  a.tanfovx = s->tanfovx;
  a.tanfovy = s->tanfovy;
  a.focal_x = (float)a.W / (2.0f * s->tanfovx);
  a.focal_y = (float)a.H / (2.0f * s->tanfovy);
  a.scale_modifier = s->scale_modifier;
  a.sh_degree = s->sh_degree;
  a.sh_coeffs = g->shs ? s->sh_coeffs : 0;
  a.raw = g->raw;
  a.means3D = g->means3D;
  a.scales = g->scales;
  a.rotations = g->rotations;
  a.opacities = g->opacities;
  a.shs = g->shs;
  a.shs_rest = g->shs_rest;
  a.colors_precomp = g->colors_precomp;
  a.cov3D_precomp = g->cov3D_precomp;
  a.viewmatrix = s->viewmatrix;
  a.projmatrix = s->projmatrix;
  a.campos = s->campos;
  a.bg = s->bg;
  return a;
}

int check_gaussians(const dmgs_settings* s, const dmgs_gaussians* g, const void* state) {
  if (!g) return bfail(DMGS_EINVAL, "gaussians is null");
  const int rc = dmgs::check_view(s, g->count, g->means3D, g->opacities, g->shs, g->colors_precomp, g->scales,
                                  g->rotations, g->cov3D_precomp);
  if (rc) return rc;
  if (g->count <= 0) return bfail(DMGS_EINVAL, "no Gaussians");
  if (!view_has_cells(s->image_width, s->image_height))
    return bfail(DMGS_EINVAL, "more than 65536 cells, or 65535 tiles a side");
  if (g->raw & ~7) return bfail(DMGS_EINVAL, "invalid raw mask %d", g->raw);
  if (g->shs_rest && (!g->shs || (s->sh_coeffs != 4 && s->sh_coeffs != 9 && s->sh_coeffs != 16)))
    return bfail(DMGS_EINVAL, "shs_rest needs shs and 4, 9 or 16 coefficients");
  for (const float* p : {g->shs, g->shs_rest, g->rotations})
    if (reinterpret_cast<uintptr_t>(p) & 15u) return bfail(DMGS_EINVAL, "tensors must be 16-byte aligned");
  if (!state || (reinterpret_cast<uintptr_t>(state) & 255u))
    return bfail(DMGS_EINVAL, "state is required, 256-byte aligned");
  return DMGS_OK;
}

}  // namespace

extern "C" {

int dmgs_batched_prepare_views(dmgs_view* views, int32_t B, int32_t* total_tiles, int32_t* total_cells,
                               int32_t* max_view_cells, int64_t* total_pixels) {
  if (!views || B <= 0 || !total_tiles || !total_cells || !max_view_cells || !total_pixels)
    return bfail(DMGS_EINVAL, "bad arguments");
  int64_t tiles = 0, cells = 0, pixels = 0, max_cells = 0;
  for (int v = 0; v < B; ++v) {
    dmgs_view& d = views[v];
    if (d.width <= 0 || d.height <= 0 || !(d.tanfovx > 0.f) || !(d.tanfovy > 0.f))
      return bfail(DMGS_EINVAL, "view %d: invalid size or field of view", v);
    if (!tiles_fit_rect(d.width, d.height)) return bfail(DMGS_EINVAL, "view %d: more than 65535 tiles a side", v);
    d.focal_x = (float)d.width / (2.0f * d.tanfovx);
    d.focal_y = (float)d.height / (2.0f * d.tanfovy);
    d.grid_x = (d.width + DMGS_BLOCK_X - 1) / DMGS_BLOCK_X;
    d.grid_y = (d.height + DMGS_BLOCK_Y - 1) / DMGS_BLOCK_Y;
    d.tile_base = (int32_t)tiles;
    d.cell_base = (int32_t)cells;
    d.pixel_base = pixels;
    tiles += (int64_t)d.grid_x * d.grid_y;
    const int E = 1 << DMGS_CELL_SHIFT;
    const int64_t vc = (int64_t)((d.grid_x + E - 1) / E) * ((d.grid_y + E - 1) / E);
    cells += vc;
    max_cells = std::max(max_cells, vc);
    pixels += (int64_t)d.width * d.height;
    if (tiles > (int64_t)0x7fffffff) return bfail(DMGS_EINVAL, "too many tiles");
  }
  *total_tiles = (int32_t)tiles;
  *total_cells = (int32_t)std::min<int64_t>(cells, 0x7fffffff);
  *max_view_cells = (int32_t)std::min<int64_t>(max_cells, 0x7fffffff);
  *total_pixels = pixels;
  return DMGS_OK;
}

int dmgs_batched_tile_view(const dmgs_view* views, int32_t B, int32_t* tile_view, int32_t total_tiles) {
  if (!views || B <= 0 || !tile_view || total_tiles <= 0) return bfail(DMGS_EINVAL, "bad arguments");
  for (int v = 0; v < B; ++v) {
    const int32_t n = views[v].grid_x * views[v].grid_y;
    if (views[v].tile_base < 0 || views[v].tile_base + n > total_tiles)
      return bfail(DMGS_EINVAL, "view %d: tile range outside the total (prepare the views first)", v);
    for (int32_t t = 0; t < n; ++t) tile_view[views[v].tile_base + t] = v;
  }
  return DMGS_OK;
}

size_t dmgs_batched_state_size(int32_t B, int64_t P, int32_t total_tiles, int64_t total_pixels) {
  if (B <= 0 || P <= 0 || total_tiles <= 0 || total_pixels <= 0) return 0;
  return StateLayout((size_t)B * P, (size_t)total_tiles, (size_t)total_pixels).total;
}

size_t dmgs_batched_forward_state_size(int32_t B, int64_t P, int32_t total_tiles, int64_t total_pixels) {
  if (B <= 0 || P <= 0 || total_tiles <= 0 || total_pixels <= 0) return 0;
  return StateLayout((size_t)B * P, (size_t)total_tiles, (size_t)total_pixels, false).total;
}

size_t dmgs_batched_lists_size(int64_t capacity) {
  if (capacity <= 0) return 0;
  return ListLayout((size_t)capacity).total;
}

size_t dmgs_batched_backward_size(int32_t B, int64_t P) {
  if (B <= 0 || P <= 0) return 0;
  return align_up((size_t)B * P * DMGS_GACC_STRIDE * 4);  // whole 16-byte vectors for the forward's clear
}

int dmgs_batched_offsets(int32_t B, int64_t P, int32_t total_tiles, int64_t total_pixels, int64_t capacity,
                         size_t offsets[9]) {
  if (B <= 0 || P <= 0 || total_tiles <= 0 || total_pixels <= 0 || capacity < 0 || (int64_t)B * P > (int64_t)0x7fffffff)
    return bfail(DMGS_EINVAL, "invalid batch sizes");
  if (!offsets) return bfail(DMGS_EINVAL, "offsets is null");
  const size_t N = (size_t)B * P;
  StateLayout S(N, (size_t)total_tiles, (size_t)total_pixels);
  ListLayout Ls((size_t)capacity);
  offsets[6] = Ls.tkeys_a;  // one-pass view-major sorts leave the lists at tkeys_b / vals_b (see cell_lists)
  offsets[7] = Ls.vals_a;
  offsets[0] = S.radii;                  // (B*P) int32 radii, view-major
  offsets[1] = S.offsets + 4 * (N - 1);  // uint32 instance count of the batch
  offsets[2] = S.ranges;
  offsets[3] = S.final_T;
  offsets[4] = S.n_contrib;
  offsets[5] = S.splats;
  offsets[8] = S.status;
  return DMGS_OK;
}

int dmgs_batched_list_offsets(const dmgs_batch* b, size_t* keys, size_t* ids) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!keys || !ids) return bfail(DMGS_EINVAL, "bad arguments");
  const Ctx c(b);
  *keys = c.lists_in_b() ? c.L.tkeys_b : c.L.tkeys_a;
  *ids = c.lists_in_b() ? c.L.vals_b : c.L.vals_a;
  return DMGS_OK;
}

int dmgs_batched_cell_sort_bits(const dmgs_batch* b) {
  int rc = check_batch(b);
  if (rc) return rc;
  return Ctx(b).cell_sort_bits();
}

int dmgs_batched_forward(const dmgs_batch* b, const float* params, float* images, int32_t stages,
                         dmgs_stream_t stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!params) return bfail(DMGS_EINVAL, "params is required");
  if (stages <= 0 || (stages & ~DMGS_STAGES_ALL)) return bfail(DMGS_EINVAL, "invalid stage mask %d", stages);
  if ((stages & (DMGS_STAGE_BINNING | DMGS_STAGE_BLEND)) && (b->capacity == 0 || !b->lists || !b->tile_view))
    return bfail(DMGS_EINVAL, "binning and blend need lists, a capacity and the tile map");
  if ((stages & DMGS_STAGE_BLEND) && !images) return bfail(DMGS_EINVAL, "images is required for the blend");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const Ctx c(b);
  bool chunks_ready = false;  // the duplicate's chunk table was filled by this call's scan
  if (stages & DMGS_STAGE_GEOMETRY) {
    dmgs::MVArgs a = mv_args(b, c, params);
    a.status = at<uint32_t>(b->state, c.S.status);  // zeroed by the preprocess, set by the depth sort
    dmgs::launch_mv_preprocess(a, st);
    // the binning may follow in this call: the scan then also fills the duplicate's chunk table
    chunks_ready = (stages & DMGS_STAGE_BINNING) && b->capacity > 0 && b->lists;
    order_entries(b, c, chunks_ready, st);
    if ((rc = bcheck("batch preprocess / depth sort / scan", st))) return rc;
  }
  if (stages & DMGS_STAGE_BINNING) {
    if ((rc = bin_entries(b, c, chunks_ready, st))) return rc;
  }
  if (stages & DMGS_STAGE_BLEND) {
    if ((rc = blend_views(b, c, images, st))) return rc;
  }
  return DMGS_OK;
}

int dmgs_batched_backward(const dmgs_batch* b, const float* params, const float* dL_dimages, float* grads,
                          int32_t stages, dmgs_stream_t stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!params || !b->bwd_ws || !b->lists || !b->tile_view || b->capacity == 0)
    return bfail(DMGS_EINVAL, "params, lists, a capacity, the tile map and the backward workspace are required");
  if (stages <= 0 || (stages & ~(DMGS_STAGE_GEOMETRY | DMGS_STAGE_BLEND)))
    return bfail(DMGS_EINVAL, "invalid stage mask %d", stages);
  if ((stages & DMGS_STAGE_BLEND) && !dL_dimages) return bfail(DMGS_EINVAL, "dL_dimages is required");
  if ((stages & DMGS_STAGE_GEOMETRY) && !grads) return bfail(DMGS_EINVAL, "grads is required");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const Ctx c(b);
  dmgs::MVArgs a = mv_args(b, c, params);
  if (stages & DMGS_STAGE_BLEND) {
    if ((rc = blend_views_backward(b, c, dL_dimages, st))) return rc;
  }
  if (stages & DMGS_STAGE_GEOMETRY) {
    a.grads = grads;
    dmgs::launch_mv_geometry_bwd(a, st);
    if ((rc = bcheck("batch geometry backward", st))) return rc;
  }
  return DMGS_OK;
}

int dmgs_view_supported(int32_t width, int32_t height) { return view_has_cells(width, height) ? 1 : 0; }

size_t dmgs_view_state_size(int64_t P, int32_t width, int32_t height, int32_t keep) {
  if (P <= 0 || P > (int64_t)0x7fffffff || !view_has_cells(width, height)) return 0;
  return ViewLayout(P, width, height, keep != 0).total;
}

int dmgs_view_geometry(const dmgs_settings* s, const dmgs_gaussians* g, int32_t keep, int32_t* radii, void* state,
                       uint32_t counts[2], dmgs_stream_t stream) {
  int rc = check_gaussians(s, g, state);
  if (rc) return rc;
  if (!radii || !counts) return bfail(DMGS_EINVAL, "radii and counts are required");
  // pinned memory is written by the kernel itself: the wait ends one copy earlier (about 5 us).  Asked before the first
  // launch, so that the error which the question leaves for plain host memory is not taken for a launch's, nor clears one.
  hipPointerAttribute_t attr{};
  void* mapped = nullptr;
  const bool pinned = hipPointerGetAttributes(&attr, counts) == hipSuccess && attr.type == hipMemoryTypeHost &&
                      hipHostGetDevicePointer(&mapped, counts, 0) == hipSuccess && mapped;
  if (!pinned) (void)hipGetLastError();
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const ViewLayout V(g->count, s->image_width, s->image_height, keep != 0);
  const dmgs_batch b = view_batch(s, g->count, V, state, 0, nullptr, nullptr);
  const Ctx c(&b, keep != 0);
  dmgs::ViewArgs a = view_args(s, g, V);
  a.view = at<dmgs::ViewDesc>(state, V.record);
  a.tile_sums = at<uint32_t>(state, V.tile_sums);
  a.radii = radii;
  a.splats = at<float4>(state, c.S.splats);
  a.rects = at<uint2>(state, c.S.rects);
  a.depth_keys = at<uint32_t>(state, c.S.keys_a);
  dmgs::launch_view_preprocess(a, st);
  order_entries(&b, c, false, st);
  uint32_t* dev = pinned ? static_cast<uint32_t*>(mapped) : at<uint32_t>(state, V.counts);
  dmgs::launch_view_counts(c.count(&b), a.tile_sums, dev, st);
  if ((rc = bcheck("view preprocess / depth sort / scan", st))) return rc;
  if (!pinned && hipMemcpyAsync(counts, dev, 8, hipMemcpyDeviceToHost, st) != hipSuccess)
    return bcheck("view counts", st) ? DMGS_EHIP : bfail(DMGS_EHIP, "requesting the instance counts failed");
  return DMGS_OK;
}

int dmgs_view_counts(dmgs_stream_t stream) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (hipStreamSynchronize(st) != hipSuccess)
    return bcheck("view counts", st) ? DMGS_EHIP : bfail(DMGS_EHIP, "reading the instance counts failed");
  return DMGS_OK;
}

int dmgs_view_binning(const dmgs_settings* s, int64_t P, int32_t keep, int64_t K, void* state, void* lists,
                      dmgs_stream_t stream) {
  if (!s || P <= 0 || K <= 0 || !state || !lists || !view_has_cells(s->image_width, s->image_height))
    return bfail(DMGS_EINVAL, "invalid view");
  const ViewLayout V(P, s->image_width, s->image_height, keep != 0);
  const dmgs_batch b = view_batch(s, P, V, state, K, lists, nullptr);
  const int rc = check_batch(&b);
  return rc ? rc : bin_entries(&b, Ctx(&b, keep != 0), false, reinterpret_cast<hipStream_t>(stream));
}

int dmgs_view_blend(const dmgs_settings* s, int64_t P, int32_t keep, int64_t K, void* state, void* lists, void* bwd_ws,
                    float* out_color, dmgs_stream_t stream) {
  if (!s || P <= 0 || K <= 0 || !state || !lists || !out_color || (keep != 0) != (bwd_ws != nullptr) ||
      !view_has_cells(s->image_width, s->image_height))
    return bfail(DMGS_EINVAL, "invalid view");
  const ViewLayout V(P, s->image_width, s->image_height, keep != 0);
  const dmgs_batch b = view_batch(s, P, V, state, K, lists, bwd_ws);
  const int rc = check_batch(&b);
  return rc ? rc : blend_views(&b, Ctx(&b, keep != 0), out_color, reinterpret_cast<hipStream_t>(stream));
}

int dmgs_view_blend_backward(const dmgs_settings* s, int64_t P, int64_t K, void* state, void* lists, void* bwd_ws,
                             const float* dL_dout, dmgs_stream_t stream) {
  if (!s || P <= 0 || K <= 0 || !state || !lists || !bwd_ws || !dL_dout ||
      !view_has_cells(s->image_width, s->image_height))
    return bfail(DMGS_EINVAL, "invalid view");
  const ViewLayout V(P, s->image_width, s->image_height, true);
  const dmgs_batch b = view_batch(s, P, V, state, K, lists, bwd_ws);
  const int rc = check_batch(&b);
  return rc ? rc : blend_views_backward(&b, Ctx(&b), dL_dout, reinterpret_cast<hipStream_t>(stream));
}

int dmgs_sh_sigmoid(int64_t n, int32_t coeffs, int32_t degree, int32_t color_major, const float* feats,
                    const float* xyz, const float* campos, float* colors, const float* dL_dcolors, float* dL_dfeats,
                    float* dL_dxyz, dmgs_stream_t stream) {
  if (n < 0 || n > (int64_t)0x7fffffff - 256) return bfail(DMGS_EINVAL, "invalid n");
  if ((coeffs != 1 && coeffs != 4 && coeffs != 9 && coeffs != 16) || degree < 0 || degree > 3 ||
      (degree + 1) * (degree + 1) > coeffs)
    return bfail(DMGS_EINVAL, "degree %d needs 1, 4, 9 or 16 coefficients, at least (degree + 1)^2", degree);
  if (n == 0) return DMGS_OK;
  if (!feats || !xyz || !campos || !colors || (dL_dcolors && (!dL_dfeats || !dL_dxyz)))
    return bfail(DMGS_EINVAL, "null pointer");
  if ((reinterpret_cast<uintptr_t>(feats) | reinterpret_cast<uintptr_t>(dL_dfeats)) & 15u)
    return bfail(DMGS_EINVAL, "features must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dmgs::ShSigmoidArgs a{(int)n, degree, feats, xyz, campos, colors, dL_dcolors, dL_dfeats, dL_dxyz};
  dmgs::launch_sh_sigmoid(a, coeffs, color_major != 0, dL_dcolors != nullptr, st);
  return bcheck("sh sigmoid", st);
}

int dmgs_view_geometry_backward(const dmgs_settings* s, const dmgs_gaussians* g, const int32_t* radii,
                                const void* bwd_ws, const dmgs_gaussian_grads* d, dmgs_stream_t stream) {
  int rc = check_gaussians(s, g, bwd_ws);
  if (rc) return rc;
  if (!radii || !d || !d->means2D || !d->means3D || !d->opacities || (g->shs && !d->shs) ||
      (g->shs_rest && !d->shs_rest) || (g->scales && (!d->scales || !d->rotations)))
    return bfail(DMGS_EINVAL, "missing gradients");
  for (const float* p : {d->shs, d->shs_rest, d->rotations})
    if (reinterpret_cast<uintptr_t>(p) & 15u) return bfail(DMGS_EINVAL, "gradients must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const ViewLayout V(g->count, s->image_width, s->image_height, true);
  dmgs::ViewArgs a = view_args(s, g, V);
  a.radii = const_cast<int32_t*>(radii);
  a.gacc = static_cast<const float*>(bwd_ws);
  a.dL_dmeans2D = d->means2D;
  a.dL_dmeans3D = d->means3D;
  a.dL_dopacity = d->opacities;
  a.dL_dsh = d->shs;
  a.dL_dsh_rest = d->shs_rest;
  a.dL_dcolors = d->colors;
  a.dL_dcov3D = d->cov3D;
  a.dL_dscales = d->scales;
  a.dL_drotations = d->rotations;
  dmgs::launch_view_geometry_bwd(a, st);
  return bcheck("view geometry backward", st);
}

}  // extern "C"
