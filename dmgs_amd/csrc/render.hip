// Front-to-back alpha blending (forward) and its reverse-traversal backward
// for gfx950.
//
// Semantics follow the reference renderer [U] (diff-gaussian-rasterization,
// called from gaussian_renderer/__init__.py:86-94): per pixel, in sorted
// order, power = -1/2 (a dx^2 + c dy^2) - b dx dy, skip if power > 0,
// alpha = min(0.99, o exp(power)), skip if alpha < 1/255, stop (without
// adding) once T (1 - alpha) < 1e-4, C += c alpha T; output C + T bg.
//
// Forward (render_fwd_quads_kernel): one 256-lane work-group per 16x16 binning tile, each of its four waves
// owning one 8x8 quadrant, one pixel per lane.  Backward (render_bwd_strips_kernel): one wave per tile, or per
// segment of a tile's list, each lane owning four pixels.
//
// Backward: the list is walked from the back, starting at the largest
// n_contrib of the tile (entries behind every pixel's last contributor
// cannot contribute), transmittance is recomputed (times 1 / (1 - alpha), one
// reciprocal) instead of being stored, and the wave sums its 9 per-splat
// partial gradients into a set of LDS accumulators, flushed with one global
// atomic per (splat, value) and tile.
//
// Several views in one launch: a global tile id indexes the ranges; the view
// table gives each tile's image size, background and packed output offset.
//
// List segments.  A lone wave takes 400 ns per (tile, splat) in the backward (a chain of dependent
// operations), so a launch of few tiles with long lists (a 200x200 view: 169 tiles, up to 900 entries
// walked) takes as long as its longest list: 350 us.  With at most kSegmentTiles tiles a pass of its own
// (render_bwd_chain_kernel) therefore first walks the lists for the pixels' recursion alone, a quarter of the
// work a splat and one pixel a lane, and leaves its state at every 64th member, so that every 64-member
// segment is a work-group of the backward proper.  The pass has the forward's bound and takes as long as it.
// The recursion is the backward's own, from final_T with the same reciprocals in the same order: each
// (tile, splat) sum is the same to the last bit with segments, however many slots there are, as without.
// (States that the forward leaves as it goes by cost no pass, but its transmittances are other roundings of
// the same products: gradients of scales and rotations, small differences of these sums, moved by up to 2e-3
// of their rms.)  Slots are 2 KB.
// Forward, pass and backward of one view, us, whole lists and segments (MI355X): 10k Gaussians at 200x200
// 36+353 and 36+51+38, 1M at 800x800 53+196 and 53+52+92, 491k face-bound at 800x800 207+1288 and 207+222+178.
#include "dmgs_common.h"
#include "dmgs_kernels.h"

namespace dmgs {

// The blend evaluates alpha = o exp(power) as o exp2(p) with p = log2(e) power,
// from the conic scaled once per staged splat: q = log2(e) (-a/2, -b, -c/2).
constexpr float kLog2e = 1.44269504088896341f;

// A staged splat is three 16-byte fields, all indexed alike: one address register serves every field (fixed
// offsets between them).  The two kernels pair the values differently: the forward reads whole fields (ten
// values in two 16-byte reads and one of 8), the backward the narrow parts it needs next.
struct StagedSplat {
  float x, y;            // pixel position
  float qx, qy, qz, o;   // scaled conic, opacity
  float r, g, b;
  uint32_t pos, mask, id;  // list position, reach mask (reach_mask), splat id
};
// In a forward mask: the colour is not finite (see render_fwd_quads_kernel).
constexpr uint32_t kOddColor = 16u;
template <int SLOTS>
struct FwdSplats {
  float4 xyq[SLOTS];   // x, y, q.x, q.y
  float4 qorg[SLOTS];  // q.z, opacity, red, green
  float4 bpmi[SLOTS];  // blue, position, mask, id
  __device__ __forceinline__ void put(int j, const StagedSplat& s) {
    xyq[j] = make_float4(s.x, s.y, s.qx, s.qy);
    qorg[j] = make_float4(s.qz, s.o, s.r, s.g);
    const bool odd = s.r * 0.f + s.g * 0.f + s.b * 0.f != 0.f;  // NaN unless all three are finite
    bpmi[j] = make_float4(s.b, __uint_as_float(s.pos), __uint_as_float(s.mask | (odd ? kOddColor : 0u)), __uint_as_float(s.id));
  }
  __device__ __forceinline__ uint32_t mask(int j) const { return __float_as_uint(bpmi[j].z); }
  __device__ __forceinline__ uint32_t pos(int j) const { return __float_as_uint(bpmi[j].y); }
};
template <int SLOTS>
struct BwdSplats {
  float4 xym[SLOTS];     // x, y, mask, position
  float4 qo[SLOTS];      // scaled conic, opacity
  float4 rgb_id[SLOTS];  // r, g, b, id
  __device__ __forceinline__ void put(int j, const StagedSplat& s) {
    xym[j] = make_float4(s.x, s.y, __uint_as_float(s.mask), __uint_as_float(s.pos));
    qo[j] = make_float4(s.qx, s.qy, s.qz, s.o);
    rgb_id[j] = make_float4(s.r, s.g, s.b, __uint_as_float(s.id));
  }
  __device__ __forceinline__ uint32_t mask(int j) const { return __float_as_uint(xym[j].z); }
  __device__ __forceinline__ uint32_t pos(int j) const { return __float_as_uint(xym[j].w); }
  __device__ __forceinline__ uint32_t id(int j) const { return __float_as_uint(rgb_id[j].w); }
};

// The element of an LDS array at a byte offset.
template <typename T, int N>
__device__ __forceinline__ T lds_at(const T (&a)[N], uint32_t byte_offset) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(&a[0]) + byte_offset);
}

// Which pixel rectangles of the work-group a splat can reach.  A splat passes
// the alpha test only inside the ellipse  d^T Q d <= tau,  tau = 2 ln(255 o)
// (o exp(-d^T Q d / 2) >= 1/255, Q the conic).  Staging tests that ellipse
// against each rectangle of pixel centres a wave (or a strip of the tile)
// covers and keeps one bit per rectangle; a wave skips the splat when its
// bit is clear: no pixel there could pass the alpha test, so results are
// unchanged.  Margins (rectangle +0.01 px, tau x 1.001 + 0.001, and 1e-6 of the
// form's terms at the work-group's far edges, which bounds what rounding adds to
// it here and in a pixel) keep the test conservative.
struct PixelRects {  // four rectangles of w x h pixels, `cols` (1 or 2) to a row, the first at (x0, y0)
  float x0, y0, w, h;
  int cols;
};

// Per rectangle: the minimum over it of q(d) = a dx^2 + 2 b dx dy + c dy^2, d = p - centre, against t.  q grows along
// every ray from the centre (or is negative on all of it), so what counts are the edges that face the centre: at most
// one vertical and one horizontal, each with its one-dimensional minimiser clamped to the edge.  Where the centre
// lies between two edges the line through it stands in for them, whose point is in the rectangle too; for a
// rectangle that holds the centre that is the centre.  (An approximate reciprocal only moves the edge point off the
// minimiser, which raises the value found by far less than the margins.)  Rectangles side by side share a row's or
// column's terms, and the logarithm is the hardware's: against four edges of each rectangle behind a branch, 158 vector
// instructions less per staged splat in the forward's code and 129 in the backward's.  Issued on 8 views of 800x800 of
// 1M Gaussians 202.5M -> 189.8M in the forward, 6.4M fewer in the backward; one 333x251 view of 500k, near, 319 -> 303 us.
template <int NX, int NY>
__device__ __forceinline__ uint32_t reach_rects(float cx, float cy, float a, float b, float c, float t,
                                                const PixelRects& rr) {
  constexpr float m = 0.01f;
  const float ia = __builtin_amdgcn_rcpf(a), ic = __builtin_amdgcn_rcpf(c);
  const float b2 = b + b, to_y = -b * ic, to_x = -b * ia;
  const float ox = rr.x0 - cx, oy = rr.y0 - cy;
  float xl[NX], xh[NX], ey_at[NX], xb[NX], xx[NX];  // of a column: its edges, and the terms of the edge that counts
  float yl[NY], yh[NY], ex_at[NY], yb[NY], yy[NY];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    xl[i] = ox + (i ? rr.w * (float)i - m : -m);
    xh[i] = ox + (rr.w * (float)(i + 1) - 1.0f + m);
    const float e = __builtin_amdgcn_fmed3f(xl[i], 0.f, xh[i]);
    ey_at[i] = to_y * e;
    xb[i] = b2 * e;
    xx[i] = a * e * e;
  }
#pragma unroll
  for (int j = 0; j < NY; ++j) {
    yl[j] = oy + (j ? rr.h * (float)j - m : -m);
    yh[j] = oy + (rr.h * (float)(j + 1) - 1.0f + m);
    const float e = __builtin_amdgcn_fmed3f(yl[j], 0.f, yh[j]);
    ex_at[j] = to_x * e;
    yb[j] = b2 * e;
    yy[j] = c * e * e;
  }
  const float fx = fmaxf(fabsf(xl[0]), fabsf(xh[NX - 1])), fy = fmaxf(fabsf(yl[0]), fabsf(yh[NY - 1]));
  t = fmaf(1e-6f, fmaf(a * fx, fx, c * fy * fy), t);
  uint32_t mask = 0;
#pragma unroll
  for (int j = 0; j < NY; ++j) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const float dy = __builtin_amdgcn_fmed3f(yl[j], ey_at[i], yh[j]);
      const float dx = __builtin_amdgcn_fmed3f(xl[i], ex_at[j], xh[i]);
      const float q = fminf(fmaf(dy, fmaf(c, dy, xb[i]), xx[i]), fmaf(dx, fmaf(a, dx, yb[j]), yy[j]));
      mask |= q > t ? 0u : 1u << (j * NX + i);
    }
  }
  return mask;
}

__device__ __forceinline__ uint32_t reach_mask(float cx, float cy, float a, float b, float c, float o,
                                               const PixelRects& rr) {
  const float t = fmaf(1.001f * 1.3862943611f, __builtin_amdgcn_logf(255.0f * o), 0.001f);  // tau from a log2
  const uint32_t mask =
      rr.cols == 2 ? reach_rects<2, 2>(cx, cy, a, b, c, t, rr) : reach_rects<1, 4>(cx, cy, a, b, c, t, rr);
  if (!(255.0f * o > 1.0f)) return 0u;  // alpha never reaches the threshold
  return (a > 0.0f) & (c > 0.0f) ? mask : 0xFu;
}

// p = log2(e) power = (q.x dx) dx + dy (q.y dx + q.z dy) for power = -1/2 (a dx^2
// + c dy^2) - b dx dy.  The dx terms depend only on the splat and the pixel
// column, so a lane owning several pixels of one column forms them once
// (power_dx).  The rounding sequence is fixed (explicit products, no compiler
// contraction), so every kernel variant, and the backward's recomputation,
// gets bit-identical values.
struct PowerDx {
  float xx, xy;  // q.x dx dx, q.y dx
};
__device__ __forceinline__ PowerDx power_dx(float qx, float qy, float dx) {
  return {__fmul_rn(__fmul_rn(qx, dx), dx), __fmul_rn(qy, dx)};
}
__device__ __forceinline__ float power_at(const PowerDx& d, float qz, float dy) {
  return fmaf(fmaf(qz, dy, d.xy), dy, d.xx);
}
// exp2 on the hardware exponential (one instruction)
__device__ __forceinline__ float splat_exp2(float p) { return __builtin_amdgcn_exp2f(p); }

#define DMGS_DPP_ADD(v, ctrl) ((v) + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), (ctrl), 0xF, 0xF, true)))

// Sums over a one-wave work-group of eight per-lane values, through LDS: each
// lane stores its values (red[q][lane]); lane (row r, row position p) then adds
// value 2r + (p >> 3) of the eight lanes 8 (p & 7) .. 8 (p & 7) + 7 (two 16-byte
// reads, seven adds), and two quad butterflies plus a shift by four lanes leave
// the sum over all 64 lanes in row positions 7 and 15: 11 VALU instructions.
// A ninth value would take ten more by itself; it waits in a row of LDS until
// four splats' fill the wave (row_sums4, 7 for the four).  The same tree in
// registers (half-wave and row exchanges) takes 24 and 8.
struct WaveSum8 {
  int q;       // the value this lane sums in the LDS step (0..7)
  int src;     // the first of its eight source lanes
  bool owner;  // row position 7 or 15: ends with the total of value q
};
__device__ __forceinline__ WaveSum8 wave_sum8_lane(unsigned lane) {
  const unsigned p = lane & 15u, r = lane >> 4;
  return {(int)(2u * r + (p >> 3)), (int)(8u * (p & 7u)), (p & 7u) == 7u};
}
// Orders the LDS accesses of a one-wave work-group.  The LDS serves a wave's accesses in their order, so no wait for
// the stores is needed before a load of what they wrote; only the compiler has to keep the order.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// acc[0..7] receive the totals by plain stores.  Called by the whole wave.
__device__ __forceinline__ void wave_sums8(const float (&v)[8], float (*red)[DMGS_WAVE], const WaveSum8& w,
                                           float* acc) {
  const unsigned lane = threadIdx.x & 63;
  wave_lds_order();  // the previous call's reads of red
#pragma unroll
  for (int q = 0; q < 8; ++q) red[q][lane] = v[q];
  wave_lds_order();
  const float4 a = *reinterpret_cast<const float4*>(&red[w.q][w.src]);
  const float4 b = *reinterpret_cast<const float4*>(&red[w.q][w.src + 4]);
  float s = ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
  s = DMGS_DPP_ADD(s, 0xB1);   // quad_perm [1,0,3,2]
  s = DMGS_DPP_ADD(s, 0x4E);   // quad_perm [2,3,0,1]: each quad holds its four sources' sum
  s = DMGS_DPP_ADD(s, 0x114);  // row_shr 4: position 7 (15) adds position 3 (11)
  if (w.owner) acc[w.q] = s;
}
// The sums of four rows of 64 values: row r of the wave leaves with that of rows[r] in each of its lanes.
__device__ __forceinline__ float row_sums4(const float (*rows)[DMGS_WAVE]) {
  const unsigned lane = threadIdx.x & 63;
  wave_lds_order();  // the rows are written
  const float4 a = *reinterpret_cast<const float4*>(&rows[0][4u * lane]);
  float s = (a.x + a.y) + (a.z + a.w);
  s = DMGS_DPP_ADD(s, 0xB1);
  s = DMGS_DPP_ADD(s, 0x4E);
  return DMGS_DPP_ADD(DMGS_DPP_ADD(s, 0x124), 0x128);  // row_ror 4, row_ror 8
}

// Backward state of one pixel, walking its list back to front.  The reference
// keeps per channel ch an accumulator acc_ch (colour behind the current splat)
// and needs only  sum_ch (col_ch - acc_ch) g_ch  (g = dL/dpixel), so one
// recursion on S = sum_ch acc_ch g_ch replaces three:
// S <- (1 - alpha) S + alpha <col, g>.  The background stays out of S: its
// share of dL/dalpha is -T_final <bg, g> / (1 - alpha), one multiply-add from
// a per-pixel constant, whose rounding does not grow along the list (as the
// start of S, <bg, g> is rounded once per splat in front).
struct BwdPixel {
  float T;  // transmittance in front of the splat last processed
  float S;  // sum_ch acc_ch g_ch behind the next one
};

// One contributing splat (alpha, colour col) at a pixel with dL/dpixel =
// (g0, g1, g2): updates the state and returns dL/dalpha; w = alpha T is
// dL/dcolour_ch / g_ch.  The rounding sequence is fixed: gradients of scales
// and rotations are small differences of these values' sums, so another
// sequence of equal accuracy moves single elements by up to 1e-3 of their rms
// (S + alpha (<col, g> - S), one instruction less, and the background in S:
// 4e-7 of the gradients' norm, a repeated run 1e-7).
__device__ __forceinline__ float bwd_step(BwdPixel& st, float alpha, const float4& col, float g0, float g1,
                                          float g2, float bg_term, float& w) {
  const float om = 1.f - alpha;
  const float inv = __builtin_amdgcn_rcpf(om);  // T before this splat = T / (1 - alpha)
  st.T *= inv;
  w = alpha * st.T;
  const float cg = fmaf(col.z, g2, fmaf(col.y, g1, col.x * g0));
  const float d = cg - st.S;
  st.S = fmaf(om, st.S, __fmul_rn(alpha, cg));
  return fmaf(bg_term, inv, __fmul_rn(d, st.T));
}

// Gradients through G = exp(power), with t = dL/dG G = o G dL/dalpha (the
// reference ignores the 0.99 clamp): dL/d(dx) = -t (a dx + b dy), dL/d(dy) =
// -t (b dx + c dy), dL/d(a, b, c) = -t (dx^2, dx dy, dy^2) / 2, dL/do =
// t / o.  From the scaled conic q = log2(e) (-a/2, -b, -c/2):
// -(a X + b Y) = ln 2 (2 q.x X + q.y Y) and -(b X + c Y) = ln 2 (q.y X + 2 q.z Y).
// The kernel sums, per splat, (2 q.x X + q.y Y, q.y X + 2 q.z Y, t dx^2,
// t dx dy, t dy^2, t / o, w g_ch) with X = t dx, Y = t dy over the pixels; the
// flush applies the constant factors.
__device__ __forceinline__ float grad_scale(int k, float ddelx_dx, float ddely_dy) {
  constexpr float kLn2 = 0.693147180559945309f;
  return k == 0 ? kLn2 * ddelx_dx : (k == 1 ? kLn2 * ddely_dy : (k < 5 ? -0.5f : 1.0f));
}
__device__ __forceinline__ float dmean_x(const float4& q, float X, float Y) { return fmaf(q.x, X + X, q.y * Y); }
__device__ __forceinline__ float dmean_y(const float4& q, float X, float Y) { return fmaf(q.z, Y + Y, q.y * X); }

// Stages a splat record (s0, s1, s2) of the list position `pos`.
template <typename L>
__device__ __forceinline__ void put_splat(L& lds, int slot, float4 s0, float4 s1, float4 s2, uint32_t id, uint32_t P,
                                          const PixelRects& rr, uint32_t pos) {
  StagedSplat t{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, pos, 0u, 0u};
  if (id < P) {  // always, for lists built by the binning step; a zero-opacity splat never contributes
    constexpr float kHalf = -0.5f * kLog2e;
    t = {s0.x, s0.y, kHalf * s0.z, -kLog2e * s0.w, kHalf * s1.x, s1.y, s1.z, s1.w, s2.x, pos,
         reach_mask(s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, rr), id};
  }
  lds.put(slot, t);
}

template <typename L>
__device__ __forceinline__ void stage_splat(L& lds, int slot, const float4* __restrict__ splats, uint32_t id,
                                            uint32_t P, const PixelRects& rr, uint32_t pos) {
  const float4* sp = splats + (size_t)DMGS_SPLAT_F4 * min(id, P - 1);
  put_splat(lds, slot, sp[0], sp[1], sp[2], id, P, rr, pos);
}

// Everything a workgroup needs to know about its pixels.
struct TileCtx {
  int tile;            // global tile id (indexes ranges)
  int px, py;          // this lane's pixel
  int W, H;
  bool inside;
  size_t pix;          // index into the per-pixel buffers
  size_t plane;        // W * H of the view
  size_t img;          // offset of the view's colour planes
  float bg0, bg1, bg2;
  uint32_t bit;        // multi-view: this tile's bit in its cell's key masks
  uint2 range;         // single view: the tile's list; multi-view: its cell's list
  PixelRects rows;     // the work-group's pixel rectangles: 8x8 quadrants or 16x4 strips
};

// The tile in dispatch slot `slot`; a stale or unset order entry falls back to the identity.
__device__ __forceinline__ int ordered_tile(const RenderArgs& a, int slot) {
  if (a.tile_order) {
    const uint32_t t = a.tile_order[slot];
    if (t < (uint32_t)a.num_tiles) return (int)t;
  }
  return slot;
}

// QUADS (256 lanes): wave k covers the 8x8 quadrant k (k & 1: right, k >> 1: lower); otherwise (64 lanes) a
// lane's first pixel is in the tile's top 16x4 strip.
// half: a work-group of the whole tile (-1), or of its upper (0) or lower (1) 16x8 pixels, of which each wave then
// owns 8x4 with two lanes each (see render_fwd_quads_kernel).
template <bool QUADS>
__device__ __forceinline__ TileCtx tile_ctx(const RenderArgs& a, int tile, int half = -1) {
  TileCtx c;
  c.tile = tile;
  int lt = c.tile, gx = a.grid_x;
  int64_t pbase = 0;
  int list = c.tile;
  c.bit = 0;
  if (a.views) {
    const ViewDesc& v = a.views[a.tile_view ? a.tile_view[c.tile] : 0];
    lt = c.tile - v.tile_base;
    gx = v.grid_x;
    const int ltx = lt % gx, lty = lt / gx;
    constexpr int E = 1 << DMGS_CELL_SHIFT;
    list = v.cell_base + (lty >> DMGS_CELL_SHIFT) * cells_x(gx) + (ltx >> DMGS_CELL_SHIFT);
    c.bit = 1u << ((lty & (E - 1)) * E + (ltx & (E - 1)));
    c.W = v.W;
    c.H = v.H;
    c.bg0 = v.bg[0];
    c.bg1 = v.bg[1];
    c.bg2 = v.bg[2];
    pbase = v.pixel_base;
  } else {
    c.W = a.W;
    c.H = a.H;
    c.bg0 = a.bg[0];
    c.bg1 = a.bg[1];
    c.bg2 = a.bg[2];
  }
  const int tx = lt % gx, ty = lt / gx;
  int lx = threadIdx.x % DMGS_BLOCK_X, ly = threadIdx.x / DMGS_BLOCK_X;
  if constexpr (QUADS) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    lx = (wave & 1) * 8 + (lane & 7);
    ly = half < 0 ? (wave >> 1) * 8 + (lane >> 3) : half * 8 + (wave >> 1) * 4 + (lane >> 3 & 3);
  }
  const int ox = tx * DMGS_BLOCK_X, oy = ty * DMGS_BLOCK_Y;
  c.px = ox + lx;
  c.py = oy + ly;
  // rectangle k: quadrant k of the tile or of its half, or 16x4 strip k
  c.rows.x0 = (float)ox;
  c.rows.y0 = (float)(half > 0 ? oy + 8 : oy);
  c.rows.w = QUADS ? 8.0f : 16.0f;
  c.rows.h = QUADS && half < 0 ? 8.0f : 4.0f;
  c.rows.cols = QUADS ? 2 : 1;
  c.inside = c.px < c.W && c.py < c.H;
  c.plane = (size_t)c.W * c.H;
  c.pix = (size_t)pbase + (size_t)c.py * c.W + c.px;
  c.img = 3 * (size_t)pbase;
  uint32_t K = a.K;
  if (a.K_dev) K = min(K, *a.K_dev);
  uint2 r = a.ranges[list];
  r.y = min(r.y, K);
  r.x = min(r.x, r.y);
  c.range = r;
  return c;
}

// A forward work-group's share of clearing the backward accumulator: run
// after its blend work, so the stores delay no load of the blend.
__device__ __forceinline__ void clear_share(const RenderArgs& a) {
  if (a.clear_words && blockIdx.x == 0)
    for (int i = threadIdx.x; i < a.clear_words_n; i += blockDim.x) a.clear_words[i] = 0u;
  if (!a.clear) return;
  const size_t per = (a.clear_n + gridDim.x - 1) / gridDim.x;
  const size_t lo = (size_t)blockIdx.x * per, hi = min(a.clear_n, lo + per);
  for (size_t i = lo + threadIdx.x; i < hi; i += blockDim.x) a.clear[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Stage the next instances of this tile from its cell list, back to front (one wave): visit the list
// positions cursor-1, cursor-2, ... down to lo, four times 64 a round, and keep those whose key holds this tile's
// bit, in visit order, until BATCH are found; then stage the kept records in one pass, one lane per record.  Full
// batches share the loads, the footprint test (250 instructions) and the waits among 64 members; about a third of a
// cell's positions are a tile's members, so a batch of one round of 64 held 20.  Moves cursor down to the last
// position taken; returns the number staged; ends with a barrier.
template <int BATCH>
__device__ __forceinline__ int stage_cell_batch(BwdSplats<BATCH>& L, const RenderArgs& a, const TileCtx& c, int& cursor,
                                                int lo) {
  constexpr int U = 4;  // positions per lane and round
  const int s = (int)threadIdx.x;
  const uint64_t lt = lanemask_lt();
  int run = 0;
  do {
    const int base = cursor;
    // The entry ids are requested with the keys, all without a branch (lanes
    // past the list read its first entry and ignore it): one memory round
    // trip per round.
    uint32_t key[U], id[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = base - 1 - s - u * DMGS_WAVE;
      const uint32_t at = c.range.x + (q >= lo ? (uint32_t)q : 0u);
      key[u] = a.list_keys[at];
      id[u] = a.point_list[at];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (run == BATCH) break;  // the rest of the round is read again
      const int q = base - 1 - s - u * DMGS_WAVE;
      const bool member = q >= lo && ((key[u] >> DMGS_CELL_KEY_BITS) & c.bit);
      const uint64_t bal = __ballot(member);
      const int slot = run + (int)__popcll(bal & lt);
      if (member && slot < BATCH)  // id and position wait in the record for the staging pass
        L.xym[slot] = make_float4(0.f, 0.f, __uint_as_float(id[u]), __uint_as_float((uint32_t)q));
      run += (int)__popcll(bal);
      cursor = base - (u + 1) * DMGS_WAVE;
      if (run > BATCH) {  // the batch ends before its first member without a slot
        const uint64_t first = __ballot(member && slot == BATCH);
        cursor = base - u * DMGS_WAVE - (int)__builtin_ctzll(first);
        run = BATCH;
      }
    }
  } while (run < BATCH && cursor > lo);
  __syncthreads();
  for (int s = (int)threadIdx.x; s < run; s += DMGS_WAVE) {
    const float4 t = L.xym[s];
    stage_splat(L, s, a.splats, __float_as_uint(t.z), a.P, c.rows, __float_as_uint(t.w));
  }
  __syncthreads();
  return run;
}

// A group of four staged splats in registers, and the LDS byte offsets of the next group's.
struct FwdGroup {
  static constexpr int kN = 4;
  uint4 at;
  float4 xyq[kN], qorg[kN];
};

// Two pairs of staged splats as one of a pixel's two lanes reads them: of each pair its own splat's shape, and both
// splats' colours in its channels (red and green, or blue); and the LDS byte offsets of the next four splats.
struct FwdPairs {
  uint4 at;
  float4 xyq[2];
  float2 qo[2], col[2][2];
  uint32_t pos[2];
};

// The members of a tile in one chunk of its list (every position of a single view's tile list; the instances
// of a cell list whose mask holds the tile's bit), packed in list order.
template <int N>
struct MemberList {
  uint32_t id[N], pos[N];
};

// Forward: four waves per 16x16 tile, one pixel per lane, wave k covering the 8x8 quadrant k.  VALU issue
// bounds it where tiles are many, and one wave's own instruction stream where they are few (a wave issues
// one instruction in four cycles at best, 190 cycles per splat measured), so the loop is made of as few
// instructions of any kind as possible: each wave first packs the LDS offsets of the staged splats that reach
// its quadrant, then takes four at a time, reading the next four while it evaluates the four alphas (whose
// latencies overlap) and applies them in order with selects instead of branches.  Against one wave per tile
// with four pixels per lane: 8 views of 800x800 of 1M Gaussians 400 -> 294 us, 16 uneven views of 3M
// 5.33 -> 2.99 ms, one 800x800 view 154 -> 48 us, 333x251 of 500k 1377 -> 195 us.  Quadrants because a splat
// reaches fewer 8x8 blocks than 16x4 strips.  The arithmetic of a pixel and its order do not depend on
// CELLS, SPLIT or the launch.
// SPLIT: a tile's list is a chain (each pixel's transmittance goes from splat to splat), so a launch of few tiles
// takes as long as its longest list, however empty the GPU is: 24 instructions a splat in each of four waves.  Two
// work-groups blend a tile then, 16x8 pixels each with two lanes a pixel: the lanes evaluate the alphas of two
// consecutive splats side by side, exchange them, and both carry the transmittance over the two in order; one adds
// red and green, the other blue.  16 instructions a splat, in twice as many waves, with the same operations in the
// same order on every value.  (Eight waves of one work-group share a CU's SIMDs and gain nothing.)
// Five waves per SIMD where one work-group blends a tile: the compiler takes 106 registers (four
// waves) if left alone and 96 without a spill if asked; 16 uneven views 3.34 -> 2.99 ms, 8 views of 800x800 312 -> 294 us,
// 1920x1080 134 -> 125 us.  Six waves spill 48 bytes (8 views of 800x800 330 us); two work-groups a tile have
// few waves in flight at any register count.
template <bool CELLS, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SPLIT ? 1 : 5, 8))) void render_fwd_quads_kernel(
    RenderArgs a) {
  constexpr int NT = 256, U = FwdGroup::kN;
  constexpr int kPad = NT * 16;      // offset of the filling splat
  __shared__ FwdSplats<NT + 1> L;    // slot NT: a splat of zero opacity, which fills up groups
  constexpr int C = CELLS ? 4 : 1;   // list positions per lane and chunk
  __shared__ MemberList<C * NT> M;
  __shared__ uint32_t s_wc[2][C][NT / DMGS_WAVE];
  __shared__ __align__(16) uint32_t s_reach[NT / DMGS_WAVE][NT + 12];
  const int half = SPLIT ? (int)(blockIdx.x & 1u) : -1;
  const TileCtx c = tile_ctx<true>(a, ordered_tile(a, SPLIT ? (int)(blockIdx.x >> 1) : (int)blockIdx.x), half);
  const float pxf = (float)c.px, pyf = (float)c.py;
  const int len = (int)(c.range.y - c.range.x);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) L.xyq[NT] = L.qorg[NT] = L.bpmi[NT] = make_float4(0.f, 0.f, 0.f, 0.f);
  // T > 0 while the pixel blends; a finished pixel (saturated, or outside the image) keeps -T
  float T = c.inside ? 1.0f : -1.0f;
  float C0 = 0.f, C1 = 0.f, C2 = 0.f;
  uint32_t last_contributor = 0;

  // Three overlapping steps: the keys and ids of a chunk of the list are on their way while the records of
  // the next 256 members are, and while the 256 before those are blended.  A chunk of a cell list is four
  // positions per lane: about a third of them are members, and a round of fewer than 256 costs as much to
  // stage.  One position per lane: one view of 333x251 of 500k Gaussians 364 us (195 with four), 16 uneven views
  // 4.21 ms (3.51); two: 255 us and 3.69 ms; on shallow lists (8 views of 800x800) the three are within 4 %.
  uint32_t key[C], id[C];
  int next_chunk = 0;  // the first position not asked for
  auto request = [&]() {  // positions past the list read its first entry and are no members
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const int q = next_chunk + k * NT + (int)threadIdx.x;
      const uint32_t p = c.range.x + (q < len ? (uint32_t)q : 0u);
      if constexpr (CELLS) key[k] = a.list_keys[p];
      id[k] = a.point_list[p];
    }
    next_chunk += C * NT;
  };
  // packs the requested chunk; returns the number of members (the barrier that follows is the caller's)
  int flip = 0;
  auto pack = [&]() {
    const int at = next_chunk - C * NT;
    uint64_t bal[C];
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const bool member = at + k * NT + (int)threadIdx.x < len && (!CELLS || ((key[k] >> DMGS_CELL_KEY_BITS) & c.bit));
      bal[k] = __ballot(member);
      if (lane == 0) s_wc[flip][k][wave] = (uint32_t)__popcll(bal[k]);
    }
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int k = 0; k < C; ++k) {
      int before = total + (int)__popcll(bal[k] & lanemask_lt());
#pragma unroll
      for (int w = 0; w < NT / DMGS_WAVE; ++w) {
        const int cnt = (int)s_wc[flip][k][w];
        before += w < wave ? cnt : 0;
        total += cnt;
      }
      if ((bal[k] >> lane) & 1u) {
        M.id[before] = id[k];
        M.pos[before] = (uint32_t)(at + k * NT + (int)threadIdx.x);
      }
    }
    flip ^= 1;
    return total;
  };
  float4 r0, r1, r2;  // this lane's record of the next round
  uint32_t my_id = 0, my_pos = 0;
  int members = 0, used = 0;  // of the packed chunk: all, and those whose records were asked for
  auto gather = [&]() {
    const int n = min(NT, members - used);
    const int s = used + min((int)threadIdx.x, max(n - 1, 0));  // no lane's loads are conditional
    my_id = M.id[min(s, C * NT - 1)];
    my_pos = M.pos[min(s, C * NT - 1)];
    const float4* sp = a.splats + (size_t)DMGS_SPLAT_F4 * min(my_id, a.P - 1);
    r0 = sp[0];
    r1 = sp[1];
    r2 = sp[2];
    used += n;
    return n;
  };
  int n_next = 0;  // members whose records are on their way
  bool asked = false;  // a chunk is on its way
  auto ask = [&]() {  // only once the packed one runs out: a tile may be finished before
    if (used == members && next_chunk < len) {
      request();
      asked = true;
    }
  };
  if (len > 0) {
    request();
    members = pack();
    __syncthreads();
    n_next = gather();
    ask();
  }
  while (n_next > 0 || asked) {
    if (__syncthreads_count(T < 0.f) == NT) break;
    const int n = n_next;
    if ((int)threadIdx.x < n) put_splat(L, threadIdx.x, r0, r1, r2, my_id, a.P, c.rows, my_pos + 1);
    if (asked) {
      members = pack();  // its barrier also orders the records
      used = 0;
      asked = false;
    }
    __syncthreads();
    n_next = gather();
    ask();
    if (__ballot(T > 0.f) == 0) continue;  // wave-uniform: this quadrant is finished
    // the round's splats that reach this quadrant, as LDS offsets in list order, filled up for whole groups
    // and for the two groups read ahead
    uint32_t* const reach = s_reach[wave];
    int count = 0;
    uint64_t odd = 0;
#pragma unroll
    for (int k = 0; k < NT; k += 64) {
      const int s = k + lane;
      const uint32_t mask = L.mask(min(s, NT));
      const bool reached = s < n && ((mask >> wave) & 1u);
      const uint64_t bits = __ballot(reached);
      odd |= __ballot(reached && (mask & kOddColor));
      if ((bits >> lane) & 1u) reach[count + (int)__popcll(bits & lanemask_lt())] = (uint32_t)s * 16u;
      count += (int)__popcll(bits);
    }
    if (count == 0) continue;
    if (odd != 0) {
      // The groups below add skipped splats with weight zero, which a colour that is not finite would turn into
      // NaN in pixels that it does not touch: such a round goes splat by splat, adding only what contributes.
      for (int i = 0; i < count; ++i) {
        const uint32_t o = reach[i];
        const float4 g = lds_at(L.xyq, o), q = lds_at(L.qorg, o), b = lds_at(L.bpmi, o);
        const float power = power_at(power_dx(g.z, g.w, g.x - pxf), q.x, g.y - pyf);
        const float alpha = fminf(0.99f, q.y * splat_exp2(power));
        if (!((power <= 0.0f) & (alpha >= 1.0f / 255.0f) & (T > 0.f))) continue;
        const float test_T = T * (1.0f - alpha), w = alpha * T;
        if (test_T >= 0.0001f) {
          const bool blue = SPLIT && lane >= 32;  // of a pixel's two lanes the one that adds blue, in C0
          C0 = fmaf(blue ? b.x : q.z, w, C0);
          C1 = fmaf(q.w, w, C1);
          C2 = fmaf(b.x, w, C2);
          T = test_T;
          last_contributor = __float_as_uint(b.y);
        } else {
          T = -T;
        }
      }
      continue;
    }
    int pad = lane;
    asm volatile("" : "+v"(pad));  // its address is made here: kept over the rounds it would be the register too many
    if (pad < 12) reach[count + pad] = kPad;
    if constexpr (SPLIT) {
      const bool second = lane >= 32;  // of the pixel's two lanes
      const char* const channels =
          second ? reinterpret_cast<const char*>(L.bpmi) : reinterpret_cast<const char*>(L.qorg) + 8;
      auto fetch = [&](FwdPairs& g, const uint4& at, int next) {
        const uint32_t own[2] = {second ? at.y : at.x, second ? at.w : at.z};
        const uint32_t both[2][2] = {{at.x, at.y}, {at.z, at.w}};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          g.xyq[p] = lds_at(L.xyq, own[p]);
          g.qo[p] = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(L.qorg) + own[p]);
          g.pos[p] = __float_as_uint(lds_at(L.bpmi, own[p]).y);
#pragma unroll
          for (int e = 0; e < 2; ++e) g.col[p][e] = *reinterpret_cast<const float2*>(channels + both[p][e]);
        }
        g.at = *reinterpret_cast<const uint4*>(reach + next);
      };
      // blends `cur` while `next` is on its way; false when nothing is left to do
      int done = 0;
      auto step = [&](FwdPairs& cur, FwdPairs& next) {
        fetch(next, cur.at, done + 8);
        float alpha[2];
        bool ok[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const float4 g = cur.xyq[p];
          const float power = power_at(power_dx(g.z, g.w, g.x - pxf), cur.qo[p].x, g.y - pyf);
          const float al = fminf(0.99f, cur.qo[p].y * splat_exp2(power));
          ok[p] = (power <= 0.0f) & (al >= 1.0f / 255.0f);
          alpha[p] = ok[p] ? al : 0.0f;
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(alpha[p]), __float_as_uint(alpha[p]), false, false);
          bool take[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {  // both lanes: the first lane's splat, then the second's
            const float al = __uint_as_float(x[e]);
            const float test_T = T * (1.0f - al);
            take[e] = test_T >= 0.0001f;
            const float w = take[e] ? al * T : 0.0f;
            C0 = fmaf(cur.col[p][e].x, w, C0);
            C1 = fmaf(cur.col[p][e].y, w, C1);  // the blue lane's is not used
            T = take[e] ? test_T : -fabsf(T);
          }
          const bool mine = (second & take[1]) | (!second & take[0]);
          last_contributor = (mine & ok[p]) ? cur.pos[p] : last_contributor;
        }
        done += 4;
        return done < count && __ballot(T > 0.f) != 0;
      };
      FwdPairs g0, g1;
      fetch(g0, *reinterpret_cast<const uint4*>(reach), 4);
      while (step(g0, g1) && step(g1, g0)) {
      }
      continue;
    }
    auto fetch = [&](FwdGroup& g, const uint4& at, int next) {
      const uint32_t o[U] = {at.x, at.y, at.z, at.w};
#pragma unroll
      for (int u = 0; u < U; ++u) {
        g.xyq[u] = lds_at(L.xyq, o[u]);
        g.qorg[u] = lds_at(L.qorg, o[u]);
      }
      g.at = *reinterpret_cast<const uint4*>(reach + next);
    };
    // blends `cur` (at the offsets `at`) while `next` is on its way; false when nothing is left to do
    int done = 0;
    auto step = [&](FwdGroup& cur, uint4& at, FwdGroup& next) {
      const uint32_t o[U] = {at.x, at.y, at.z, at.w};
      float4 bp[U];
#pragma unroll
      for (int u = 0; u < U; ++u) bp[u] = lds_at(L.bpmi, o[u]);
      fetch(next, cur.at, done + 2 * U);
      at = cur.at;
      float alpha[U];
      bool ok[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {  // independent of each other: their latencies overlap
        const float p = power_at(power_dx(cur.xyq[u].z, cur.xyq[u].w, cur.xyq[u].x - pxf), cur.qorg[u].x, cur.xyq[u].y - pyf);
        const float al = fminf(0.99f, cur.qorg[u].y * splat_exp2(p));
        ok[u] = (p <= 0.0f) & (al >= 1.0f / 255.0f);
        alpha[u] = ok[u] ? al : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float test_T = T * (1.0f - alpha[u]);  // T itself where the splat is skipped
        const bool take = test_T >= 0.0001f;         // never for a finished pixel
        const float w = take ? alpha[u] * T : 0.0f;
        C0 = fmaf(cur.qorg[u].z, w, C0);
        C1 = fmaf(cur.qorg[u].w, w, C1);
        C2 = fmaf(bp[u].x, w, C2);
        T = take ? test_T : -fabsf(T);
        last_contributor = (take & ok[u]) ? __float_as_uint(bp[u].y) : last_contributor;
      }
      done += U;
      return done < count && __ballot(T > 0.f) != 0;
    };
    FwdGroup g0, g1;
    uint4 at_now = *reinterpret_cast<const uint4*>(reach);
    fetch(g0, at_now, U);
    while (step(g0, at_now, g1) && step(g1, at_now, g0)) {
    }
  }
  if constexpr (CELLS && !SPLIT) {
    if (a.tile_work) {  // the backward walks list positions below the tile's largest last contributor
      __shared__ uint32_t s_max[NT / DMGS_WAVE];
      uint32_t m = last_contributor;
      for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
      if (lane == 0) s_max[wave] = m;
      __syncthreads();
      if (threadIdx.x == 0) a.tile_work[c.tile] = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
    }
  }
  if constexpr (SPLIT) {
    last_contributor = max(last_contributor, (uint32_t)__shfl_xor((int)last_contributor, 32, 64));
    if (lane >= 32) C2 = C0;
  }
  if (c.inside) {
    const size_t pid = c.pix - c.img / 3;  // pixel index within the view
    T = fabsf(T);
    float* out = a.out_color + c.img;
    if (!SPLIT || lane < 32) {
      a.final_T[c.pix] = T;
      a.n_contrib[c.pix] = last_contributor;
      out[pid] = C0 + T * c.bg0;
      out[c.plane + pid] = C1 + T * c.bg1;
    }
    if (!SPLIT || lane >= 32) out[2 * c.plane + pid] = C2 + T * c.bg2;
  }
  clear_share(a);
}

// The state of the backward recursion at every 64th member of a tile's list, from the back (see the head of this
// file): one work-group per tile, the forward's quadrants, one pixel per lane.  First the members are counted and the
// tile takes as many slots as it has boundaries; then T and S go from splat to splat with the operations of bwd_step
// on the same values, so that a segment which starts from them goes on exactly as the walk of the whole list would.
// Bound like the forward by its waves' instructions, and where tiles are few by the longest list's; the same three
// overlapping steps.  Rounds are whole (256 members, except the last), so that groups of 64 never straddle two: what
// is left of a packed chunk moves to its front.  Five waves per SIMD instead of four change nothing (1M Gaussians at
// 800x800 59.5 and 62.8 us).
__global__ __launch_bounds__(256) void render_bwd_chain_kernel(RenderArgs a) {
  constexpr int NT = 256, U = FwdGroup::kN, C = 4, G = kSegmentLength;
  static_assert(G == DMGS_WAVE, "a group is what one wave tests at once");
  constexpr int kPad = NT * 16;    // offset of the filling splat
  __shared__ FwdSplats<NT + 1> L;  // slot NT: a splat of zero opacity, which fills up groups
  __shared__ MemberList<(C + 1) * NT> M;
  __shared__ uint32_t s_wc[2][C][NT / DMGS_WAVE];
  __shared__ int s_hi[kTileSegments + 1];  // [i]: one past the position of member 64 i
  __shared__ uint32_t s_max[NT / DMGS_WAVE], s_first;
  __shared__ int s_stride;
  __shared__ __align__(16) uint32_t s_reach[NT / DMGS_WAVE][G + 12];
  const TileCtx c = tile_ctx<true>(a, ordered_tile(a, (int)blockIdx.x));
  const float pxf = (float)c.px, pyf = (float)c.py;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pixel = ((wave >> 1) * 8 + (lane >> 3)) * 16 + (wave & 1) * 8 + (lane & 7);  // row-major in the tile
  if (tid == 0) L.xyq[NT] = L.qorg[NT] = L.bpmi[NT] = make_float4(0.f, 0.f, 0.f, 0.f);
  float T = 0.f, S = 0.f, g0 = 0.f, g1 = 0.f, g2 = 0.f;
  uint32_t last = 0;
  if (c.inside) {
    const size_t pid = c.pix - c.img / 3;
    const float* dp = a.dL_dpix + c.img;
    T = a.final_T[c.pix];
    last = a.n_contrib[c.pix];
    g0 = dp[pid];
    g1 = dp[c.plane + pid];
    g2 = dp[2 * c.plane + pid];
  }
  uint32_t wave_last = last;  // positions at or past it contribute to none of the wave's pixels
  for (int off = 32; off > 0; off >>= 1) wave_last = max(wave_last, (uint32_t)__shfl_xor((int)wave_last, off, 64));
  wave_last = __builtin_amdgcn_readfirstlane(wave_last);
  if (lane == 0) s_max[wave] = wave_last;
  __syncthreads();
  const int len = min((int)(c.range.y - c.range.x), (int)max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3])));

  // The visit's k-th position of this lane in the chunk that starts after `at` positions from the back.
  auto position = [&](int at, int k) { return len - 1 - (at + k * NT + tid); };
  auto key_of = [&](int pos) { return a.list_keys[c.range.x + (uint32_t)max(pos, 0)]; };
  // Hands each member of the chunk its number, counted from `first`; returns how many there are.  One barrier.
  int flip = 0;
  auto number = [&](int at, const uint32_t(&key)[C], int first, auto&& each) {
    uint64_t bal[C];
#pragma unroll
    for (int k = 0; k < C; ++k) {
      bal[k] = __ballot(position(at, k) >= 0 && ((key[k] >> DMGS_CELL_KEY_BITS) & c.bit));
      if (lane == 0) s_wc[flip][k][wave] = (uint32_t)__popcll(bal[k]);
    }
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int k = 0; k < C; ++k) {
      int before = first + total + (int)__popcll(bal[k] & lanemask_lt());
#pragma unroll
      for (int w = 0; w < NT / DMGS_WAVE; ++w) {
        const int cnt = (int)s_wc[flip][k][w];
        before += w < wave ? cnt : 0;
        total += cnt;
      }
      if ((bal[k] >> lane) & 1u) each(before, k);
    }
    flip ^= 1;
    return total;
  };

  int members = 0;
  if (len > G) {
    uint32_t key[C], ahead[C];
#pragma unroll
    for (int k = 0; k < C; ++k) key[k] = key_of(position(0, k));
    for (int at = 0; at < len; at += C * NT) {
#pragma unroll
      for (int k = 0; k < C; ++k) ahead[k] = key_of(position(at + C * NT, k));
      members += number(at, key, members, [&](int i, int k) {
        if (i % G == 0 && i / G <= kTileSegments) s_hi[i / G] = position(at, k) + 1;
      });
#pragma unroll
      for (int k = 0; k < C; ++k) key[k] = ahead[k];
    }
  }
  // Slots come from one of kSegmentParts counters (one for all: atomics of 3844 tiles on one address took 100 us).
  // Segments get longer as its slots are used up (64 members until half of them are gone, then 128 until a quarter is
  // left, and so on): the longest lists come first, and every tile still finds some.  The backward proper of 1.5M
  // Gaussians at 800x800 takes 203 us (whole lists 781), 885 with 64 members while slots last.
  const int boundaries = members > 0 ? min((members - 1) / G, kTileSegments) : 0;
  const int part = (int)blockIdx.x % kSegmentParts, part_cap = a.seg.cap / kSegmentParts;
  if (tid == 0) {
    uint32_t* const head = a.seg.head + part * kSegmentHeadStride;
    int stride = 1;
    if (boundaries > 0) {
      const uint32_t taken = __hip_atomic_load(head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int left = part_cap - (int)min(taken, (uint32_t)part_cap);
      while (stride < kTileSegments && left < part_cap / (2 * stride)) stride *= 2;
    }
    s_stride = stride;
    s_first = boundaries >= stride ? atomicAdd(head, (uint32_t)(boundaries / stride)) : 0u;
  }
  __syncthreads();
  const int stride = s_stride;  // groups of 64 per segment
  const int usable = min(boundaries / stride, part_cap - (int)min(s_first, (uint32_t)part_cap));
  const uint32_t first = (uint32_t)(part * part_cap) + s_first;
  for (int i = tid; i < usable; i += NT)  // the segment in front of boundary i + 1; the last one takes what is left
    a.seg.rec[first + i] = make_uint4((uint32_t)c.tile, (uint32_t)(i + 1 < usable ? s_hi[(i + 2) * stride] : 0),
                                      (uint32_t)s_hi[(i + 1) * stride], 0u);
  if (tid == 0) a.seg.tile_last[c.tile] = usable > 0 ? (uint32_t)s_hi[stride] : 0u;
  if (usable == 0) return;

  uint32_t key[C], id[C];
  int next_chunk = 0;  // the first position (from the back) not asked for
  auto request = [&]() {
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const int pos = position(next_chunk, k);
      key[k] = key_of(pos);
      id[k] = a.point_list[c.range.x + (uint32_t)max(pos, 0)];
    }
    next_chunk += C * NT;
  };
  int used = 0;        // of the packed members those whose records were asked for
  bool asked = false;  // a chunk is on its way
  members = 0;         // packed
  // Packs the chunk on its way, and more until there is a whole round or the list ends; ends with a barrier.
  auto fill = [&]() {
    while (asked) {
      const int left = members - used;  // fewer than a round: where they are and where they go is disjoint
      if (used > 0 && tid < left) {
        M.id[tid] = M.id[used + tid];
        M.pos[tid] = M.pos[used + tid];
      }
      const int at = next_chunk - C * NT;
      used = 0;
      members = left + number(at, key, left, [&](int i, int k) {
        M.id[i] = id[k];
        M.pos[i] = (uint32_t)position(at, k);
      });
      asked = members < NT && next_chunk < len;
      if (asked) request();
    }
    __syncthreads();
  };
  auto ask = [&]() {
    if (members - used < NT && next_chunk < len) {
      request();
      asked = true;
    }
  };
  float4 r0, r1, r2;  // this lane's record of the next round
  uint32_t my_id = 0, my_pos = 0;
  auto gather = [&]() {
    const int n = min(NT, members - used);
    const int s = used + min(tid, max(n - 1, 0));  // no lane's loads are conditional
    my_id = M.id[min(s, (C + 1) * NT - 1)];
    my_pos = M.pos[min(s, (C + 1) * NT - 1)];
    const float4* sp = a.splats + (size_t)DMGS_SPLAT_F4 * min(my_id, a.P - 1);
    r0 = sp[0];
    r1 = sp[1];
    r2 = sp[2];
    used += n;
    return n;
  };
  request();
  asked = true;
  fill();
  int n_next = gather();
  ask();
  int next_state = 0, to_state = stride;  // the boundary that comes next, and the groups up to it
  while (next_state < usable && n_next > 0) {
    const int n = n_next;
    __syncthreads();  // the round before has been read
    if (tid < n) put_splat(L, tid, r0, r1, r2, my_id, a.P, c.rows, my_pos);
    fill();
    n_next = gather();
    ask();
    for (int h = 0; h < n && next_state < usable; h += G) {
      uint32_t* const reach = s_reach[wave];
      const uint64_t bits =
          __ballot(h + lane < n && ((L.mask(h + lane) >> wave) & 1u) && L.pos(h + lane) < wave_last);
      const int count = (int)__popcll(bits);
      if (count > 0) {
        if ((bits >> lane) & 1u) reach[(int)__popcll(bits & lanemask_lt())] = (uint32_t)(h + lane) * 16u;
        if (lane < 12) reach[count + lane] = kPad;
        auto fetch = [&](FwdGroup& g, const uint4& at, int next) {
          const uint32_t o[U] = {at.x, at.y, at.z, at.w};
#pragma unroll
          for (int u = 0; u < U; ++u) {
            g.xyq[u] = lds_at(L.xyq, o[u]);
            g.qorg[u] = lds_at(L.qorg, o[u]);
          }
          g.at = *reinterpret_cast<const uint4*>(reach + next);
        };
        // walks `cur` (at the offsets `at`) while `next` is on its way; false when nothing is left to do
        int walked = 0;
        auto step = [&](FwdGroup& cur, uint4& at, FwdGroup& next) {
          const uint32_t o[U] = {at.x, at.y, at.z, at.w};
          float4 bp[U];
#pragma unroll
          for (int u = 0; u < U; ++u) bp[u] = lds_at(L.bpmi, o[u]);
          fetch(next, cur.at, walked + 2 * U);
          at = cur.at;
          float om[U], inv[U], add[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {  // independent of each other: their latencies overlap
            const float4 g = cur.xyq[u], q = cur.qorg[u];
            const float p = power_at(power_dx(g.z, g.w, g.x - pxf), q.x, g.y - pyf);
            const float alpha = fminf(0.99f, q.y * splat_exp2(p));
            const bool ok = (p <= 0.0f) & (alpha >= 1.0f / 255.0f) & (__float_as_uint(bp[u].y) < last);
            om[u] = ok ? 1.f - alpha : 1.f;  // a skipped splat multiplies by one and adds zero
            inv[u] = __builtin_amdgcn_rcpf(om[u]);
            const float cg = fmaf(bp[u].x, g2, fmaf(q.w, g1, q.z * g0));
            add[u] = ok ? __fmul_rn(alpha, cg) : 0.f;
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            T *= inv[u];
            S = fmaf(om[u], S, add[u]);
          }
          walked += U;
          return walked < count;
        };
        FwdGroup e0, e1;
        uint4 at_now = *reinterpret_cast<const uint4*>(reach);
        fetch(e0, at_now, U);
        while (step(e0, at_now, e1) && step(e1, at_now, e0)) {
        }
      }
      if (--to_state == 0) {
        a.seg.state[(size_t)(first + (uint32_t)next_state) * 256 + pixel] = make_float2(T, S);
        ++next_state;
        to_state = stride;
      }
    }
  }
}

// Backward with one wave per 16x16 tile: lane (lx, ly) owns the pixels
// (lx, ly + 4k), k = 0..3, i.e. one pixel in each of four 16x4 strips.  The
// footprint test runs per strip, each pixel is evaluated exactly as in the
// forward, and a lane first sums its four pixels' partial gradients, so each
// (tile, splat) pays for one wave reduction instead of four.
//
// Bound by the instructions of its waves, vector and scalar, at five waves per
// SIMD (95 registers; six spill, and four take 24 % longer): so a batch is
// filled before it is walked, what can be decided for 64 staged splats at once
// (which strips are live) is, one lane per splat, and the ninth sum waits for
// three others'.  Before and now: sixteen uneven views of 3 M Gaussians 6.91
// and 5.33 ms, eight 800x800 views of 1 M 483 and 438 us (5.06 ms and 424 us
// with the background in the recursion and the linear forms after the sums,
// whose gradients differ, see bwd_step).
//
// SEGS: the first a.num_tiles work-groups each take the last segment of a tile's
// list (or all of it), which starts at the list's end, the others one that
// starts from a state (see Segments).
template <bool CELLS, bool SEGS>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5, 8))) void render_bwd_strips_kernel(RenderArgs a) {
  constexpr int NT = 64, BATCH = 64;
  int tile, lo = 0, hi = 0x7fffffff;                   // this work-group's list positions [lo, hi)
  uint32_t seg_end = kNoSegment;                       // the slot of the state at hi (none: the list's end)
  if constexpr (SEGS) {
    if ((int)blockIdx.x < a.num_tiles) {
      tile = ordered_tile(a, blockIdx.x);
      lo = max((int)a.seg.tile_last[tile], 0);
    } else {  // the parts' used slots in turn, before the unused ones (16k work-groups that only end take 20 us)
      const uint32_t b = blockIdx.x - (uint32_t)a.num_tiles, part = b % kSegmentParts, i = b / kSegmentParts;
      if (i >= a.seg.head[part * kSegmentHeadStride]) return;
      seg_end = part * (uint32_t)(a.seg.cap / kSegmentParts) + i;
      const uint4 r = a.seg.rec[seg_end];
      if (r.x >= (uint32_t)a.num_tiles) return;
      tile = (int)r.x;
      lo = max((int)r.y, 0);
      hi = (int)r.z;
    }
  } else {
    tile = ordered_tile(a, blockIdx.x);
  }
  __shared__ BwdSplats<BATCH> L;
  // Two accumulator sets of a quarter of a batch: a set's global atomics are
  // issued after the next batch has been staged (or before the batch's next
  // quarter), so no staging load waits behind them (the memory counter is in
  // order) and they complete while that one is computed.
  constexpr int SET = BATCH / 4;
  __shared__ float s_acc[2][SET][DMGS_GACC_USED];
  uint32_t set_id = 0;  // lane i: the Gaussian of slot i of the set to be flushed
  __shared__ __align__(16) float s_red[8][DMGS_WAVE];    // a splat's per-lane values 0..7
  __shared__ __align__(16) float s_ninth[4][DMGS_WAVE];  // value 8 of the last splats, until there are four
  const TileCtx c = tile_ctx<false>(a, tile);  // pixel k = 0 of this lane: (lx, ly), ly in 0..3
  const unsigned lane = threadIdx.x & 63;
  const WaveSum8 wsum = wave_sum8_lane(lane);
  const float pxf = (float)c.px;
  const float ddelx_dx = 0.5f * (float)c.W, ddely_dy = 0.5f * (float)c.H;  // d pixel / d NDC
  float pyf[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) pyf[k] = (float)(c.py + 4 * k);

  float g0[4], g1[4], g2[4], bg_term[4];
  BwdPixel st[4];
  uint32_t last_contributor[4];
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int py = c.py + 4 * k;
    const bool inside = c.px < c.W && py < c.H;
    float T_final = 0.f;
    g0[k] = g1[k] = g2[k] = 0.f;
    last_contributor[k] = 0;
    if (inside) {
      const size_t pix = c.pix + (size_t)(4 * k) * c.W;
      const size_t pid = pix - c.img / 3;
      const float* dp = a.dL_dpix + c.img;
      T_final = a.final_T[pix];
      last_contributor[k] = a.n_contrib[pix];
      g0[k] = dp[pid];
      g1[k] = dp[c.plane + pid];
      g2[k] = dp[2 * c.plane + pid];
    }
    bg_term[k] = -T_final * (c.bg0 * g0[k] + c.bg1 * g1[k] + c.bg2 * g2[k]);
    st[k] = {T_final, 0.f};
    if constexpr (SEGS) {
      if (seg_end != kNoSegment) {  // start from the state at hi
        const float2 e = a.seg.state[(size_t)seg_end * 256 + threadIdx.x + 64 * k];
        st[k] = {e.x, e.y};
      }
    }
  }
  // per strip, the largest last contributor of its 64 pixels (wave-uniform):
  // list positions at or past it cannot contribute to the strip
  uint32_t strip_max[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    uint32_t x = last_contributor[k];
    for (int off = 32; off > 0; off >>= 1) x = max(x, (uint32_t)__shfl_xor((int)x, off, 64));
    strip_max[k] = __builtin_amdgcn_readfirstlane(x);
    m = max(m, strip_max[k]);
  }
  const int todo_total = min(min((int)(c.range.y - c.range.x), (int)m), hi);

  // one set's sums -> one global atomic per (splat, value)
  auto flush = [&](int buf, uint32_t slots) {
    static_assert(SET * DMGS_GACC_USED <= 3 * NT, "slot positions of three rounds");
#pragma unroll 1
    for (int r = 0; r < 3; ++r) {  // whole rounds: every lane hands out its slot's id
      const int i = r * NT + (int)threadIdx.x;
      const int slot = i / DMGS_GACC_USED, q = i - slot * DMGS_GACC_USED;
      const uint32_t gid = (uint32_t)__shfl((int)set_id, slot);
      if (!((slots >> slot) & 1u)) continue;
      const float val = s_acc[buf][slot][q] * grad_scale(q, ddelx_dx, ddely_dy);
      if (val != 0.f) unsafeAtomicAdd(a.gacc + gacc_index(a.P, gid, q), val);
    }
  };
  int buf = 0;
  uint32_t summed = 0;      // slots of set buf that hold sums
  int cursor = todo_total;  // list positions in [lo, cursor) are still to do
  while (cursor > lo) {
    __syncthreads();
    const int top = cursor;
    int n;
    if constexpr (CELLS) {
      n = stage_cell_batch(L, a, c, cursor, lo);
    } else {
      for (int s = threadIdx.x; s < BATCH; s += NT) {
        const int pos = top - 1 - s;
        if (pos >= lo) stage_splat(L, s, a.splats, a.point_list[c.range.x + pos], a.P, c.rows, (uint32_t)pos);
      }
      __syncthreads();
      n = min(BATCH, top - lo);
      cursor -= n;
    }
    // Every staging load has landed here; saying so keeps the compiler from
    // waiting later (behind the atomics below) for a load it cannot rule out.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    // lane s: the strips that slot s reaches and that still have pixels behind it
    const uint32_t pos = L.pos(lane);
    uint32_t live_of = (int)lane < n ? L.mask(lane) : 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (pos >= strip_max[k]) live_of &= ~(1u << k);
    const uint64_t todo = __ballot(live_of != 0u);
    for (int j0 = 0; j0 < n; j0 += SET) {
      uint32_t left = (uint32_t)(todo >> j0) & ((1u << SET) - 1u);
      if (left == 0u) continue;
      flush(buf, summed);  // overlaps this quarter
      buf ^= 1;
      summed = 0;
      set_id = L.id(j0 + (int)(lane & (SET - 1u)));
      uint32_t ninth = 0, ninths = 0;  // slots of s_ninth's rows, a byte each, the last one lowest
      auto sum_ninths = [&]() {
        const float e = row_sums4(s_ninth);
        const uint32_t r = lane >> 4;
        if (r < ninths && (lane & 15u) == 0u) s_acc[buf][(ninth >> (8u * (ninths - 1u - r))) & (SET - 1u)][8] = e;
        ninths = 0;
      };
      while (left) {
        const int slot = __builtin_ctz(left), j = j0 + slot;
        left &= left - 1u;
        const uint32_t live = __builtin_amdgcn_readlane(live_of, j), contributor = __builtin_amdgcn_readlane(pos, j);
        const float2 xy = make_float2(L.xym[j].x, L.xym[j].y);
        const float4 q = L.qo[j];
        const float4 col = L.rgb_id[j];
        const float dx = xy.x - pxf;
        const PowerDx pd = power_dx(q.x, q.y, dx);  // shared by the lane's four pixels (one column)
        // per-lane sums over its pixels: sum t, sum t dy, sum t dy^2 (dx is the
        // same for the four pixels, so its powers multiply in once per splat)
        float s_t = 0.f, s_tdy = 0.f, s_tdy2 = 0.f, c0 = 0.f, c1 = 0.f, c2 = 0.f;
        bool any = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (!((live >> k) & 1u)) continue;  // wave-uniform
          const float dy = xy.y - pyf[k];
          const float p = power_at(pd, q.z, dy);
          const float G = splat_exp2(p);
          const float ga = q.w * G;  // o G: alpha before the 0.99 clamp
          const float alpha = fminf(0.99f, ga);
          if (contributor < last_contributor[k] && p <= 0.0f && alpha >= 1.0f / 255.0f) {
            any = true;
            float w;
            const float t = ga * bwd_step(st[k], alpha, col, g0[k], g1[k], g2[k], bg_term[k], w);
            c0 = fmaf(w, g0[k], c0);
            c1 = fmaf(w, g1[k], c1);
            c2 = fmaf(w, g2[k], c2);
            s_t += t;
            const float tdy = t * dy;
            s_tdy += tdy;
            s_tdy2 = fmaf(tdy, dy, s_tdy2);
          }
        }
        if (__ballot(any) == 0) continue;
        const float s_tdx = s_t * dx;
        // the linear forms before the sums over the lanes: X and Y of a long splat cancel in them
        const float v[8] = {dmean_x(q, s_tdx, s_tdy), dmean_y(q, s_tdx, s_tdy), s_tdx * dx, s_tdy * dx, s_tdy2,
                            s_t * __builtin_amdgcn_rcpf(q.w), c0, c1};
        int at = (buf * SET + slot) * DMGS_GACC_USED;
        asm("" : "+s"(at));  // a scalar product, not a 64-bit one per lane
        wave_sums8(v, s_red, wsum, &s_acc[0][0][0] + at);
        s_ninth[ninths][lane] = c2;
        ninth = ninth << 8 | (uint32_t)slot;
        summed |= 1u << slot;
        if (++ninths == 4u) sum_ninths();
      }
      if (ninths) sum_ninths();
      __syncthreads();
    }
  }
  flush(buf, summed);
  if (a.clear_words && blockIdx.x == 0)  // the tile-order histogram, ready for another backward's
    for (int i = threadIdx.x; i < a.clear_words_n; i += NT) a.clear_words[i] = 0u;
}

// Longest-first scheduling of the blend: a tile's cost is about the length
// of its binning cell's list, so tiles are bucketed by log2 of that length
// (8 buckets per octave, 256 in all) and emitted heaviest bucket first.  Only
// the dispatch order changes; every tile's result is the same in any order.
__device__ __forceinline__ uint32_t tile_cost_bucket(const RenderArgs& a, int t, uint32_t K, bool use_work) {
  const ViewDesc& v = a.views[a.tile_view ? a.tile_view[t] : 0];
  const int lt = t - v.tile_base, gx = v.grid_x;
  const int ltx = lt % gx, lty = lt / gx;
  const int cell = v.cell_base + (lty >> DMGS_CELL_SHIFT) * cells_x(gx) + (ltx >> DMGS_CELL_SHIFT);
  const uint2 r = a.ranges[cell];
  const uint32_t hi = min(r.y, K), lo = min(r.x, hi);
  uint32_t len = hi - lo;
  if (use_work) len = min(len, a.tile_work[t]);
  if (len == 0) return 255u;
  return 254u - min(254u, (uint32_t)(8.0f * __log2f((float)len)));
}

// Pass 1 (all tiles in parallel): bucket per tile, global bucket histogram.
__global__ __launch_bounds__(256) void tile_bucket_kernel(RenderArgs a, uint8_t* __restrict__ bucket,
                                                          uint32_t* __restrict__ hist, int use_work) {
  __shared__ uint32_t cnt[256];
  uint32_t K = a.K;
  if (a.K_dev) K = min(K, *a.K_dev);
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < a.num_tiles) {
    const uint32_t b = tile_cost_bucket(a, t, K, use_work != 0);
    bucket[t] = (uint8_t)b;
    atomicAdd(&cnt[b], 1u);
  }
  __syncthreads();
  if (cnt[threadIdx.x]) atomicAdd(&hist[threadIdx.x], cnt[threadIdx.x]);
}

// Pass 2 (all tiles in parallel): every work-group scans the 256-bucket
// histogram (hist[0..255]), reserves a run per bucket for its tiles from the
// cursors (hist[256..511], zero on entry) and writes its tiles there.
__global__ __launch_bounds__(256) void tile_order_kernel(const uint8_t* __restrict__ bucket, uint32_t* __restrict__ hist,
                                                         int num_tiles, uint32_t* __restrict__ order) {
  __shared__ uint32_t start[256], cnt[256], base[256];
  __shared__ uint32_t s_wave[4];
  const int t = blockIdx.x * 256 + threadIdx.x;
  const uint32_t h = hist[threadIdx.x];
  uint32_t total;
  start[threadIdx.x] = block_exclusive_scan<4>(h, s_wave, total);  // 256-lane work-group
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  uint32_t b = 0, rank = 0;
  if (t < num_tiles) {
    b = bucket[t];
    rank = atomicAdd(&cnt[b], 1u);
  }
  __syncthreads();
  if (cnt[threadIdx.x]) base[threadIdx.x] = start[threadIdx.x] + atomicAdd(&hist[256 + threadIdx.x], cnt[threadIdx.x]);
  __syncthreads();
  if (t < num_tiles && base[b] + rank < (uint32_t)num_tiles) order[base[b] + rank] = (uint32_t)t;
}

// The same for few tiles, one work-group and one launch: 5 us where the two passes and the gap between them take 10
// (400 tiles); with more tiles than its lanes hold in registers the two passes win.
constexpr int kOrderLanes = 1024, kOrderTiles = 4;  // per lane
__global__ __launch_bounds__(kOrderLanes) void tile_order_few_kernel(RenderArgs a, uint32_t* __restrict__ order) {
  __shared__ uint32_t cnt[256], start[256];
  __shared__ uint32_t s_wave[kOrderLanes / 64];
  const int tid = threadIdx.x;
  uint32_t K = a.K;
  if (a.K_dev) K = min(K, *a.K_dev);
  if (tid < 256) cnt[tid] = 0u;
  __syncthreads();
  uint32_t b[kOrderTiles], rank[kOrderTiles];
#pragma unroll
  for (int i = 0; i < kOrderTiles; ++i)  // no load is conditional: they are in flight together
    b[i] = tile_cost_bucket(a, min(i * kOrderLanes + tid, a.num_tiles - 1), K, false);
#pragma unroll
  for (int i = 0; i < kOrderTiles; ++i) {
    const int t = i * kOrderLanes + tid;
    if (t >= a.num_tiles) continue;
    rank[i] = atomicAdd(&cnt[b[i]], 1u);
  }
  __syncthreads();
  uint32_t total;
  const uint32_t before = block_exclusive_scan<kOrderLanes / 64>(tid < 256 ? cnt[tid] : 0u, s_wave, total);
  if (tid < 256) start[tid] = before;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kOrderTiles; ++i) {
    const int t = i * kOrderLanes + tid;
    if (t < a.num_tiles) order[start[b[i]] + rank[i]] = (uint32_t)t;
  }
}

static void tile_order_impl(const RenderArgs& a, uint32_t* order, uint8_t* bucket, uint32_t* hist, bool use_work,
                            hipStream_t s, bool hist_zeroed) {
  if (a.num_tiles <= 0 || !a.views) return;
  const unsigned blocks = (unsigned)((a.num_tiles + 255) / 256);
  if (!hist_zeroed) launch_fill_u32(hist, 512, 0u, s);
  hipLaunchKernelGGL(tile_bucket_kernel, dim3(blocks), dim3(256), 0, s, a, bucket, hist, use_work ? 1 : 0);
  hipLaunchKernelGGL(tile_order_kernel, dim3(blocks), dim3(256), 0, s, (const uint8_t*)bucket, hist, a.num_tiles,
                     order);
}

void launch_tile_order(const RenderArgs& a, uint32_t* order, uint8_t* bucket, uint32_t* hist, hipStream_t s,
                       bool hist_zeroed) {
  if (a.views && a.num_tiles > 0 && a.num_tiles <= kOrderLanes * kOrderTiles)
    hipLaunchKernelGGL(tile_order_few_kernel, dim3(1), dim3(kOrderLanes), 0, s, a, order);
  else
    tile_order_impl(a, order, bucket, hist, false, s, hist_zeroed);
}

void launch_tile_order_bwd(const RenderArgs& a, uint32_t* order, uint8_t* bucket, uint32_t* hist, hipStream_t s,
                           bool hist_zeroed) {
  if (a.tile_work) tile_order_impl(a, order, bucket, hist, true, s, hist_zeroed);
}

// Two work-groups per tile while they find idle SIMDs, us before and after: 336 tiles of long lists (500k Gaussians,
// 333x251, near) 196 and 150, 169 tiles (10k, 200x200) 48 and 39, 475 tiles 220 and 171; 512 tiles of 2 views 72 and
// 59, or 23 and 26 where the lists end after a few splats.  625 tiles of such lists 20 and 28, 1024 24 and 33.
constexpr int kSplitTiles = 512;
void launch_render_fwd(const RenderArgs& a, hipStream_t s) {
  if (a.num_tiles <= 0) return;
  const dim3 grid(a.num_tiles), block(256);
  if (a.views && a.num_tiles <= kSplitTiles)
    hipLaunchKernelGGL((render_fwd_quads_kernel<true, true>), dim3(2 * a.num_tiles), block, 0, s, a);
  else if (a.views)
    hipLaunchKernelGGL((render_fwd_quads_kernel<true, false>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((render_fwd_quads_kernel<false, false>), grid, block, 0, s, a);
}

void launch_render_bwd(const RenderArgs& a, hipStream_t s) {
  if (a.num_tiles <= 0) return;
  if (a.seg.cap > 0) {
    launch_fill_u32(a.seg.head, kSegmentParts * kSegmentHeadStride, 0u, s);
    hipLaunchKernelGGL(render_bwd_chain_kernel, dim3(a.num_tiles), dim3(256), 0, s, a);
    hipLaunchKernelGGL((render_bwd_strips_kernel<true, true>), dim3(a.seg.cap + a.num_tiles), dim3(64), 0, s, a);
  } else if (a.views)
    hipLaunchKernelGGL((render_bwd_strips_kernel<true, false>), dim3(a.num_tiles), dim3(64), 0, s, a);
  else
    hipLaunchKernelGGL((render_bwd_strips_kernel<false, false>), dim3(a.num_tiles), dim3(64), 0, s, a);
}

}  // namespace dmgs
