// Internal kernel argument structs and launchers (not part of the C-ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "dmgs_common.h"

namespace dmgs {

struct PreprocessArgs {
  int P;
  int W, H, grid_x, grid_y;
  float tanfovx, tanfovy, focal_x, focal_y, scale_modifier;
  int sh_degree, sh_coeffs;
  const float* means3D;
  const float* scales;
  const float* rotations;
  const float* opacities;
  const float* shs;
  const float* colors_precomp;
  const float* cov3D_precomp;
  const float* viewmatrix;
  const float* projmatrix;
  const float* campos;
  // outputs
  int32_t* radii;
  float4* splats;
  uint32_t* tiles_touched;
  uint32_t* depth_keys;
  uint32_t* order;
};

void launch_preprocess_fwd(const PreprocessArgs& a, hipStream_t s);
void launch_mark_visible(int P, const float* means3D, const float* viewmatrix, uint8_t* present, hipStream_t s);

// ---- scan / sort / binning ----
// Inclusive scan of n uint32 values; scratch must hold scan_scratch_words(n) words.
size_t scan_scratch_words(size_t n);
void launch_inclusive_scan(const uint32_t* in, uint32_t* out, size_t n, uint32_t* scratch, hipStream_t s);
// The same over instance counts, also filling the duplicate's chunk table
// (DupArgs::chunk_first for K output slots; then set DupArgs::chunk_ready).
void launch_inclusive_scan_chunks(const uint32_t* in, uint32_t* out, size_t n, uint32_t* scratch,
                                  uint32_t* chunk_first, uint32_t K, hipStream_t s);

// Depth sort key of a culled entry (never a sort key of a visible one), and
// the far-depth bucket bits of view-major keys.
constexpr uint32_t kSortSkip = 0xFFFFFFFFu;
constexpr uint32_t kFarBucketBits = 0x0F000000u;

// Stable LSD radix sort of (key, value) pairs over bits [0, bits), in passes of
// at most 8 bits.  Data starts in (k0, v0); (k1, v1) is the ping-pong buffer.
// The number of passes is always even, so the result ends in (k0, v0).
size_t radix_scratch_words(size_t n);
// n_dev (optional) holds the actual length on the device; n is then the capacity.
void radix_sort_pairs(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, size_t n, int bits,
                      uint32_t* scratch, hipStream_t s, const uint32_t* n_dev = nullptr);
// The same with as few passes as the bits need (one pass up to 8 bits);
// returns true when the result is in (k1, v1).  first_hist_ready: the first
// pass's block histogram is already in the scratch (see DupArgs::hist).
bool radix_sort_pairs_min_passes(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, size_t n, int bits,
                                 uint32_t* scratch, hipStream_t s, const uint32_t* n_dev = nullptr,
                                 bool first_hist_ready = false);
// Depth sort of a batch's entries straight from the preprocess's keys: k0
// holds n per-entry 32-bit keys, kSortSkip for culled entries.  The first of
// the four passes drops the skipped keys and takes each entry's index as its
// value, and stores the number of kept keys in *n_out, which bounds the
// other passes; the sorted (key, entry) pairs end in (k0, v0).  flags
// (optional, view-major keys only): bit 0 is set when a key lies in the
// far-depth bucket.  The three low bytes are close to uniform and are
// counted with plain LDS atomics.
void radix_sort_entry_keys(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, size_t n, uint32_t* scratch,
                           hipStream_t s, uint32_t* n_out, uint32_t* flags);
// Whether the cell lists are sorted in one pass (of 8 bits, or of 9 on lists of at least 4 M).
bool radix_one_pass(size_t n, int bits);
// One pass of 9 bits over pairs whose digits the duplicate has counted; the sorted pairs are in k1, v1.
void radix_sort_pairs_wide_digit(const uint32_t* k0, const uint32_t* v0, uint32_t* k1, uint32_t* v1, size_t n,
                                 uint32_t* scratch, hipStream_t s, const uint32_t* n_dev);
size_t radix_list_scratch_words(size_t n);  // of either cell-list sort
// Digit width of the first pass of radix_sort_pairs_min_passes, or -1 when
// its blocks are not 4096 keys (the duplicate's chunks) for this n.
int radix_min_passes_first_width(size_t n, int bits);

// tiles_touched gathered into depth order, ready for the scan.
void launch_gather_u32(const uint32_t* src, const uint32_t* idx, uint32_t* dst, int n, hipStream_t s);

// Emit (tile, splat) pairs in depth order.  Single view: grid_x/grid_y give
// the tile grid.  Several views: entry g belongs to view g / per_view, the
// pairs are (binning cell | tile mask << 16, splat) with cells numbered
// globally from that view's cell_base, or with view_major as
// (cell within the view | view << 12 | tile mask << 16).
struct DupArgs {
  int P;                        // depth-sorted entries
  const uint32_t* order;
  const uint32_t* offsets;      // inclusive prefix of tiles touched, in depth order
  const float4* splats;         // single view: radius in s2.z
  const uint2* rects;           // several views: tile rectangles in depth order (pack_rect)
  int grid_x, grid_y;
  const ViewDesc* views;
  uint32_t per_view;
  uint32_t* tile_keys;
  uint32_t* values;
  uint32_t K;                   // capacity of tile_keys / values
  const uint32_t* K_dev;        // optional device count (clamped to K)
  uint32_t* chunk_first;        // duplicate_scratch_words(K) words
  uint32_t slots;               // per chunk (set by the launcher)
  bool chunk_ready;             // chunk_first already filled (launch_inclusive_scan_chunks)
  bool view_major;
  // optional: the first radix pass's histogram (digits = the low hist_bits of
  // a key), written per chunk into the sort scratch (from the K on whose chunks are the sort's blocks)
  uint32_t* hist;
  int hist_bits;
  // optional: words a later step needs zeroed (cleared in shares by the work-groups)
  uint32_t* zero;
  size_t zero_n;
};
size_t duplicate_scratch_words(size_t K);
void launch_duplicate(const DupArgs& a, hipStream_t s);
// key_mask selects the tile / cell id bits of a key (the rest is carried data).
void launch_tile_ranges(const uint32_t* tile_keys, size_t K, uint2* ranges, int num_tiles, hipStream_t s,
                        const uint32_t* K_dev = nullptr, uint32_t key_mask = 0xFFFFFFFFu);
void launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s);
// Ranges of view-major lists sorted on the cell-within-view bits: each
// (view, cell) run is contiguous; ranges are indexed by global cell id
// (views[view].cell_base + cell).
void launch_view_cell_ranges(const uint32_t* keys, size_t K, uint2* ranges, int num_cells, const ViewDesc* views,
                             hipStream_t s, const uint32_t* K_dev, bool ranges_zeroed = false);

// ---- multi-view per-Gaussian stages ----
// Component-major scene parameters (channels x P).
#define DMGS_MV_XYZ 0
#define DMGS_MV_SCALE 3
#define DMGS_MV_ROT 6
#define DMGS_MV_OPACITY 10
#define DMGS_MV_SH 11
#define DMGS_MV_CHANNELS 59
struct MVArgs {
  int P, B, sh_degree;
  float scale_modifier;
  const ViewDesc* views;
  const float* params;       // (59, P)
  float4* splats;            // (B*P) records
  int32_t* radii;            // (B*P)
  uint2* rects;              // (B*P) tile rectangle, pack_rect; 0 when culled
  uint32_t* depth_keys;      // (B*P) depth sort keys (entry_sort_key), kSortSkip for culled entries
  uint32_t* order;           // (B*P)
  float* gacc;               // B*P x DMGS_GACC_STRIDE blend-backward accumulator (gacc_index); zero between backward passes
  float* grads;              // (59, P)
  float* dens;               // optional (3, P): densification statistics (see dmgs_batch)
  uint32_t* status;          // optional: zeroed by the preprocess (flags set by the depth sort)
  int view_major;            // depth keys also order by view (at most 16 views)
};
void launch_mv_preprocess(const MVArgs& a, hipStream_t s);
// rects_sorted[i] = rects[order[i]], counts[i] = its number of binning cells
// (0 for i >= *n_dev when given).
void launch_gather_rects(const uint2* rects, const uint32_t* order, uint2* rects_sorted, uint32_t* counts, size_t n,
                         hipStream_t s, const uint32_t* n_dev = nullptr);
// Reads the accumulator rows of visible entries (the forward blend cleared
// the accumulator; the blend backward filled it).
void launch_mv_geometry_bwd(const MVArgs& a, hipStream_t s);

// ---- one view over a model's own tensors (view.hip) ----
#define DMGS_RAW_SCALES 1     // scales are log-scales
#define DMGS_RAW_ROTATIONS 2  // rotations are not normalised
#define DMGS_RAW_OPACITIES 4  // opacities are logits
constexpr int kTileSums = 64;
struct ViewArgs {
  int P, W, H, grid_x, grid_y;
  float tanfovx, tanfovy, focal_x, focal_y, scale_modifier;
  int sh_degree, sh_coeffs, raw;
  const float* means3D;
  const float* scales;
  const float* rotations;
  const float* opacities;
  const float* shs;             // (P, M, 3), or (P, 1, 3) beside shs_rest
  const float* shs_rest;        // (P, M - 1, 3) with M 4, 9 or 16, or null
  const float* colors_precomp;
  const float* cov3D_precomp;
  const float* viewmatrix;
  const float* projmatrix;
  const float* campos;
  const float* bg;
  // forward outputs
  ViewDesc* view;               // the view's record for the list and blend kernels
  uint32_t* tile_sums;          // kTileSums partial sums of tiles touched
  int32_t* radii;
  float4* splats;
  uint2* rects;
  uint32_t* depth_keys;         // kSortSkip for culled Gaussians
  // backward
  const float* gacc;
  float* dL_dmeans2D;
  float* dL_dmeans3D;
  float* dL_dopacity;
  float* dL_dsh;                // like shs
  float* dL_dsh_rest;
  float* dL_dcolors;            // these may be null
  float* dL_dcov3D;
  float* dL_dscales;
  float* dL_drotations;
};
void launch_view_preprocess(const ViewArgs& a, hipStream_t s);
// counts[0] = *cells, counts[1] = the sum of tile_sums
void launch_view_counts(const uint32_t* cells, const uint32_t* tile_sums, uint32_t* counts, hipStream_t s);
void launch_view_geometry_bwd(const ViewArgs& a, hipStream_t s);
// sigmoid of the SH sum in the view direction (coeffs 1, 4, 9 or 16 per colour)
struct ShSigmoidArgs {
  int n, degree;
  const float* feats;   // (n, 3 M), colour-major or coefficient-major
  const float* xyz;     // (n, 3)
  const float* campos;  // 3
  float* colors;        // (n, 3); read by the backward
  const float* dL_dcolors;
  float* dL_dfeats;
  float* dL_dxyz;
};
void launch_sh_sigmoid(const ShSigmoidArgs& a, int coeffs, bool color_major, bool backward, hipStream_t s);

// ---- blend ----
// List segments of the blend's backward (render.hip).  At most kSegmentTiles tiles: forward and backward blend, us,
// whole lists and segments: 60k / 300k / 1.5M Gaussians, uniform, at 992x992 (3844 tiles) 217 and 203, 367 and 291,
// 861 and 651, face-bound 491k 918 and 573, and 300k and 1.5M clustered 502 and 349, 234 and 297 (lists of few
// members up to where they saturate); at 1920x1080 (8160 tiles, which fill the GPU without) 308 and 397, 389 and 494,
// 739 and 1026, clustered 449 and 550, 349 and 488.  Only lists of more than 256 members: 64 to 300 us slower with 300k.
constexpr int kSegmentTiles = 4096;
constexpr int kSegmentLength = 64;
constexpr int kTileSegments = 256;  // segments of one tile that start from a state, at most
constexpr int kSegmentParts = 16;   // counters of slots, each with its share of them
constexpr int kSegmentHeadStride = 32;  // words between two
constexpr uint32_t kNoSegment = 0xFFFFFFFFu;
struct Segments {
  int cap;               // slots (0: no segments)
  uint32_t* head;        // per part: slots asked for
  uint4* rec;            // per slot: tile, first and one past the last list position
  float2* state;         // per slot: the tile's 256 pixels' BwdPixel behind the segment
  uint32_t* tile_last;   // per tile: where its last segment, which starts from the list's end, begins
};
// Single view: W, H, grid_x, grid_y, bg and the image pointers describe the
// view.  Several views: `views` / `tile_view` map each global tile to its
// view; images, final_T and n_contrib are packed at each view's pixel_base.
struct RenderArgs {
  int W, H, grid_x, grid_y;
  int num_tiles;          // tiles in the launch (all views)
  uint32_t P, K;          // splat records and list capacity (guards for the gathers)
  const uint32_t* K_dev;  // optional device list length (clamped to K)
  const ViewDesc* views;  // optional view table (multi-view)
  const int32_t* tile_view;
  const uint2* ranges;
  const uint32_t* point_list;
  const uint32_t* list_keys;  // multi-view: sorted keys (cell | tile mask << 16) beside point_list
  const float4* splats;
  const float* bg;
  float* out_color;      // (3, H, W)
  float* final_T;        // (H, W)
  uint32_t* n_contrib;   // (H, W)
  // backward only
  const float* dL_dpix;  // (3, H, W)
  float* gacc;           // P x DMGS_GACC_STRIDE floats, two planes (gacc_index)
  // optional (multi-view): work-group slot -> tile, heaviest tiles first
  const uint32_t* tile_order;
  // optional (multi-view, one work-group a tile in the forward): per
  // tile, the largest last contributor of its pixels (the backward's list length)
  uint32_t* tile_work;
  // optional (forward): the backward accumulator, zeroed by the forward's
  // work-groups in equal shares after their blend work
  float4* clear;
  size_t clear_n;  // float4 count
  // and these words (work-group 0): the tile-order histogram the backward's
  // dispatch order starts from
  uint32_t* clear_words;
  int clear_words_n;
  Segments seg;
};
void launch_render_fwd(const RenderArgs& a, hipStream_t s);
// Multi-view: order the a.num_tiles tiles by decreasing list length (a
// binned estimate of their cost) so the longest start first.  bucket: one
// byte per tile, hist: 512 words of scratch.
void launch_tile_order(const RenderArgs& a, uint32_t* order, uint8_t* bucket, uint32_t* hist, hipStream_t s,
                       bool hist_zeroed = false);
// The same with a.tile_work (written by the forward) as each tile's
// cost: the backward's exact list length.
void launch_tile_order_bwd(const RenderArgs& a, uint32_t* order, uint8_t* bucket, uint32_t* hist, hipStream_t s,
                           bool hist_zeroed = false);
void launch_render_bwd(const RenderArgs& a, hipStream_t s);

// ---- geometry backward ----
struct GeometryBwdArgs {
  int P;
  int W, H;
  float tanfovx, tanfovy, focal_x, focal_y, scale_modifier;
  int sh_degree, sh_coeffs;
  const float* means3D;
  const float* scales;
  const float* rotations;
  const float* shs;
  const float* cov3D_precomp;
  const float* viewmatrix;
  const float* projmatrix;
  const float* campos;
  const int32_t* radii;
  const float* gacc;
  // outputs (each may be null when the caller does not want it)
  float* dL_dmeans2D;    // (P, 3)
  float* dL_dcolors;     // (P, 3)
  float* dL_dopacity;    // (P, 1)
  float* dL_dconic;      // (P, 4)
  float* dL_dmeans3D;    // (P, 3)
  float* dL_dcov3D;      // (P, 6)
  float* dL_dsh;         // (P, M, 3)
  float* dL_dscales;     // (P, 3)
  float* dL_drotations;  // (P, 4)
};
void launch_geometry_bwd(const GeometryBwdArgs& a, hipStream_t s);

// ---- mesh binding ----
struct BindArgs {
  int F, G;                 // faces, Gaussians per face
  const float* verts;       // (V, 3)
  const int32_t* faces;     // (F, 3)
  const float* bc;          // (G, 3) shared, or (F*G, 3) per Gaussian
  int bc_per_gaussian;
  // stage 3 parameters (may be null)
  const float* rot2d;       // (F*G, 2)
  const float* scale2d;     // (F*G, 2) log-scales
  float thin_z;
  // stage 2 parameters
  const float* k;           // device scalar tanh(scale_factor) * max_scale
  float rad_base, flat_scale;
  int adaptive;
  // forward outputs
  float* xyz;               // (F*G, 3)
  float* rot;               // (F*G, 4)
  float* scale;             // (F*G, 3)
  float* cov;               // (F*G, 6)
  float* Lmat;              // (F, 9) stage-2 triangle matrices (written by the forward)
  // backward inputs / outputs
  const float* dxyz;
  const float* drot;
  const float* dscale;
  const float* dcov;
  float* dverts;            // (V, 3), accumulated
  float* drot2d;
  float* dscale2d;
  float* dk;                // device scalar, accumulated
  double* dk_ws;            // optional, zeroed: the blocks' parts of dk (bind_cov_workspace_bytes)
};
void launch_bind_fwd(const BindArgs& a, hipStream_t s);
void launch_bind_cov_fwd(const BindArgs& a, hipStream_t s);
void launch_bind_bwd(const BindArgs& a, hipStream_t s);
size_t bind_cov_workspace_bytes();
void launch_faces_in_frustum(int F, const float* verts, const int32_t* faces, const float* proj, uint8_t* mask,
                             hipStream_t s);

// ---- fused L1 + SSIM loss ----
size_t dssim_partials(int C, int H, int W);
uint32_t dssim_tiles(int C, int H, int W);
// RGB views of any sizes in one launch (views: a device table; tile0 and index ascend).
struct DssimView {
  int32_t H, W;
  uint32_t tile0, pix0;  // its first tile of the launch, its first pixel of the packed images
  uint32_t index;        // its place among the losses
  uint32_t pad[3];
};
struct DssimViews {
  const DssimView* views;
  int n;
  uint32_t tiles;
};
void launch_dssim_forward_views(const float* x, const float* y, const float* ystats, const DssimViews& vs,
                                const float* w11, float lam, float* coef, float* partials, float* out, hipStream_t s);
void launch_dssim_backward_views(const float* x, const float* y, const float* coef, const DssimViews& vs,
                                 const float* w11, float lam, const float* dloss, float* dx, hipStream_t s);
// C planes in C / group loss groups of `group` consecutive planes each.
// ystats: the target's blurred maps from launch_dssim_target, or null.
void launch_dssim_forward(const float* x, const float* y, const float* ystats, int C, int group, int H, int W,
                          const float* w11, float lam, float* coef, float* partials, float* out, hipStream_t s);
// stats (2 C planes): G*y, then G*y^2.
void launch_dssim_target(const float* y, int C, int H, int W, const float* w11, float* stats, hipStream_t s);
void launch_dssim_backward(const float* x, const float* y, const float* coef, int C, int group, int H, int W,
                           const float* w11, float lam, const float* dloss, float* dx, hipStream_t s);

// ---- scene / frame conversions ----
constexpr int kMaxRowFloats = 128;   // properties per PLY vertex row
constexpr int kMaxChannels = 128;
struct ChannelMap {
  int channels;                      // entries used in col
  int col[kMaxChannels];             // source index per destination (-1: zero)
};
// params[c][g] = rows[g][map.col[c]] for c < map.channels (59 scene channels)
void launch_rows_to_channels(const float* rows, int64_t P, int row_len, const ChannelMap& map, float* params,
                             hipStream_t s);
// rows[g][j] = params[map.col[j]][g] for j < row_len
void launch_channels_to_rows(const float* params, int64_t P, int row_len, const ChannelMap& map, float* rows,
                             hipStream_t s);
// (3, H*W) float -> H*W*3 bytes of uint8(clamp(x, 0, 1) * 255)
void launch_rgb8(const float* chw, int64_t plane, uint8_t* hwc, hipStream_t s);

}  // namespace dmgs
