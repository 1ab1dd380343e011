// Per-Gaussian stages of one view over a model's own tensors, for gfx950.
//
// The drop-in renderer takes one camera and the tensors a model holds, (P, k) rows; the lists, the blend and
// the sorts are the batched engine's with one view.  Two things are done here so that no pass over HBM exists
// only to prepare an input:
//   * activations: scales may be log-scales, rotations raw quaternions and opacities logits (DMGS_RAW_*); the
//     exp, normalisation and sigmoid then run in these kernels, rounded exactly as torch rounds them, and the
//     backward returns raw gradients;
//   * SH coefficients may come as two tensors, (P, 1, 3) and (P, M - 1, 3).  A row of the second is 180 bytes
//     at degree 3, which no aligned vector load fits, so a work-group copies its 256 rows through LDS with
//     16-byte accesses and its lanes read them there (odd row strides: no bank conflicts).
// The math is the single-view kernels' (gs_math.h), written out with every fused multiply-add named and
// contraction off, in the order the compiler gives preprocess_fwd_kernel and geometry_bwd_kernel: which of two
// products it fuses depends on the surrounding code.  A last-bit difference in a covariance changes a few radii in a
// million Gaussians and the pixels that sit on a blend threshold, and the gradients of long splats are differences
// that magnify one (4e-6 to 1e-3 of the scale and rotation gradients' norm between two choices).  So this route's
// radii and images equal the per-tile-list route's bit for bit, and its gradients those of the same blend sums,
// through torch's activations where the kernels activate.  (The SH gradient is gs_math.h's in both; the tests
// compare it too.)
#include "dmgs_common.h"
#include "dmgs_kernels.h"
#include "gs_math.h"

namespace dmgs {

constexpr int kRows = 256;  // Gaussians per work-group

// kRows rows of R floats in LDS at an odd row stride.
template <int R>
struct LdsRows {
  static constexpr int S = R % 2 ? R : R + 1;
  static constexpr int kIter = (kRows * R / 4 + kRows - 1) / kRows;
  __align__(16) float v[kRows * S];
  __device__ __forceinline__ float* row(int t) { return v + t * S; }
  // rows [0, n) from / to consecutive global rows (16-byte aligned: the first row is a multiple of kRows)
  __device__ __forceinline__ void load(const float* __restrict__ src, int n) {
    float4 x[kIter];  // every load before the first LDS store
    request(src, n, x);
    put(src, n, x);
  }
  // load in two halves; positions past the end read the last vector
  __device__ __forceinline__ void request(const float* __restrict__ src, int n, float4 (&x)[kIter]) {
    const int f4 = n * R / 4;
    const float4* s4 = reinterpret_cast<const float4*>(src);
    if (f4 > 0) {
#pragma unroll
      for (int i = 0; i < kIter; ++i) x[i] = s4[min(i * kRows + (int)threadIdx.x, f4 - 1)];
    }
  }
  __device__ __forceinline__ void put(const float* __restrict__ src, int n, const float4 (&x)[kIter]) {
    const int f4 = n * R / 4, rest = n * R - 4 * f4;
#pragma unroll
    for (int i = 0; i < kIter; ++i) {
      const int f = i * kRows + (int)threadIdx.x;
      if (f < f4) put4(f, x[i]);
    }
    if ((int)threadIdx.x < rest) at(4 * f4 + (int)threadIdx.x) = src[4 * f4 + threadIdx.x];
  }
  __device__ __forceinline__ void store(float* __restrict__ dst, int n) {
    const int f4 = n * R / 4, rest = n * R - 4 * f4;
    float4* d4 = reinterpret_cast<float4*>(dst);
    for (int f = threadIdx.x; f < f4; f += kRows) d4[f] = get4(f);
    if ((int)threadIdx.x < rest) dst[4 * f4 + threadIdx.x] = at(4 * f4 + (int)threadIdx.x);
  }

 private:
  __device__ __forceinline__ float& at(int e) {
    if constexpr (S == R) return v[e];
    return v[e / R * S + e % R];
  }
  __device__ __forceinline__ void put4(int f, float4 x) {
    if constexpr (S == R) {
      reinterpret_cast<float4*>(v)[f] = x;
    } else {
      at(4 * f) = x.x;
      at(4 * f + 1) = x.y;
      at(4 * f + 2) = x.z;
      at(4 * f + 3) = x.w;
    }
  }
  __device__ __forceinline__ float4 get4(int f) {
    if constexpr (S == R) return reinterpret_cast<float4*>(v)[f];
    return make_float4(at(4 * f), at(4 * f + 1), at(4 * f + 2), at(4 * f + 3));
  }
};

__device__ __forceinline__ float view_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// torch.nn.functional.normalize of a row of four, x / max(norm, 1e-12): the norm's pairwise sum without contraction
constexpr float kNormEps = 1e-12f;
__device__ __forceinline__ float quat_norm(float4 q) {
#pragma clang fp contract(off)
  return sqrtf((q.x * q.x + q.y * q.y) + (q.z * q.z + q.w * q.w));
}
// Its gradient, rounded as torch's operations round it: dq / n, and through the norm, whose own gradient is the
// pairwise sum of -dq (q / n) (q the normalised row).
__device__ __forceinline__ float4 quat_norm_backward(float4 q, float norm, float4 dq) {
#pragma clang fp contract(off)
  const float n = fmaxf(norm, kNormEps);
  const float dn = norm >= kNormEps ? (-dq.x * (q.x / n) + -dq.y * (q.y / n)) + (-dq.z * (q.z / n) + -dq.w * (q.w / n)) : 0.f;
  return make_float4(dq.x / n + dn * q.x, dq.y / n + dn * q.y, dq.z / n + dn * q.z, dq.w / n + dn * q.w);
}

// One Gaussian's SH coefficients: the first three from registers, the others from its LDS row.
struct ShSplit {
  const float* dc;
  const float* rest;
  int n;
  __device__ __forceinline__ float operator[](int k) const { return k < 3 ? dc[k] : (k - 3 < n ? rest[k - 3] : 0.f); }
};
struct ShRow {
  const float* row;
  int n;
  __device__ __forceinline__ float operator[](int k) const { return k < n ? row[k] : 0.f; }
};

struct ViewGaussian {
  float3 e, s;   // scale, modifier x scale
  float4 q;      // rotation as the covariance uses it
  float qn;      // norm of the raw quaternion
  float R[9], c3[6];
};

// Rotation matrix and Sigma = R diag(s)^2 R^T (quat_to_R, cov3d_from_sR).
__device__ __forceinline__ void view_cov3d(ViewGaussian& G) {
#pragma clang fp contract(off)
  const float r = G.q.x, x = G.q.y, y = G.q.z, z = G.q.w;
  const float zz = z * z, rz = r * z, ry = r * y, yz = y * z, yy = y * y;
  float* R = G.R;
  R[0] = fmaf(fmaf(y, y, zz), -2.0f, 1.0f);
  R[1] = 2.0f * fmaf(x, y, -rz);
  R[2] = 2.0f * fmaf(x, z, ry);
  R[3] = 2.0f * fmaf(x, y, rz);
  R[4] = fmaf(fmaf(x, x, zz), -2.0f, 1.0f);
  R[5] = 2.0f * fmaf(-r, x, yz);
  R[6] = 2.0f * fmaf(x, z, -ry);
  R[7] = 2.0f * fmaf(r, x, yz);
  R[8] = fmaf(fmaf(x, x, yy), -2.0f, 1.0f);
  const float M00 = G.s.x * R[0], M01 = G.s.y * R[1], M02 = G.s.z * R[2];
  const float M10 = G.s.x * R[3], M11 = G.s.y * R[4], M12 = G.s.z * R[5];
  const float M20 = G.s.x * R[6], M21 = G.s.y * R[7], M22 = G.s.z * R[8];
  G.c3[0] = fmaf(M02, M02, fmaf(M01, M01, M00 * M00));
  G.c3[1] = fmaf(M02, M12, fmaf(M10, M00, M01 * M11));
  G.c3[2] = fmaf(M02, M22, fmaf(M01, M21, M20 * M00));
  G.c3[3] = fmaf(M12, M12, fmaf(M10, M10, M11 * M11));
  G.c3[4] = fmaf(M12, M22, fmaf(M10, M20, M21 * M11));
  G.c3[5] = fmaf(M22, M22, fmaf(M20, M20, M21 * M21));
}

// project_splat of gs_math.h.
__device__ __forceinline__ bool view_project(float3 p, const float (&c)[6], const ViewParams& v, SplatGeom& o) {
#pragma clang fp contract(off)
  const float* vm = v.vm;
  const float* pm = v.pm;
  const float tz = fmaf(vm[10], p.z, fmaf(vm[2], p.x, vm[6] * p.y)) + vm[14];
  if (tz <= 0.2f) return false;
  const float tx0 = fmaf(vm[8], p.z, fmaf(vm[4], p.y, vm[0] * p.x)) + vm[12];
  const float ty0 = fmaf(vm[9], p.z, fmaf(vm[5], p.y, vm[1] * p.x)) + vm[13];
  const float limx = 1.3f * v.tanx, limy = 1.3f * v.tany;
  const float tx = fminf(limx, fmaxf(-limx, tx0 / tz)) * tz;
  const float ty = fminf(limy, fmaxf(-limy, ty0 / tz)) * tz;
  const float iz = 1.0f / tz, iz2 = iz * iz;
  const float j00 = v.fx * iz, j02 = -(v.fx * tx) * iz2;
  const float j11 = v.fy * iz, j12 = -(v.fy * ty) * iz2;
  const float m00 = fmaf(j00, vm[0], j02 * vm[2]), m01 = fmaf(j00, vm[4], j02 * vm[6]);
  const float m02 = fmaf(j00, vm[8], j02 * vm[10]);
  const float m10 = fmaf(j11, vm[1], j12 * vm[2]), m11 = fmaf(j11, vm[5], j12 * vm[6]);
  const float m12 = fmaf(j11, vm[9], j12 * vm[10]);
  const float s0x = fmaf(c[2], m02, fmaf(c[0], m00, c[1] * m01));
  const float s0y = fmaf(c[4], m02, fmaf(c[1], m00, c[3] * m01));
  const float s0z = fmaf(c[5], m02, fmaf(c[2], m00, c[4] * m01));
  const float s1x = fmaf(c[2], m12, fmaf(c[0], m10, c[1] * m11));
  const float s1y = fmaf(c[4], m12, fmaf(c[1], m10, c[3] * m11));
  const float s1z = fmaf(c[5], m12, fmaf(c[2], m10, c[4] * m11));
  const float ca = fmaf(m02, s0z, fmaf(m00, s0x, m01 * s0y)) + 0.3f;
  const float cb = fmaf(m12, s0z, fmaf(m10, s0x, m11 * s0y));
  const float cc = fmaf(m12, s1z, fmaf(m10, s1x, m11 * s1y)) + 0.3f;
  const float det = fmaf(cc, ca, -(cb * cb));
  if (det == 0.0f) return false;
  const float phw = (fmaf(pm[11], p.z, fmaf(pm[3], p.x, pm[7] * p.y)) + pm[15]) + 0.0000001f;
  const float phx = fmaf(pm[8], p.z, fmaf(pm[0], p.x, pm[4] * p.y)) + pm[12];
  const float phy = fmaf(pm[9], p.z, fmaf(pm[1], p.x, pm[5] * p.y)) + pm[13];
  const float pw = 1.0f / phw, det_inv = 1.0f / det;
  const float sum = ca + cc, mid = 0.5f * sum;
  const float disc = sqrtf(fmaxf(0.1f, fmaf(mid, mid, -det)));
  const float radius = ceilf(3.f * sqrtf(fmaxf(fmaf(0.5f, sum, disc), fmaf(0.5f, sum, -disc))));
  o.pix = make_float2(0.5f * fmaf(fmaf(phx, pw, 1.0f), (float)v.W, -1.0f),
                      0.5f * fmaf(fmaf(phy, pw, 1.0f), (float)v.H, -1.0f));
  tile_rect(o.pix, (int)radius, v.gx, v.gy, o.rmin, o.rmax);
  o.tiles = (o.rmax.x - o.rmin.x) * (o.rmax.y - o.rmin.y);
  if (o.tiles == 0) return false;
  o.conic = make_float3(cc * det_inv, -cb * det_inv, ca * det_inv);
  o.radius = (int)radius;
  o.depth = tz;
  return true;
}

// ewa_backward of gs_math.h as geometry_bwd_kernel has it: dL/dSigma in dc, dL/dmean returned.
__device__ __forceinline__ float3 view_ewa_backward(float3 p, const float (&c)[6], const ViewParams& v, float dmx,
                                                    float dmy, float dqa, float dqb, float dqc, float (&dc)[6]) {
#pragma clang fp contract(off)
  const float* vm = v.vm;
  const float* pm = v.pm;
  const float tz = fmaf(vm[10], p.z, fmaf(vm[2], p.x, vm[6] * p.y)) + vm[14];
  const float tx0 = fmaf(vm[8], p.z, fmaf(vm[0], p.x, vm[4] * p.y)) + vm[12];
  const float ty0 = fmaf(vm[9], p.z, fmaf(vm[1], p.x, vm[5] * p.y)) + vm[13];
  const float limx = 1.3f * v.tanx, limy = 1.3f * v.tany;
  const float txtz = tx0 / tz, tytz = ty0 / tz;
  const float tx = tz * fminf(limx, fmaxf(-limx, txtz)), ty = tz * fminf(limy, fmaxf(-limy, tytz));
  const float xmul = (txtz < -limx || txtz > limx) ? 0.f : 1.f;
  const float ymul = (tytz < -limy || tytz > limy) ? 0.f : 1.f;
  const float iz = __builtin_amdgcn_rcpf(tz), iz2 = iz * iz, iz3 = iz * iz2;
  const float fx = v.fx, fy = v.fy;
  const float j00 = fx * iz, j02 = iz2 * (fx * -tx), j11 = fy * iz, j12 = iz2 * (fy * -ty);
  const float V0[3] = {vm[0], vm[4], vm[8]}, V1[3] = {vm[1], vm[5], vm[9]}, V2[3] = {vm[2], vm[6], vm[10]};
  float m0[3], m1[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    m0[k] = fmaf(V0[k], j00, V2[k] * j02);
    m1[k] = fmaf(V1[k], j11, V2[k] * j12);
  }
  float S0[3], S1[3];  // Sigma m0, Sigma m1
  S0[0] = fmaf(c[2], m0[2], fmaf(c[0], m0[0], c[1] * m0[1]));
  S0[1] = fmaf(c[4], m0[2], fmaf(c[1], m0[0], c[3] * m0[1]));
  S0[2] = fmaf(c[5], m0[2], fmaf(c[2], m0[0], c[4] * m0[1]));
  S1[0] = fmaf(c[2], m1[2], fmaf(c[0], m1[0], c[1] * m1[1]));
  S1[1] = fmaf(c[4], m1[2], fmaf(c[1], m1[0], c[3] * m1[1]));
  S1[2] = fmaf(c[5], m1[2], fmaf(c[2], m1[0], c[4] * m1[1]));
  const float ca = fmaf(m0[2], S0[2], fmaf(m0[0], S0[0], m0[1] * S0[1])) + 0.3f;
  const float cb = fmaf(m1[2], S0[2], fmaf(m1[0], S0[0], m1[1] * S0[1]));
  const float cc = fmaf(m1[2], S1[2], fmaf(m1[0], S1[0], m1[1] * S1[1])) + 0.3f;
  // conic -> cov2D
  const float ac = ca * cc, denom = fmaf(-cb, cb, ac);
  const float d2inv = __builtin_amdgcn_rcpf(fmaf(denom, denom, 0.0000001f));
  float dLa = 0.f, dLb = 0.f, dLc = 0.f;
  if (d2inv != 0.f) {
    const float cb2 = cb + cb, e = denom - ac;
    dLa = d2inv * fmaf(dqc, e, fmaf(dqb, cb2 * cc, -(dqa * (cc * cc))));
    dLc = d2inv * fmaf(dqa, e, fmaf(dqb, cb * (ca + ca), -(dqc * (ca * ca))));
    dLb = (d2inv + d2inv) * fmaf(dqc, cb * ca, fmaf(dqa, cb * cc, -(dqb * fmaf(cb, cb2, denom))));
  }
  // cov2D -> cov3D (6-vector)
  const float dLa2 = dLa + dLa, dLc2 = dLc + dLc;
  auto square = [&](int k) { return fmaf(m1[k], m1[k] * dLc, fmaf(m1[k], m0[k] * dLb, m0[k] * (m0[k] * dLa))); };
  auto mixed = [&](int i, int j) {
    return fmaf(m1[j], m1[i] * dLc2, fmaf(fmaf(m1[j], m0[i], m1[i] * m0[j]), dLb, m0[j] * (m0[i] * dLa2)));
  };
  dc[0] = square(0);
  dc[1] = mixed(0, 1);
  dc[2] = mixed(0, 2);
  dc[3] = square(1);
  dc[4] = mixed(1, 2);
  dc[5] = square(2);
  // cov2D -> J -> t -> mean
  float dm0[3], dm1[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    dm0[k] = fmaf(S1[k], dLb, S0[k] * dLa2);
    dm1[k] = fmaf(S1[k], dLc2, S0[k] * dLb);
  }
  auto along = [](const float (&V)[3], const float (&d)[3]) { return fmaf(V[2], d[2], fmaf(V[0], d[0], V[1] * d[1])); };
  const float dj00 = along(V0, dm0), dj02 = along(V2, dm0), dj11 = along(V1, dm1), dj12 = along(V2, dm1);
  const float dtx = iz2 * (xmul * -fx) * dj02, dty = iz2 * (ymul * -fy) * dj12;
  const float dtz = fmaf(iz3 * ((fy + fy) * ty), dj12,
                         fmaf(iz3 * ((fx + fx) * tx), dj02, fmaf(iz2 * -fx, dj00, -((fy * iz2) * dj11))));
  // projection (means2D gradient is in NDC)
  const float phw = fmaf(pm[11], p.z, fmaf(pm[3], p.x, pm[7] * p.y)) + pm[15];
  const float phx = fmaf(pm[8], p.z, fmaf(pm[0], p.x, pm[4] * p.y)) + pm[12];
  const float phy = fmaf(pm[9], p.z, fmaf(pm[1], p.x, pm[5] * p.y)) + pm[13];
  const float mw = __builtin_amdgcn_rcpf(phw + 0.0000001f);
  const float mul1 = mw * (phx * mw), mul2 = mw * (phy * mw);
  auto mean = [&](int k) {
    return fmaf(dmx, fmaf(pm[4 * k], mw, -(pm[4 * k + 3] * mul1)),
                dmy * fmaf(pm[4 * k + 1], mw, -(pm[4 * k + 3] * mul2))) +
           fmaf(vm[4 * k + 2], dtz, fmaf(vm[4 * k + 1], dty, vm[4 * k] * dtx));
  };
  return make_float3(mean(0), mean(1), mean(2));
}

// cov3d_backward of gs_math.h, likewise.
__device__ __forceinline__ void view_cov3d_backward(const float (&dc)[6], float3 s3, const float (&R)[9], float4 q,
                                                    float3& ds, float4& dq) {
#pragma clang fp contract(off)
  // dL/dM = 2 G M, M = R diag(s); off the diagonal G has half of dc
  const float G01 = 0.5f * dc[1], G02 = 0.5f * dc[2], G12 = 0.5f * dc[4];
  const float sv[3] = {s3.x, s3.y, s3.z};
  float d[3], g[9];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const float two_s = sv[j] + sv[j], R0 = R[j], R1 = R[3 + j], R2 = R[6 + j];
    const float dM0 = two_s * fmaf(R2, G02, fmaf(R0, dc[0], R1 * G01));
    const float dM1 = two_s * fmaf(R2, G12, fmaf(R1, dc[3], R0 * G01));
    const float dM2 = two_s * fmaf(R2, dc[5], fmaf(R0, G02, R1 * G12));
    d[j] = fmaf(R2, dM2, fmaf(R0, dM0, R1 * dM1));
    g[j] = sv[j] * dM0;
    g[3 + j] = sv[j] * dM1;
    g[6 + j] = sv[j] * dM2;
  }
  ds = make_float3(d[0], d[1], d[2]);
  const float r = q.x, x = q.y, y = q.z, z = q.w, x2 = x + x, y2 = y + y, z2 = z + z;
  const float dr = fmaf(x, g[7], fmaf(-y, g[6], fmaf(-x, g[5], fmaf(z, g[3], fmaf(y, g[2], -(z * g[1]))))));
  const float dx = fmaf(-x2, g[8], fmaf(r, g[7], fmaf(z, g[6], fmaf(-r, g[5],
                        fmaf(-x2, g[4], fmaf(y, g[3], fmaf(y, g[1], z * g[2])))))));
  const float dy = fmaf(-y2, g[8], fmaf(z, g[7], fmaf(-r, g[6], fmaf(z, g[5],
                        fmaf(x, g[3], fmaf(r, g[2], fmaf(x, g[1], -(y2 * g[0]))))))));
  const float dz = fmaf(y, g[7], fmaf(x, g[6], fmaf(y, g[5], fmaf(-z2, g[4],
                        fmaf(r, g[3], fmaf(x, g[2], fmaf(-z2, g[0], -(r * g[1]))))))));
  dq = make_float4(dr + dr, dx + dx, dy + dy, dz + dz);
}

// The SH sum of sh_to_rgb (gs_math.h) in the view direction.
template <typename SH>
__device__ __forceinline__ float3 view_sh(int deg, const SH& sh, float3 p, const float (&campos)[3]) {
#pragma clang fp contract(off)
  float3 r = make_float3(kSH_C0 * sh[0], kSH_C0 * sh[1], kSH_C0 * sh[2]);
  auto add = [&](int k, float b) {
    r = make_float3(fmaf(b, sh[3 * k], r.x), fmaf(b, sh[3 * k + 1], r.y), fmaf(b, sh[3 * k + 2], r.z));
  };
  if (deg > 0) {
    const float dx = p.x - campos[0], dy = p.y - campos[1], dz = p.z - campos[2];
    const float inv = 1.0f / sqrtf(fmaf(dz, dz, fmaf(dx, dx, dy * dy)));
    const float x = dx * inv, y = dy * inv, z = dz * inv;
    const float b1 = -kSH_C1 * y, b2 = kSH_C1 * z, b3 = -kSH_C1 * x;
    r = make_float3(fmaf(b3, sh[9], fmaf(b2, sh[6], b1 * sh[3])) + r.x, fmaf(b3, sh[10], fmaf(b2, sh[7], b1 * sh[4])) + r.y,
                    fmaf(b3, sh[11], fmaf(b2, sh[8], b1 * sh[5])) + r.z);
    if (deg > 1) {
      const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
      const float d = fmaf(x, x, -yy);
      add(4, kSH_C2[0] * xy);
      add(5, kSH_C2[1] * yz);
      add(6, kSH_C2[2] * fmaf(-y, y, fmaf(zz, 2.0f, -xx)));
      add(7, kSH_C2[3] * xz);
      add(8, kSH_C2[4] * d);
      if (deg > 2) {
        const float q = fmaf(zz, 4.0f, -xx) - yy;
        add(9, (kSH_C3[0] * y) * fmaf(xx, 3.0f, -yy));
        add(10, z * (kSH_C3[1] * xy));
        add(11, (kSH_C3[2] * y) * q);
        add(12, (kSH_C3[3] * z) * fmaf(-3.0f, yy, fmaf(-3.0f, xx, zz + zz)));
        add(13, (kSH_C3[4] * x) * q);
        add(14, (kSH_C3[5] * z) * d);
        add(15, (kSH_C3[6] * x) * fmaf(-3.0f, yy, xx));
      }
    }
  }
  return r;
}
template <typename SH>
__device__ __forceinline__ float3 view_rgb(int deg, const SH& sh, float3 p, const float (&campos)[3]) {
  const float3 r = view_sh(deg, sh, p, campos);
  return make_float3(fmaxf(r.x + 0.5f, 0.0f), fmaxf(r.y + 0.5f, 0.0f), fmaxf(r.z + 0.5f, 0.0f));
}

__device__ __forceinline__ void load_shape(const ViewArgs& a, int g, ViewGaussian& G) {
  if (a.cov3D_precomp) {
#pragma unroll
    for (int k = 0; k < 6; ++k) G.c3[k] = a.cov3D_precomp[6 * (size_t)g + k];
    return;
  }
  G.e = make_float3(a.scales[3 * (size_t)g], a.scales[3 * (size_t)g + 1], a.scales[3 * (size_t)g + 2]);
  G.q = reinterpret_cast<const float4*>(a.rotations)[g];
}
__device__ __forceinline__ void make_shape(const ViewArgs& a, ViewGaussian& G) {
  if (a.cov3D_precomp) return;
  if (a.raw & DMGS_RAW_SCALES) G.e = make_float3(expf(G.e.x), expf(G.e.y), expf(G.e.z));
  const float m = a.scale_modifier;
  G.s = make_float3(m * G.e.x, m * G.e.y, m * G.e.z);
  G.qn = 1.0f;
  if (a.raw & DMGS_RAW_ROTATIONS) {
    G.qn = quat_norm(G.q);
    const float n = fmaxf(G.qn, kNormEps);
    G.q = make_float4(G.q.x / n, G.q.y / n, G.q.z / n, G.q.w / n);
  }
  view_cov3d(G);
}

__global__ __launch_bounds__(64) void view_setup_kernel(ViewArgs a) {
  const int t = threadIdx.x;
  ViewDesc& v = *a.view;
  a.tile_sums[t] = 0u;
  if (t < 16) {
    v.view[t] = a.viewmatrix[t];
    v.proj[t] = a.projmatrix[t];
  }
  if (t < 4) {
    v.campos[t] = t < 3 ? a.campos[t] : 0.f;
    v.bg[t] = t < 3 ? a.bg[t] : 0.f;
  }
  if (t == 0) {
    v.tanfovx = a.tanfovx;
    v.tanfovy = a.tanfovy;
    v.focal_x = a.focal_x;
    v.focal_y = a.focal_y;
    v.W = a.W;
    v.H = a.H;
    v.grid_x = a.grid_x;
    v.grid_y = a.grid_y;
    v.tile_base = v.cell_base = 0;
    v.pixel_base = 0;
  }
}

// REST: floats in a row of the second SH tensor (3 (M - 1)), or -1: one SH tensor of any M, or given colours.
// Bound by memory: 1 M Gaussians of degree
// 3 at 1080p 62 us (240 bytes a row read, 60 written: 4.8 TB/s), at 800 x 800 with a backward's buffers 76; 82 before
// the Gaussian's own loads went out ahead of the rows.  Over one SH tensor it takes 56 us, after the concatenation
// (124 us) and the activations that this kernel does without.
template <int REST>
__global__ __launch_bounds__(kRows) void view_preprocess_kernel(ViewArgs a) {
  __shared__ LdsRows<(REST > 0 ? REST : 1)> rows;
  __shared__ uint32_t s_tiles;
  const int g0 = blockIdx.x * kRows, g = g0 + (int)threadIdx.x;
  const bool live = g < a.P;
  const size_t i = live ? (size_t)g : 0;
  if (threadIdx.x == 0) s_tiles = 0u;
  // the Gaussian's own loads, then the rows', all in flight together; the projection runs while the rows arrive
  const float3 p = make_float3(a.means3D[3 * i], a.means3D[3 * i + 1], a.means3D[3 * i + 2]);
  ViewGaussian G;
  load_shape(a, i, G);
  const float op = a.opacities[i];
  float dc[3] = {0.f, 0.f, 0.f};
  if constexpr (REST >= 0)
    if (!a.colors_precomp)
      for (int k = 0; k < 3; ++k) dc[k] = a.shs[3 * i + k];
  float4 x[LdsRows<(REST > 0 ? REST : 1)>::kIter];
  const int n = min(kRows, a.P - g0);
  if constexpr (REST > 0) rows.request(a.shs_rest + (size_t)g0 * REST, n, x);
  const ViewParams v = view_params(a.viewmatrix, a.projmatrix, a.campos, a.W, a.H, a.grid_x, a.grid_y, a.focal_x,
                                   a.focal_y, a.tanfovx, a.tanfovy);
  make_shape(a, G);
  SplatGeom o;
  const bool seen = view_project(p, G.c3, v, o) && live;
  if constexpr (REST > 0) rows.put(a.shs_rest + (size_t)g0 * REST, n, x);
  __syncthreads();
  uint32_t tiles = 0;
  if (live) {
    if (!seen) {
      a.radii[g] = 0;
      a.depth_keys[g] = kSortSkip;
    } else {
      float3 rgb;
      if (a.colors_precomp) {
        rgb = make_float3(a.colors_precomp[3 * (size_t)g], a.colors_precomp[3 * (size_t)g + 1],
                          a.colors_precomp[3 * (size_t)g + 2]);
      } else {
        if constexpr (REST >= 0) {
          rgb = view_rgb(a.sh_degree, ShSplit{dc, rows.row(threadIdx.x), REST}, p, v.campos);
        } else {
          float sh[48];
          load_sh16(a.shs + (size_t)g * a.sh_coeffs * 3, a.sh_coeffs, sh);
          rgb = view_rgb(a.sh_degree, sh, p, v.campos);
        }
      }
      float4* sp = a.splats + (size_t)DMGS_SPLAT_F4 * g;
      sp[0] = make_float4(o.pix.x, o.pix.y, o.conic.x, o.conic.y);
      sp[1] = make_float4(o.conic.z, a.raw & DMGS_RAW_OPACITIES ? view_sigmoid(op) : op, rgb.x, rgb.y);
      sp[2] = make_float4(rgb.z, o.depth, __int_as_float(o.radius), 0.0f);
      a.radii[g] = o.radius;
      a.rects[g] = pack_rect(o.rmin, o.rmax);
      a.depth_keys[g] = __float_as_uint(o.depth);
      tiles = (uint32_t)o.tiles;
    }
  }
  if (tiles) atomicAdd(&s_tiles, tiles);
  __syncthreads();
  if (threadIdx.x == 0 && s_tiles) atomicAdd(&a.tile_sums[blockIdx.x % kTileSums], s_tiles);
}

__global__ __launch_bounds__(64) void view_counts_kernel(const uint32_t* __restrict__ cells,
                                                         const uint32_t* __restrict__ tile_sums,
                                                         uint32_t* __restrict__ counts) {
  uint32_t x = tile_sums[threadIdx.x];
  for (int off = 32; off > 0; off >>= 1) x += (uint32_t)__shfl_xor((int)x, off, 64);
  if (threadIdx.x == 0) {
    counts[0] = *cells;
    counts[1] = x;
  }
}

// The blend backward's accumulator to the gradients of the model's tensors.  Bound by memory: 1 M Gaussians of degree 3
// 97 us (496 MB at 5.1 TB/s), where a kernel of strided rows took 167 and the gradients' split and the activations'
// backward 93 and 100 more.
// SPLIT: two SH tensors of 1 and M - 1 coefficients; M = 0: given colours; M < 0: one SH tensor of any M.
template <int M, bool SPLIT>
__global__ __launch_bounds__(kRows) void view_geometry_bwd_kernel(ViewArgs a) {
  constexpr int R = M > 0 ? (SPLIT ? 3 * (M - 1) : 3 * M) : 0;
  __shared__ LdsRows<(R > 0 ? R : 1)> rows;
  const int g0 = blockIdx.x * kRows, g = g0 + (int)threadIdx.x;
  const int n = min(kRows, a.P - g0);
  if constexpr (R > 0) rows.load((SPLIT ? a.shs_rest : a.shs) + (size_t)g0 * R, n);
  const bool live = g < a.P;
  const size_t i = live ? (size_t)g : 0;
  const float2* gg = reinterpret_cast<const float2*>(a.gacc + gacc_index(a.P, i, 0));
  const float2 r0 = gg[0], r1 = gg[1], r2 = gg[2];
  const float* gc = a.gacc + gacc_index(a.P, i, DMGS_GACC_GEO);
  const float3 dcol = make_float3(gc[0], gc[1], gc[2]);
  const bool vis = live && a.radii[i] > 0;
  const float3 p = make_float3(a.means3D[3 * i], a.means3D[3 * i + 1], a.means3D[3 * i + 2]);
  float3 dmean = make_float3(0.f, 0.f, 0.f), ds = dmean;
  float4 dq = make_float4(0.f, 0.f, 0.f, 0.f);
  float dc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const ViewParams v = view_params(a.viewmatrix, a.projmatrix, a.campos, a.W, a.H, 0, 0, a.focal_x, a.focal_y,
                                   a.tanfovx, a.tanfovy);
  if (vis) {
    ViewGaussian G;
    load_shape(a, g, G);
    make_shape(a, G);
    dmean = view_ewa_backward(p, G.c3, v, r0.x, r0.y, r1.x, r1.y, r2.x, dc);
    if (!a.cov3D_precomp) {
      view_cov3d_backward(dc, G.s, G.R, G.q, ds, dq);
      if (a.raw & DMGS_RAW_SCALES)  // scale = exp(log-scale)
        ds = make_float3(ds.x * G.e.x, ds.y * G.e.y, ds.z * G.e.z);
      if (a.raw & DMGS_RAW_ROTATIONS) dq = quat_norm_backward(G.q, G.qn, dq);
    }
  }
  if constexpr (M != 0) {
    float b[16];
    float3 gm = make_float3(0.f, 0.f, 0.f);
    auto add = [&](float3 d) { dmean = make_float3(dmean.x + d.x, dmean.y + d.y, dmean.z + d.z); };
#pragma unroll
    for (int k = 0; k < 16; ++k) b[k] = 0.f;
    if constexpr (M > 0) {
      __syncthreads();  // the rows are in LDS
      float* row = rows.row(threadIdx.x);
      if (vis) {
        if constexpr (SPLIT) {
          const float c0[3] = {a.shs[3 * i], a.shs[3 * i + 1], a.shs[3 * i + 2]};
          add(sh_backward(a.sh_degree, ShSplit{c0, row, R}, p, v.campos, dcol, b, gm));
        } else {
          add(sh_backward(a.sh_degree, ShRow{row, R}, p, v.campos, dcol, b, gm));
        }
      }
      // the lane's row becomes its gradient
#pragma unroll
      for (int k = SPLIT ? 1 : 0; k < M; ++k) {
        const int o = 3 * (SPLIT ? k - 1 : k);
        row[o] = b[k] * gm.x;
        row[o + 1] = b[k] * gm.y;
        row[o + 2] = b[k] * gm.z;
      }
      if (SPLIT && live) {
        a.dL_dsh[3 * i] = b[0] * gm.x;
        a.dL_dsh[3 * i + 1] = b[0] * gm.y;
        a.dL_dsh[3 * i + 2] = b[0] * gm.z;
      }
      __syncthreads();
      if constexpr (R > 0) rows.store((SPLIT ? a.dL_dsh_rest : a.dL_dsh) + (size_t)g0 * R, n);
    } else if (live) {
      if (vis) {
        float sh[48];
        load_sh16(a.shs + i * 3 * a.sh_coeffs, a.sh_coeffs, sh);
        add(sh_backward(a.sh_degree, sh, p, v.campos, dcol, b, gm));
      }
      float* d = a.dL_dsh + i * 3 * a.sh_coeffs;
      for (int k = 0; k < a.sh_coeffs; ++k) {
        float bk = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) bk = j == k ? b[j] : bk;
        d[3 * k] = bk * gm.x;
        d[3 * k + 1] = bk * gm.y;
        d[3 * k + 2] = bk * gm.z;
      }
    }
  }
  if (!live) return;
  auto put3 = [&](float* o, float x, float y, float z) {
    o[3 * i] = x;
    o[3 * i + 1] = y;
    o[3 * i + 2] = z;
  };
  put3(a.dL_dmeans2D, r0.x, r0.y, 0.f);
  put3(a.dL_dmeans3D, dmean.x, dmean.y, dmean.z);
  float dop = r2.y;
  if (a.raw & DMGS_RAW_OPACITIES) {
    const float o = view_sigmoid(a.opacities[i]);
    dop = dop * (1.0f - o) * o;
  }
  a.dL_dopacity[i] = dop;
  if (a.dL_dcolors) put3(a.dL_dcolors, dcol.x, dcol.y, dcol.z);
  if (a.dL_dcov3D) {
#pragma unroll
    for (int k = 0; k < 6; ++k) a.dL_dcov3D[6 * i + k] = dc[k];
  }
  if (a.dL_dscales) put3(a.dL_dscales, ds.x, ds.y, ds.z);
  if (a.dL_drotations) reinterpret_cast<float4*>(a.dL_drotations)[i] = dq;
}

// ---- colours outside the rasterizer: sigmoid of the SH sum ----
// One pass forward and one backward instead of about 300 elementwise launches over (N, 3) and (N, 3, M) tensors.
// Bound by the rows, staged through LDS so that global accesses are 16 bytes a lane in order; 122 880 rows of 48:
// 7 us forward (26 MB) and 11 us backward (52 MB), where the elementwise launches took about 1600 us together.
// A row is M coefficients of three colours, colour-major (C, M) or coefficient-major (M, C).
template <int M, bool COLOR_MAJOR>
struct ShRowAny {
  const float* row;
  __device__ __forceinline__ static int at(int i) { return COLOR_MAJOR ? M * (i % 3) + i / 3 : i; }
  __device__ __forceinline__ float operator[](int i) const { return i < 3 * M ? row[at(i)] : 0.f; }
};

template <int M, bool COLOR_MAJOR>
__global__ __launch_bounds__(kRows) void sh_sigmoid_fwd_kernel(ShSigmoidArgs a) {
  __shared__ LdsRows<3 * M> rows;
  const int g0 = blockIdx.x * kRows, g = g0 + (int)threadIdx.x;
  rows.load(a.feats + (size_t)g0 * 3 * M, min(kRows, a.n - g0));
  __syncthreads();
  if (g >= a.n) return;
  const float3 p = make_float3(a.xyz[3 * (size_t)g], a.xyz[3 * (size_t)g + 1], a.xyz[3 * (size_t)g + 2]);
  const float cp[3] = {a.campos[0], a.campos[1], a.campos[2]};
  const float3 r = view_sh(a.degree, ShRowAny<M, COLOR_MAJOR>{rows.row(threadIdx.x)}, p, cp);
  a.colors[3 * (size_t)g] = view_sigmoid(r.x);
  a.colors[3 * (size_t)g + 1] = view_sigmoid(r.y);
  a.colors[3 * (size_t)g + 2] = view_sigmoid(r.z);
}

template <int M, bool COLOR_MAJOR>
__global__ __launch_bounds__(kRows) void sh_sigmoid_bwd_kernel(ShSigmoidArgs a) {
  __shared__ LdsRows<3 * M> rows;
  const int g0 = blockIdx.x * kRows, g = g0 + (int)threadIdx.x, n = min(kRows, a.n - g0);
  rows.load(a.feats + (size_t)g0 * 3 * M, n);
  __syncthreads();
  if (g < a.n) {
    const size_t i = 3 * (size_t)g;
    const float3 p = make_float3(a.xyz[i], a.xyz[i + 1], a.xyz[i + 2]);
    const float cp[3] = {a.campos[0], a.campos[1], a.campos[2]};
    const float3 s = make_float3(a.colors[i], a.colors[i + 1], a.colors[i + 2]);
    const float3 d = make_float3(a.dL_dcolors[i] * (1.0f - s.x) * s.x, a.dL_dcolors[i + 1] * (1.0f - s.y) * s.y,
                                 a.dL_dcolors[i + 2] * (1.0f - s.z) * s.z);
    float b[16];
    float3 gm;
    float* row = rows.row(threadIdx.x);
    const float3 dp = sh_backward<false>(a.degree, ShRowAny<M, COLOR_MAJOR>{row}, p, cp, d, b, gm);
    a.dL_dxyz[i] = dp.x;
    a.dL_dxyz[i + 1] = dp.y;
    a.dL_dxyz[i + 2] = dp.z;
#pragma unroll
    for (int k = 0; k < M; ++k) {  // the lane's row becomes its gradient
      row[ShRowAny<M, COLOR_MAJOR>::at(3 * k)] = b[k] * gm.x;
      row[ShRowAny<M, COLOR_MAJOR>::at(3 * k + 1)] = b[k] * gm.y;
      row[ShRowAny<M, COLOR_MAJOR>::at(3 * k + 2)] = b[k] * gm.z;
    }
  }
  __syncthreads();
  rows.store(a.dL_dfeats + (size_t)g0 * 3 * M, n);
}

template <int M>
static void launch_sh_sigmoid_m(const ShSigmoidArgs& a, bool color_major, bool backward, hipStream_t s) {
  const dim3 grid((a.n + kRows - 1) / kRows), block(kRows);
  if (backward && color_major)
    hipLaunchKernelGGL((sh_sigmoid_bwd_kernel<M, true>), grid, block, 0, s, a);
  else if (backward)
    hipLaunchKernelGGL((sh_sigmoid_bwd_kernel<M, false>), grid, block, 0, s, a);
  else if (color_major)
    hipLaunchKernelGGL((sh_sigmoid_fwd_kernel<M, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((sh_sigmoid_fwd_kernel<M, false>), grid, block, 0, s, a);
}

void launch_sh_sigmoid(const ShSigmoidArgs& a, int coeffs, bool color_major, bool backward, hipStream_t s) {
  switch (coeffs) {
    case 1: launch_sh_sigmoid_m<1>(a, color_major, backward, s); break;
    case 4: launch_sh_sigmoid_m<4>(a, color_major, backward, s); break;
    case 9: launch_sh_sigmoid_m<9>(a, color_major, backward, s); break;
    default: launch_sh_sigmoid_m<16>(a, color_major, backward, s); break;
  }
}

void launch_view_preprocess(const ViewArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(view_setup_kernel, dim3(1), dim3(64), 0, s, a);
  const dim3 grid((a.P + kRows - 1) / kRows), block(kRows);
  if (!a.shs_rest) {
    hipLaunchKernelGGL(view_preprocess_kernel<-1>, grid, block, 0, s, a);
    return;
  }
  switch (a.sh_coeffs) {
    case 4: hipLaunchKernelGGL(view_preprocess_kernel<9>, grid, block, 0, s, a); break;
    case 9: hipLaunchKernelGGL(view_preprocess_kernel<24>, grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL(view_preprocess_kernel<45>, grid, block, 0, s, a); break;
  }
}

void launch_view_counts(const uint32_t* cells, const uint32_t* tile_sums, uint32_t* counts, hipStream_t s) {
  hipLaunchKernelGGL(view_counts_kernel, dim3(1), dim3(64), 0, s, cells, tile_sums, counts);
}

void launch_view_geometry_bwd(const ViewArgs& a, hipStream_t s) {
  const dim3 grid((a.P + kRows - 1) / kRows), block(kRows);
  if (!a.shs) {
    hipLaunchKernelGGL((view_geometry_bwd_kernel<0, false>), grid, block, 0, s, a);
  } else if (a.shs_rest) {
    switch (a.sh_coeffs) {
      case 4: hipLaunchKernelGGL((view_geometry_bwd_kernel<4, true>), grid, block, 0, s, a); break;
      case 9: hipLaunchKernelGGL((view_geometry_bwd_kernel<9, true>), grid, block, 0, s, a); break;
      default: hipLaunchKernelGGL((view_geometry_bwd_kernel<16, true>), grid, block, 0, s, a); break;
    }
  } else {
    switch (a.sh_coeffs) {
      case 1: hipLaunchKernelGGL((view_geometry_bwd_kernel<1, false>), grid, block, 0, s, a); break;
      case 4: hipLaunchKernelGGL((view_geometry_bwd_kernel<4, false>), grid, block, 0, s, a); break;
      case 9: hipLaunchKernelGGL((view_geometry_bwd_kernel<9, false>), grid, block, 0, s, a); break;
      case 16: hipLaunchKernelGGL((view_geometry_bwd_kernel<16, false>), grid, block, 0, s, a); break;
      default: hipLaunchKernelGGL((view_geometry_bwd_kernel<-1, false>), grid, block, 0, s, a); break;
    }
  }
}

}  // namespace dmgs
