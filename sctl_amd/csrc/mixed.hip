// Mixed-precision dense Eval on gfx950: FP64 tile-centred differencing, FP32
// pairwise arithmetic, Kahan-compensated FP64 accumulation.
//
// Sources and targets are both put in Hilbert-curve order.  The sources are packed,
// TILE at a time, relative to each tile's bounding-box centre c: for every
// source the FP64 offset s - c is split into an FP32 value s' and its FP32
// residual s'' (s - c = s' + s'' to about 2^-48 relative), and the tile keeps
// H^2 = max |s'|^2.  A target (held in FP64) forms t - c once per tile the same
// way, t' + t''.
//
// Per (wave, tile or 64-source sub-tile) one of three forms runs:
//   far  -- pairs so far apart for the tile's size that the expanded r^2 =
//           |t'|^2 + |s'|^2 - 2 t'.s' is accurate to a few ulp; formed on the
//           matrix cores (k_eval_mixed_mfma; the kernels and sizes of
//           far_mfma_at).
//   mid  -- every pair has r >= H: dx = t' - s'.
//   near -- positions are differenced from both halves, dx = (t' - s') +
//           (t'' - s''), which is accurate to about 2^-23 relative to dx
//           however small r is.  A pair with r^2 == 0 makes the tile's sum
//           non-finite, and the tile is redone with r^2 == 0 masked as in the
//           reference (kernel_functions.hpp:45): the mask on every near pair
//           took 3 % of a 20 000 x 20 000 cube's apply (115.7 -> 112.4 us).
// Targets in Hilbert order keep a wave's targets together, so only tiles next
// to the wave take the near loop.  The pairs of every 64 sources are summed
// in FP32 and added into an FP64 sum of the tile, so that a tile's largest
// term does not take up the rounding of 255 FP32 additions (this halved the
// headline's error against FP64, 5.4e-7 -> 2.7e-7, at no cost in time).  A
// tile whose sum is not finite is redone by the masked near loop.  Each tile's
// sum is added into the FP64 per-target sum with Kahan compensation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "internal.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace sctl_amd {

namespace {

constexpr int WG = 256;
constexpr int TILE = 256;
constexpr float PADF = 1e18f;

// Record layout (floats) per source; far-path words first.
//   LAP_FXU  [s'x s'y s'z S | q s''x s''y s''z]                         S = |s'|^2
//   LAP_DXU  [s'x s'y s'z S | nq_x nq_y nq_z -s'.nq | s''x s''y s''z 0]   nq = q n
//   others   [s'x s'y s'z | f_0 .. f_{K0-1} | n (if any) | s''x s''y s''z], padded
//            to whole float4s, e.g.
//   STK_FXU  [s'x s'y s'z f0 | f1 f2 s''x s''y | s''z 0 0 0]
//   STK_DXU  [s'x s'y s'z f0 | f1 f2 n_x n_y | n_z s''x s''y s''z]
// FOFF / NOFF / LO: word offsets of the densities, the normal and s''.
template <int KER> struct MixLayout {
  static constexpr int FOFF = 3, NOFF = 3 + Ker<KER>::K0, LO = NOFF + Ker<KER>::ND, Q = (LO + 3 + 3) / 4;
};
template <> struct MixLayout<LAP_FXU> { static constexpr int Q = 2, LO = 5; };
template <> struct MixLayout<LAP_DXU> { static constexpr int Q = 3, LO = 8; };

template <int KER>
__device__ __forceinline__ void fill_record(float* r, const double* d, const double* n, const double* f) {
  float hi[3], lo[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    hi[k] = (float)d[k];
    lo[k] = (float)(d[k] - (double)hi[k]);
  }
  const double S = (double)hi[0] * hi[0] + (double)hi[1] * hi[1] + (double)hi[2] * hi[2];
  constexpr int LO = MixLayout<KER>::LO;
  r[0] = hi[0];
  r[1] = hi[1];
  r[2] = hi[2];
  if constexpr (KER == LAP_FXU) {
    r[3] = (float)S;
    r[4] = (float)f[0];
  } else if constexpr (KER == LAP_DXU) {
    const float nq[3] = {(float)(n[0] * f[0]), (float)(n[1] * f[0]), (float)(n[2] * f[0])};
    r[3] = (float)S;
    r[4] = nq[0];
    r[5] = nq[1];
    r[6] = nq[2];
    r[7] = (float)(-((double)hi[0] * nq[0] + (double)hi[1] * nq[1] + (double)hi[2] * nq[2]));
    r[11] = 0.0f;
  } else {
    using L = MixLayout<KER>;
#pragma unroll
    for (int k = 0; k < Ker<KER>::K0; k++) r[L::FOFF + k] = (float)f[k];
#pragma unroll
    for (int k = 0; k < Ker<KER>::ND; k++) r[L::NOFF + k] = (float)n[k];
  }
  r[LO + 0] = lo[0];
  r[LO + 1] = lo[1];
  r[LO + 2] = lo[2];
}

// Mid-range pair (r >= H): one-part FP32 differences, accurate to a few ulp of
// r there, and no mask.  th: t'; r: the record.
template <int KER, int NEWTON>
__device__ __forceinline__ void mix_mid(float* p, const float* th, const float* r, float mu) {
  const float dx = th[0] - r[0], dy = th[1] - r[1], dz = th[2] - r[2];
  if constexpr (KER == LAP_FXU) {
    const float f[1] = {r[4]};
    interact<LAP_FXU, NEWTON, false>(p, dx, dy, dz, f, f);
  } else if constexpr (KER == LAP_DXU) {
    const float one[1] = {1.0f}, nq[3] = {r[4], r[5], r[6]};
    interact<LAP_DXU, NEWTON, false>(p, dx, dy, dz, nq, one);
  } else {
    using L = MixLayout<KER>;
    interact<KER, NEWTON, false>(p, dx, dy, dz, r + L::NOFF, r + L::FOFF, mu);
  }
}

// Near-field interaction: two-part differencing.  MASK: r^2 == 0 contributes 0;
// without it such a pair makes the sum non-finite, and its tile is redone.
template <int KER, int NEWTON, bool MASK>
__device__ __forceinline__ void mix_near(float* p, const float* th, const float* tl, const float* r, float mu) {
  constexpr int LO = MixLayout<KER>::LO;
  const float dx = (th[0] - r[0]) + (tl[0] - r[LO + 0]);
  const float dy = (th[1] - r[1]) + (tl[1] - r[LO + 1]);
  const float dz = (th[2] - r[2]) + (tl[2] - r[LO + 2]);
  if constexpr (KER == LAP_FXU) {
    const float f[1] = {r[4]};
    interact<LAP_FXU, NEWTON, MASK>(p, dx, dy, dz, f, f);
  } else if constexpr (KER == LAP_DXU) {
    const float one[1] = {1.0f}, nq[3] = {r[4], r[5], r[6]};
    interact<LAP_DXU, NEWTON, MASK>(p, dx, dy, dz, nq, one);
  } else {
    using L = MixLayout<KER>;
    interact<KER, NEWTON, MASK>(p, dx, dy, dz, r + L::NOFF, r + L::FOFF, mu);
  }
}

// A kernel's far form on the matrix cores (k_eval_mixed_mfma).  NV: dot products
// with t' - s' beside r^2 (DxU: nq; Stokes: f, and n for the double layer).  GRAD:
// outputs along r = t' - s', summed as t'_k (sum g) - (sum g s'_k).  T64: |t'|^2 is
// formed in FP64 and rounded once, and the outputs take t' in FP64, where 1/r^3 or
// 1/r^5 would carry errors that are one for all of a tile's pairs into the sum (it
// costs the single layers 0.2-0.4 %, which are exact enough without).  NROW: FP32 words per
// source that the pairs read besides (s' where GRAD, then the densities).
template <int KER> struct FarForm {
  static constexpr bool ON = false;
  static constexpr int NV = 0, NROW = 0;
  static constexpr bool GRAD = false, T64 = false;
};
template <> struct FarForm<LAP_FXU> {
  static constexpr bool ON = true;
  static constexpr int NV = 0, NROW = 1;
  static constexpr bool GRAD = false, T64 = false;
};
template <> struct FarForm<LAP_DXU> {
  static constexpr bool ON = true;
  static constexpr int NV = 1, NROW = 0;
  static constexpr bool GRAD = false, T64 = true;
};
template <> struct FarForm<LAP_FXDU> {
  static constexpr bool ON = true;
  static constexpr int NV = 0, NROW = 4;
  static constexpr bool GRAD = true, T64 = true;
};
template <> struct FarForm<STK_FXU> {
  static constexpr bool ON = true;
  static constexpr int NV = 1, NROW = 6;
  static constexpr bool GRAD = true, T64 = false;
};
template <> struct FarForm<STK_DXU> {
  static constexpr bool ON = true;
  static constexpr int NV = 2, NROW = 3;
  static constexpr bool GRAD = true, T64 = true;
};

// The fourth word of a tile's meta: H^2, and in the eight bits far below its
// rounding to FP32 the exponent of the least |t'|^2 of the matrix cores
// (mfma_min_t).  (In a word of its own, H^2 stays in a scalar register, which
// costs the Stokes kernels 8 to 12 bytes of scratch.)
__device__ __forceinline__ double meta_word(double h2, float min_t) {
  return __hiloint2double(__double2hiint(h2), (__double2loint(h2) & ~0xff) | (__float_as_int(min_t) >> 23));
}
__device__ __forceinline__ float meta_min_t(double w) { return __int_as_float((__double2loint(w) & 0xff) << 23); }
// Below the |t'|^2 returned, up to its power of two, a tile's pairs take the FP32
// forms.  The matrix cores
// may flush parts and products below 2^-126.  |t'|^2 is cut to parts of 2^-16 of
// it, and v = f, n (or f n), `largest` the tile's largest, is multiplied with t' in
// products down to 2^-24 |v| |t'|.  (Stokes FxU densities of 1e-35, 70000 x 30000
// points: error 2.0e-6 on the matrix cores, 1.5e-7 so.)
__device__ __forceinline__ float mfma_min_t(float largest) {
  const float t = 0x1p-102f / largest;
  return largest > 0.0f ? fmaxf(t * t, 0x1p-100f) : 0x1p-100f;
}

// One workgroup per tile: tile centre and H^2, then the records, sources in
// the order perm[].  meta[tile] = {c_x, c_y, c_z, meta_word}; sub[4 tile + q] =
// {b_x, b_y, b_z, h^2} of sub-tile q (sources 64q .. 64q + 63, one wave):
// the centre of its FP32 offsets' bounding box, relative to the tile centre,
// and the squared radius of its offsets about that centre ({0, 0, 0, 0} for
// a sub-tile of padding only).
template <int KER>
__global__ void __launch_bounds__(WG)
k_pack_tiles(const double* __restrict__ xs, const double* __restrict__ xn, const double* __restrict__ fs, int64_t ns,
             const uint32_t* __restrict__ perm, float4* __restrict__ packed, double4* __restrict__ meta,
             float4* __restrict__ sub, int64_t ntiles, const double* __restrict__ xt, int64_t nt,
             const uint32_t* __restrict__ tperm, double* __restrict__ xt_sorted) {
  using K = Ker<KER>;
  constexpr int K0 = K::K0, ND = K::ND, Q = MixLayout<KER>::Q;
  static_assert(TILE == WG, "one source per lane");
  __shared__ double red[WG / 64][6];
  __shared__ float hred[WG / 64], vred[WG / 64][2];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if ((int64_t)blockIdx.x >= ntiles) {  // the workgroups after the tiles copy the targets into their order
    const int64_t q = ((int64_t)blockIdx.x - ntiles) * WG + tid;
    if (q < nt) {
      const int64_t t = tperm[q];
#pragma unroll
      for (int k = 0; k < 3; k++) xt_sorted[q * 3 + k] = xt[t * 3 + k];
    }
    return;
  }
  const int64_t s = (int64_t)blockIdx.x * TILE + tid;
  const bool ok = s < ns;
  const int64_t src = ok ? (int64_t)perm[s] : 0;
  // every read of the source issued at once
  double p[3] = {0, 0, 0}, n[3] = {0, 0, 0}, f[KMAX0] = {0, 0, 0, 0};
  if (ok) {
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = xs[src * 3 + k];
#pragma unroll
    for (int k = 0; k < ND; k++) n[k] = xn[src * 3 + k];
#pragma unroll
    for (int k = 0; k < K0; k++) f[k] = fs[src * K0 + k];
  }
  // tile bounding box: per wave by exchanges, then over the four waves
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double lo = wave_min(ok ? p[k] : INFINITY), hi = wave_max(ok ? p[k] : -INFINITY);
    if (lane == 0) {
      red[wv][k] = lo;
      red[wv][3 + k] = hi;
    }
  }
  __syncthreads();
  double bb[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    bb[k] = red[0][k];
#pragma unroll
    for (int w = 1; w < WG / 64; w++) bb[k] = k < 3 ? fmin(bb[k], red[w][k]) : fmax(bb[k], red[w][k]);
  }
  const double c[3] = {0.5 * (bb[0] + bb[3]), 0.5 * (bb[1] + bb[4]), 0.5 * (bb[2] + bb[5])};
  float rec[4 * Q];
#pragma unroll
  for (int k = 0; k < 4 * Q; k++) rec[k] = 0.0f;
  float h2 = 0.0f;
  if (ok) {
    const double d[3] = {p[0] - c[0], p[1] - c[1], p[2] - c[2]};
    fill_record<KER>(rec, d, n, f);
    h2 = rec[0] * rec[0] + rec[1] * rec[1] + rec[2] * rec[2];
  } else {
    rec[0] = rec[1] = rec[2] = PADF;
    if constexpr (KER == LAP_FXU || KER == LAP_DXU) rec[3] = 3.0f * PADF * PADF;
  }
  h2 = wave_max(h2);
  if (lane == 0) hred[wv] = h2;
  // the largest of the vectors that the matrix cores take, as packed
  constexpr int NV = FarForm<KER>::NV;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const float* x = rec + (KER == LAP_DXU ? 4 : 3 + 3 * v);
    const float m = wave_max(fmaxf(fabsf(x[0]), fmaxf(fabsf(x[1]), fabsf(x[2]))));
    if (lane == 0) vred[wv][v] = m;
  }
  __syncthreads();
  if (tid == 0) {
    float hm = hred[0];
#pragma unroll
    for (int w = 1; w < WG / 64; w++) hm = fmaxf(hm, hred[w]);
    float min_t = mfma_min_t(1.0f);
#pragma unroll
    for (int v = 0; v < NV; v++)
      min_t = fmaxf(min_t, mfma_min_t(fmaxf(fmaxf(vred[0][v], vred[1][v]), fmaxf(vred[2][v], vred[3][v]))));
    meta[blockIdx.x] = make_double4(c[0], c[1], c[2], meta_word((double)hm * 1.0000001, min_t));
  }
  {
    float b[3], bh2 = 0.0f;
    const bool any = __builtin_amdgcn_ballot_w64(ok) != 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float lo = wave_min(ok ? rec[k] : INFINITY), hi = wave_max(ok ? rec[k] : -INFINITY);
      b[k] = any ? 0.5f * (lo + hi) : 0.0f;
    }
    if (ok) {
      const float dx = rec[0] - b[0], dy = rec[1] - b[1], dz = rec[2] - b[2];
      bh2 = dx * dx + dy * dy + dz * dz;
    }
    bh2 = wave_max(bh2);
    if ((tid & 63) == 0) sub[(int64_t)blockIdx.x * (WG / 64) + (tid >> 6)] = make_float4(b[0], b[1], b[2], bh2 * 1.0001f);
  }
  float4* dst = packed + ((int64_t)blockIdx.x * TILE + tid) * Q;
#pragma unroll
  for (int q = 0; q < Q; q++) dst[q] = make_float4(rec[4 * q], rec[4 * q + 1], rec[4 * q + 2], rec[4 * q + 3]);
}

// Waves per SIMD that the register allocation must leave room for: the
// Helmholtz gradient kernels (6 outputs per target) need 140-143 VGPRs at one
// target per lane, which allows 3 waves; holding them to 128 allows 4.
template <int KER, int TPL> constexpr int mixed_min_waves() {
  return (KER == HLM_FXDU || KER == HLMD_FXDU) && TPL == 1 ? 4 : 1;
}

template <int KER, int TPL, int NEWTON>
__global__ void __launch_bounds__(WG, (mixed_min_waves<KER, TPL>()))
k_eval_mixed(const double* __restrict__ xt, int64_t nt, const uint32_t* __restrict__ tperm,
             const float4* __restrict__ packed, const double4* __restrict__ meta, const float4* __restrict__ sub,
             int64_t ntiles, int64_t tiles_per_split, double* __restrict__ out, int direct, double scale, double ctx) {
  using K = Ker<KER>;
  constexpr int K1 = K::K1, Q = MixLayout<KER>::Q, R = 4 * Q;
  __shared__ float4 lds[TILE * Q];
  const float mu = (float)ctx;

  const int tid = threadIdx.x;
  const SplitCoord wg = split_coord((nt + WG * TPL - 1) / (WG * TPL));
  const int64_t tile_begin = wg.split * tiles_per_split;
  const int64_t tile_end = tile_begin + tiles_per_split < ntiles ? tile_begin + tiles_per_split : ntiles;
  const int64_t q0 = wg.block * (WG * TPL) + tid;

  double t64[TPL][3], acc[TPL][K1], comp[TPL][K1];
#pragma unroll
  for (int j = 0; j < TPL; j++) {
    const int64_t q = q0 + (int64_t)j * WG;
    const bool ok = q < nt;
#pragma unroll
    for (int k = 0; k < 3; k++) t64[j][k] = ok ? xt[q * 3 + k] : 0.0;  // xt in the order tperm
#pragma unroll
    for (int k = 0; k < K1; k++) acc[j][k] = comp[j][k] = 0.0;
  }

  for (int64_t tile = tile_begin; tile < tile_end; tile++) {
    __syncthreads();
    const float4* src = packed + tile * (TILE * Q);
#pragma unroll
    for (int q = 0; q < Q; q++) lds[q * WG + tid] = src[q * WG + tid];
    const double4 m = meta[tile];
    __syncthreads();

    // A wave whose targets are all |t'| >= 2H from the tile centre (so r >= H)
    // takes the mid form over the whole tile.  Otherwise each 64-source sub-tile
    // q (centre b_q, radius h_q about it) is classified on its own, with X =
    // |t'| + H the scale of the rounding of t' and s' and r >= |t' - b_q| - h_q:
    // mid (relative error <= 3 eps) where that bound is >= X/3, else near
    // (two-part differences, masked).  A non-finite partial redoes the tile in
    // the near form.
    const float mid_r2 = 4.0f * (float)m.w;
    // p: FP32 sums of at most 64 pairs, added into the FP64 tile sums pt
    // after every 64 sources (sub64), so that a tile's dominant term does
    // not absorb the rounding of 255 FP32 additions.
    float th[TPL][3], T[TPL], p[TPL][K1];
    double pt[TPL][K1];
    bool notmid = false;
#pragma unroll
    for (int j = 0; j < TPL; j++) {
      th[j][0] = (float)(t64[j][0] - m.x);
      th[j][1] = (float)(t64[j][1] - m.y);
      th[j][2] = (float)(t64[j][2] - m.z);
      T[j] = fmad(th[j][2], th[j][2], fmad(th[j][1], th[j][1], th[j][0] * th[j][0]));
      notmid |= T[j] < mid_r2;
#pragma unroll
      for (int k = 0; k < K1; k++) {
        p[j][k] = 0.0f;
        pt[j][k] = 0.0;
      }
    }
    auto sub64 = [&]() {
#pragma unroll
      for (int j = 0; j < TPL; j++)
#pragma unroll
        for (int k = 0; k < K1; k++) {
          pt[j][k] += (double)p[j][k];
          p[j][k] = 0.0f;
        }
    };
    const float* recs = reinterpret_cast<const float*>(lds);
    bool use_near = false;
    // At more than one target per lane a wave's targets span more space and
    // the sub-tile classes would raise the kernel's registers (two targets
    // per lane: 70 -> 93 VGPRs); such shapes classify whole tiles only.
    constexpr bool SUBTILES = TPL == 1;
    const bool tile_mid = __builtin_amdgcn_ballot_w64(notmid) == 0;
    use_near = !SUBTILES && !tile_mid;
    if (use_near) {
      // the near loop below
    } else if (tile_mid) {
      for (int i0 = 0; i0 < TILE; i0 += 64) {
#pragma unroll 4
        for (int i = i0; i < i0 + 64; i++) {
          const float* rec = recs + i * R;
#pragma unroll
          for (int j = 0; j < TPL; j++) mix_mid<KER, NEWTON>(p[j], th[j], rec, mu);
        }
        sub64();
      }
    } else if constexpr (SUBTILES) {
      const float H = sqrtf((float)m.w);
#pragma unroll 1
      for (int q = 0; q < WG / 64; q++) {
        const float4 b = sub[tile * (WG / 64) + q];
        const float h = sqrtf(b.w);
        bool qnear = false;
#pragma unroll
        for (int j = 0; j < TPL; j++) {
          const float X = sqrtf(T[j]) + H;
          const float dx = th[j][0] - b.x, dy = th[j][1] - b.y, dz = th[j][2] - b.z;
          const float d2 = fmad(dz, dz, fmad(dy, dy, dx * dx));
          const float em = fmad(1.0f / 3.0f, X, h);
          qnear |= d2 < em * em;
        }
        const float* qrec = recs + q * 64 * R;
        if (__builtin_amdgcn_ballot_w64(qnear) != 0) {
          float tl[TPL][3];
#pragma unroll
          for (int j = 0; j < TPL; j++) {
            tl[j][0] = (float)((t64[j][0] - m.x) - (double)th[j][0]);
            tl[j][1] = (float)((t64[j][1] - m.y) - (double)th[j][1]);
            tl[j][2] = (float)((t64[j][2] - m.z) - (double)th[j][2]);
          }
#pragma unroll 2
          for (int i = 0; i < 64; i++) {
#pragma unroll
            for (int j = 0; j < TPL; j++) mix_near<KER, NEWTON, false>(p[j], th[j], tl[j], qrec + i * R, mu);
          }
        } else {
#pragma unroll 4
          for (int i = 0; i < 64; i++) {
#pragma unroll
            for (int j = 0; j < TPL; j++) mix_mid<KER, NEWTON>(p[j], th[j], qrec + i * R, mu);
          }
        }
        sub64();
      }
    }
    if (!use_near) {
      bool bad = false;
#pragma unroll
      for (int j = 0; j < TPL; j++)
#pragma unroll
        for (int k = 0; k < K1; k++) bad |= !__builtin_isfinite(pt[j][k]);
      use_near = __builtin_amdgcn_ballot_w64(bad) != 0;
    }
    if (use_near) {
      float tl[TPL][3];
#pragma unroll
      for (int j = 0; j < TPL; j++) {
        tl[j][0] = (float)((t64[j][0] - m.x) - (double)th[j][0]);
        tl[j][1] = (float)((t64[j][1] - m.y) - (double)th[j][1]);
        tl[j][2] = (float)((t64[j][2] - m.z) - (double)th[j][2]);
#pragma unroll
        for (int k = 0; k < K1; k++) {
          p[j][k] = 0.0f;
          pt[j][k] = 0.0;
        }
      }
      for (int i0 = 0; i0 < TILE; i0 += 64) {
#pragma unroll 2
        for (int i = i0; i < i0 + 64; i++) {
          const float* rec = recs + i * R;
#pragma unroll
          for (int j = 0; j < TPL; j++) mix_near<KER, NEWTON, true>(p[j], th[j], tl[j], rec, mu);
        }
        sub64();
      }
    }
#pragma unroll
    for (int j = 0; j < TPL; j++)
#pragma unroll
      for (int k = 0; k < K1; k++) {  // Kahan: acc += pt
        const double y = pt[j][k] - comp[j][k];
        const double s = acc[j][k] + y;
        comp[j][k] = (s - acc[j][k]) - y;
        acc[j][k] = s;
      }
  }

#pragma unroll
  for (int j = 0; j < TPL; j++) {
    const int64_t q = q0 + (int64_t)j * WG;
    if (q < nt) {
      // the target's own index is read only here, so it holds no register
      // through the tile loop
      const int64_t t = direct ? (int64_t)tperm[q] : 0;
#pragma unroll
      for (int k = 0; k < K1; k++) {
        const double v = acc[j][k] - comp[j][k];
        if (direct) out[t * K1 + k] += v * scale;
        else out[wg.split * nt * K1 + q * K1 + k] = v;
      }
    }
  }
}

// ---- The far form on the matrix cores --------------------------------------
// The far form's r^2 = |t'|^2 + |s'|^2 - 2 t'.s' (and the double layer's
// f n.r = t'.nq - s'.nq, Stokes' f.r and n.r) is a contraction over the three
// axes.  FP32 values are
// cut into three bf16 parts (8 of the 24 mantissa bits each, by truncation, so
// the parts' sum is exact), and a product of two such values is the sum of
// eight products of parts (all but the last parts' product, 2^-32 of it): the
// 8 k-slots that one lane group holds of v_mfma_f32_16x16x32_bf16.  Lane groups
// 0-2 take the axes; group 3 takes |t'|^2 (three parts against ones), and
// |s'|^2 comes in as the FP32 addend, one per row.  So one instruction forms
// r^2 for 16 sources x 16 targets in FP32 accumulation: rms error 6.5e-8
// relative where the FP32 FMA chain has 6.9e-8 (|t'| = 3H, 10^6 pairs).
//
// Cycles per 256 pairs of one SIMD on MI355X (8 waves, 2.4 GHz): 17 for the
// instruction, 33 for four v_rsq_f32, 12 for four FMAs, 55 together; the
// FP32 form needs 94.  Dense plan applies, 524288 x 524288 sphere and shell
// (FP32 form -> this): Laplace FxU 46.5 -> 29.2 ms (9.4e12 pairs/s), DxU 70.7
// -> 45.6 ms; 131072 x 131072 cube 3.36 -> 2.60 and 5.04 -> 3.84 ms.
//
// The matrix cores round sums toward minus infinity somewhere below 2^-29 of
// their largest term: a bias of one sign, which 130 001 double layer terms of
// random sign do not average out (error against 64 bits 2.0e-7 -> 6.8e-7).
// The odd sources' nq and s'.nq are therefore staged with the opposite sign
// and turned back by the FMA, so that the bias cancels between neighbours
// (2.0e-7 again).  r^2's bias is multiplied by the density, whose sign varies.
//
// D's layout (lane l: target column l & 15, source rows 4 (l >> 4) + i) leaves
// each lane with 4 sources of one target, whose densities and |s'|^2 are one
// 16-byte LDS read each, shared by the wave's four target groups.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

template <int KER> constexpr bool far_mfma() { return FarForm<KER>::ON; }

struct Parts {
  float a, b, c;  // each used by its upper 16 bits
};
__device__ __forceinline__ float upper(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }
__device__ __forceinline__ Parts parts3(float x) {
  const float r = x - upper(x);
  return {x, r, r - upper(r)};
}
// The upper halves of two words: lo's in bits 0-15, hi's in bits 16-31.
__device__ __forceinline__ uint32_t halves(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
// k-slots of a row (source) and of a column (target): slot by slot the eight products.
__device__ __forceinline__ u32x4 row_slots(float x) {
  const Parts p = parts3(x);
  return u32x4{halves(p.a, p.a), halves(p.a, p.b), halves(p.b, p.b), halves(p.c, p.c)};
}
__device__ __forceinline__ u32x4 column_slots(float x) {
  const Parts p = parts3(x);
  const uint32_t ab = halves(p.a, p.b);
  return u32x4{ab, halves(p.c, p.a), halves(p.b, p.c), ab};
}
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a and b hold a value per row of 16 lanes.  swap32: a's rows 2, 3 against b's
// rows 0, 1; swap16: a's rows 1, 3 against b's rows 0, 2.
__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(double& a, double& b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  a = __hiloint2double(hi[0], lo[0]);
  b = __hiloint2double(hi[1], lo[1]);
}
// v[j] of row g -> v[g] of row j.
__device__ __forceinline__ void transpose4(float* v) {
  swap32(v[0], v[2]);
  swap32(v[1], v[3]);
  swap16(v[0], v[1]);
  swap16(v[2], v[3]);
}
// In row j, the FP64 sum of v[j] over the four rows.
__device__ __forceinline__ double sum_rows(float a, float b, float c, float d) {
  swap32(a, c);
  swap32(b, d);
  double x = (double)a + (double)c, y = (double)b + (double)d;
  swap16(x, y);
  return x + y;
}

// One far pair: D = r^2, d = the NV dot products, row(k) = word k of the source.
template <int KER, int NEWTON, class Row>
__device__ __forceinline__ void far_pair(float* p, float& G, float r2, const float* d, Row&& row) {
  float z = rsq_deferred<NEWTON>(r2);
  if constexpr (Ker<KER>::POW == 0 && NEWTON > 0) z *= (float)newton_c2(NEWTON);
  if constexpr (KER == LAP_FXU) {
    p[0] = fmad(z, row(0), p[0]);
  } else if constexpr (KER == LAP_DXU) {
    p[0] = fmad(d[0] * z, z * z, p[0]);
  } else if constexpr (KER == STK_FXU) {  // z (f + w r), w = (f.r) z^2
    const float w = d[0] * (z * z);
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = fmad(z, fmad(-w, row(k), row(3 + k)), p[k]);
    G = fmad(w, z, G);
  } else {  // g r
    const float z2 = z * z;
    const float g = KER == LAP_FXDU ? row(3) * z * z2 : (d[0] * z2) * (d[1] * z2) * z;
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = fmad(-g, row(k), p[k]);
    G = g;
  }
}

// Mixed Eval with the far form above, 64 targets per wave.  Each tile's sources
// are staged as k-slots; the classes are those of k_eval_mixed at one target
// per lane (whole tile, else 64-source sub-tiles).  Far pairs are summed in the
// matrix layout (at most 64 per FP32 sum), mid and near ones with one target
// per lane from records that the wave stages for itself, NEAR_ST at a time.
//
// A tile's far sums go to the lane of their target (sum_rows), and the targets'
// columns come from those lanes (transpose4), both by row swaps: a lane holds
// one compensated sum per output of its own target.  With a sum per target
// group and output, and the four groups' coordinates in FP64, the single layer
// took 119 registers, not 95 (20000^2 cube 112.4 -> 108.1 us, 50000^2 445 ->
// 424), and Stokes 20 words of scratch more (DxU 131072 x 150001 6993 -> 6671
// us, FxU 6590 -> 6449).
//
// Waves per SIMD asked for: left alone the compiler took 148 registers for the
// Laplace double layer (three waves), 58.6 instead of 45.6 ms at 524288 x
// 524288; at six waves the single layer is no faster (28.6 and 28.3 ms).  Three
// outputs run three waves (128 registers spill: Stokes FxU 131072 x 150001 6.9
// against 6.4 ms), and no more are offered: else the scheduler saves registers
// by using each product right after its instruction (Laplace FxdU 524288 x
// 524288 65.2 against 59.8 ms).
template <int KER> constexpr int mfma_waves() { return Ker<KER>::K1 == 1 ? 4 : 3; }
// Chunks and sources unrolled, from sweeps of 1, 2 and 4 resp. 2, 4 and 8.
template <int KER> constexpr int far_unroll() { return Ker<KER>::K1 == 1 ? 4 : (KER == STK_FXU ? 2 : 1); }
template <int KER> constexpr int lane_unroll() { return KER == LAP_FXU || KER == LAP_FXDU ? 4 : 2; }
template <int KER, int NEWTON>
__global__ void __launch_bounds__(WG)
__attribute__((amdgpu_waves_per_eu((mfma_waves<KER>()), (Ker<KER>::K1 == 1 ? 8 : 3))))
k_eval_mixed_mfma(const double* __restrict__ xt, int64_t nt, const uint32_t* __restrict__ tperm,
                  const float4* __restrict__ packed, const double4* __restrict__ meta, const float4* __restrict__ sub,
                  int64_t ntiles, int64_t tiles_per_split, double* __restrict__ out, int direct, double scale,
                  double) {
  using F = FarForm<KER>;
  using L = MixLayout<KER>;
  constexpr int K1 = Ker<KER>::K1, Q = L::Q, R = 4 * Q, NEAR_ST = 32, GROUPS = 4, CHUNKS = TILE / 16;
  constexpr int NV = F::NV, NROW = F::NROW;
  constexpr bool LAP = KER == LAP_FXU || KER == LAP_DXU;
  // k-slots, 16 rows x 3 axes per chunk; the last entry is all of group 3's:
  // ones against |t'|^2 in rs, zeros in rv.
  constexpr int SLOTS = TILE * 3;
  __shared__ u32x4 rs[SLOTS + 1];                    // -2 s'
  __shared__ u32x4 rv[NV ? NV : 1][NV ? SLOTS + 1 : 1];  // the NV vectors v
  __shared__ float sS[TILE];                        // |s'|^2
  __shared__ float sv[NV ? NV : 1][NV ? TILE : 1];  // -s'.v
  __shared__ float srow[NROW ? NROW : 1][NROW ? TILE : 1];
  __shared__ float4 near_all[(WG / 64) * NEAR_ST * Q];

  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4;
  float4* nst = near_all + (tid >> 6) * (NEAR_ST * Q);
  const SplitCoord wg = split_coord((nt + WG - 1) / WG);
  const int64_t tile_begin = wg.split * tiles_per_split;
  const int64_t tile_end = tile_begin + tiles_per_split < ntiles ? tile_begin + tiles_per_split : ntiles;
  const int64_t q0 = wg.block * WG + (tid & ~63);  // the wave's first target

  double t64[3], acc[K1], comp[K1];  // of this lane's target, q0 + lane
#pragma unroll
  for (int k = 0; k < 3; k++) t64[k] = q0 + lane < nt ? xt[(q0 + lane) * 3 + k] : 0.0;
#pragma unroll
  for (int k = 0; k < K1; k++) acc[k] = comp[k] = 0.0;
  const int slot = (tid >> 4) * 48 + (tid & 15);  // this thread's row, written per tile
  const int my_slot = g < 3 ? lane : SLOTS, my_step = g < 3 ? 48 : 0;  // read: this lane's in chunk 0, and per chunk
  if (tid == 0) {
    rs[SLOTS] = u32x4{0x3f803f80u, 0x00003f80u, 0u, 0u};
#pragma unroll
    for (int v = 0; v < NV; v++) rv[v][SLOTS] = u32x4{0u, 0u, 0u, 0u};
  }

  for (int64_t tile = tile_begin; tile < tile_end; tile++) {
    const float4* src = packed + tile * (TILE * Q);
    float rec[R];
#pragma unroll
    for (int q = 0; q <= (L::LO - 1) / 4; q++) {  // the residuals only where they share a word with the rest
      const float4 v = src[tid * Q + q];
      rec[4 * q] = v.x;
      rec[4 * q + 1] = v.y;
      rec[4 * q + 2] = v.z;
      rec[4 * q + 3] = v.w;
    }
    const double4 m = meta[tile];
    __syncthreads();  // the previous tile's readers
#pragma unroll
    for (int k = 0; k < 3; k++) rs[slot + 16 * k] = row_slots(-2.0f * rec[k]);
    if constexpr (LAP) sS[tid] = rec[3];
    else sS[tid] = (float)((double)rec[0] * rec[0] + (double)rec[1] * rec[1] + (double)rec[2] * rec[2]);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const float* x = rec + (KER == LAP_DXU ? 4 : 3 + 3 * v);
      const float c = KER == LAP_DXU
                          ? rec[7]
                          : (float)-((double)rec[0] * x[0] + (double)rec[1] * x[1] + (double)rec[2] * x[2]);
#pragma unroll
      for (int k = 0; k < 3; k++) rv[v][slot + 16 * k] = row_slots(tid & 1 ? -x[k] : x[k]);
      sv[v][tid] = tid & 1 ? -c : c;
    }
    if constexpr (KER == LAP_FXU) {
      srow[0][tid] = rec[4];
    } else {
#pragma unroll
      for (int k = 0; k < NROW; k++) srow[k][tid] = rec[k];  // s', then the densities from FOFF = 3
    }
    __syncthreads();

    const double t[3] = {t64[0] - m.x, t64[1] - m.y, t64[2] - m.z};
    const float th[3] = {(float)t[0], (float)t[1], (float)t[2]};
    const float T = F::T64 ? (float)fmad(t[2], t[2], fmad(t[1], t[1], t[0] * t[0]))
                           : fmad(th[2], th[2], fmad(th[1], th[1], th[0] * th[0]));
    const float H2 = (float)m.w;
    u32x4 col[GROUPS];  // lane group g: axis g (3: |t'|^2) of the targets q0 + 16 j + (lane & 15)
    float cx[GROUPS] = {th[0], th[1], th[2], T};
    transpose4(cx);
#pragma unroll
    for (int j = 0; j < GROUPS; j++) col[j] = column_slots(cx[j]);
    float pf[GROUPS][K1], pG[GROUPS], pn[K1];
    double ptn[K1];
#pragma unroll
    for (int j = 0; j < GROUPS; j++) pG[j] = 0.0f;
#pragma unroll
    for (int k = 0; k < K1; k++) {
      pn[k] = 0.0f;
      ptn[k] = 0.0;
#pragma unroll
      for (int j = 0; j < GROUPS; j++) pf[j][k] = 0.0f;
    }
    auto far = [&](int ch0, auto count) {
#pragma unroll (far_unroll<KER>())
      for (int ch = ch0; ch < ch0 + decltype(count)::value; ch++) {
        auto four = [&](const float* a) { return *reinterpret_cast<const f32x4*>(a + ch * 16 + 4 * g); };
        const int at = my_slot + ch * my_step;
        const u32x4 a = rs[at];
        const f32x4 S4 = four(sS);
        u32x4 av[NV ? NV : 1];
        f32x4 v4[NV ? NV : 1], w4[NROW ? NROW : 1];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          av[v] = rv[v][at];
          v4[v] = four(sv[v]);
        }
#pragma unroll
        for (int k = 0; k < NROW; k++) w4[k] = four(srow[k]);
#pragma unroll
        for (int j = 0; j < GROUPS; j++) {
          const f32x4 r2 = mfma16(a, col[j], S4);
          f32x4 dots[NV ? NV : 1];
#pragma unroll
          for (int v = 0; v < NV; v++) dots[v] = mfma16(av[v], col[j], v4[v]);
          // The four g of g r are added up first: G's rounding is |t'| / H times that of
          // the sums of g s' in the outputs.  With T64 and the outputs' FP64 t': error
          // against FP64 for sets apart (FP32 form / before / now) Stokes DxU 3.6 / 4.0 /
          // 3.6e-7, Laplace FxdU 3.1 / 3.1 / 2.3e-7; sphere 2.48 / 2.52 / 2.49 and 1.83 /
          // 1.82 / 1.76e-7; the same time.
          constexpr bool BY4 = F::GRAD && KER != STK_FXU;
          float g4[4];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            float d[NV ? NV : 1];
#pragma unroll
            for (int v = 0; v < NV; v++) d[v] = i & 1 ? -dots[v][i] : dots[v][i];
            far_pair<KER, NEWTON>(pf[j], BY4 ? g4[i] : pG[j], r2[i], d, [&](int k) { return w4[k][i]; });
          }
          if constexpr (BY4) pG[j] += (g4[0] + g4[1]) + (g4[2] + g4[3]);
        }
      }
    };
    // Sub-tile sq0 / 64 with one target per lane: the mid form, or the near form.
    // (near: 0 mid, 1 near, 2 near with r^2 == 0 masked)
    auto by_lane = [&](int sq0, int near) {
      const float tl[3] = {(float)((t64[0] - m.x) - (double)th[0]), (float)((t64[1] - m.y) - (double)th[1]),
                           (float)((t64[2] - m.z) - (double)th[2])};
#pragma unroll 1
      for (int s0 = sq0; s0 < sq0 + 64; s0 += NEAR_ST) {
        wave_sync();
        for (int i = lane; i < NEAR_ST * Q; i += 64) nst[i] = src[s0 * Q + i];
        wave_sync();
        const float* recs = reinterpret_cast<const float*>(nst);
        if (near == 2) {
#pragma unroll 1
          for (int i = 0; i < NEAR_ST; i++) mix_near<KER, NEWTON, true>(pn, th, tl, recs + i * R, 0.0f);
        } else if (near) {
#pragma unroll (lane_unroll<KER>())
          for (int i = 0; i < NEAR_ST; i++) mix_near<KER, NEWTON, false>(pn, th, tl, recs + i * R, 0.0f);
        } else {
#pragma unroll (lane_unroll<KER>())
          for (int i = 0; i < NEAR_ST; i++) mix_mid<KER, NEWTON>(pn, th, recs + i * R, 0.0f);
        }
      }
#pragma unroll
      for (int k = 0; k < K1; k++) {
        ptn[k] += (double)pn[k];
        pn[k] = 0.0f;
      }
    };
    const bool tiny = __builtin_amdgcn_ballot_w64(T < meta_min_t(m.w)) != 0;
    if (__builtin_amdgcn_ballot_w64(T < 9.0f * H2) == 0 && !tiny) {
      far(0, std::integral_constant<int, CHUNKS>());
    } else {
      const float H = sqrtf(H2);
#pragma unroll 1
      for (int q = 0; q < TILE / 64; q++) {
        const float4 b = sub[tile * (TILE / 64) + q];
        const float h = sqrtf(b.w), X = sqrtf(T) + H;
        const float dx = th[0] - b.x, dy = th[1] - b.y, dz = th[2] - b.z;
        const float d2 = fmad(dz, dz, fmad(dy, dy, dx * dx));
        const float ef = fmad(0.5f, X, h), em = fmad(1.0f / 3.0f, X, h);
        if (__builtin_amdgcn_ballot_w64(d2 < ef * ef) == 0 && !tiny)
          far(q * (CHUNKS / 4), std::integral_constant<int, CHUNKS / 4>());
        else by_lane(q * 64, __builtin_amdgcn_ballot_w64(d2 < em * em) != 0 ? 1 : 0);
      }
    }
    bool bad = false;
#pragma unroll
    for (int k = 0; k < K1; k++) {
      bad |= !__builtin_isfinite(ptn[k]);
#pragma unroll
      for (int j = 0; j < GROUPS; j++) bad |= !__builtin_isfinite(pf[j][k]);
    }
    if constexpr (F::GRAD) {
#pragma unroll
      for (int j = 0; j < GROUPS; j++) bad |= !__builtin_isfinite(pG[j]);
    }
    if (__builtin_amdgcn_ballot_w64(bad) != 0) {  // the whole tile in the near form
#pragma unroll
      for (int k = 0; k < K1; k++) {
        ptn[k] = 0.0;
        pn[k] = 0.0f;
#pragma unroll
        for (int j = 0; j < GROUPS; j++) pf[j][k] = 0.0f;
      }
#pragma unroll
      for (int j = 0; j < GROUPS; j++) pG[j] = 0.0f;
      for (int q = 0; q < TILE / 64; q++) by_lane(q * 64, 2);
    }
    double Gt = 0.0;
    if constexpr (F::GRAD) Gt = sum_rows(pG[0], pG[1], pG[2], pG[3]);
#pragma unroll
    for (int k = 0; k < K1; k++) {
      ptn[k] += sum_rows(pf[0][k], pf[1][k], pf[2][k], pf[3][k]);
      if constexpr (F::GRAD) {
        if constexpr (F::T64) {
          double x = t64[k];
          asm volatile("" : "+v"(x));  // or the difference is held through the far loop
          ptn[k] = fmad(x - (k == 0 ? m.x : (k == 1 ? m.y : m.z)), Gt, ptn[k]);
        } else {
          float x = th[k];
          asm volatile("" : "+v"(x));  // or the conversion is done in each pass of the far loop
          ptn[k] = fmad((double)x, Gt, ptn[k]);
        }
      }
      const double y = ptn[k] - comp[k];  // Kahan: acc += ptn
      const double sum = acc[k] + y;
      comp[k] = (sum - acc[k]) - y;
      acc[k] = sum;
    }
  }

  const int64_t q = q0 + lane;
  if (q >= nt) return;
  const int64_t t = direct ? (int64_t)tperm[q] : 0;
#pragma unroll
  for (int k = 0; k < K1; k++) {
    const double v = acc[k] - comp[k];
    if (direct) out[t * K1 + k] += v * scale;
    else out[wg.split * nt * K1 + q * K1 + k] = v;
  }
}

// v_trg[tperm[q]*K1+k] += scale * sum_y part[y][q*K1+k]; one lane quad per
// element (sum_splits_quad).
__global__ void __launch_bounds__(WG)
k_reduce_splits_perm(const double* __restrict__ part, int64_t nt, int K1, int nsplit, const uint32_t* __restrict__ tperm,
                     double* __restrict__ out, double scale) {
  const int64_t i = ((int64_t)blockIdx.x * WG + threadIdx.x) >> 2;
  const int64_t n = nt * K1;
  const double s = sum_splits_quad(part, n, nsplit, i, i < n);
  if (i >= n || (threadIdx.x & 3) != 0) return;
  const int64_t q = i / K1, k = i - q * K1;
  out[(int64_t)tperm[q] * K1 + k] += s * scale;
}

using EvalMixFn = void (*)(const double*, int64_t, const uint32_t*, const float4*, const double4*, const float4*, int64_t,
                           int64_t, double*, int, double, double);
using PackFn = void (*)(const double*, const double*, const double*, int64_t, const uint32_t*, float4*, double4*,
                        float4*, int64_t, const double*, int64_t, const uint32_t*, double*);

constexpr int TPLS[3] = {1, 2, 4};
int tpl_index(int tpl) { return tpl >= 4 ? 2 : (tpl >= 2 ? 1 : 0); }

// ti: targets per lane (the matrix-core kernels have one form; the Laplace
// single and double layer have no other).
template <int KER, int NEWTON> EvalMixFn mix_fn(int ti, bool mfma) {
  if constexpr (far_mfma<KER>()) {
    if (mfma || KER == LAP_FXU || KER == LAP_DXU) return k_eval_mixed_mfma<KER, NEWTON>;
  }
  if constexpr (KER != LAP_FXU && KER != LAP_DXU) {
    constexpr int MT = max_tpl<KER>();
    if (ti >= 2 && MT >= 4) return k_eval_mixed<KER, (MT >= 4 ? 4 : 1), NEWTON>;
    if (ti >= 1 && MT >= 2) return k_eval_mixed<KER, (MT >= 2 ? 2 : 1), NEWTON>;
    return k_eval_mixed<KER, 1, NEWTON>;
  }
  return nullptr;  // not reached
}
EvalMixFn mix_fn(int ker, int newton, int ti, bool mfma) {
  return with_kernel(ker, [&](auto kc) -> EvalMixFn {
    constexpr int K = decltype(kc)::value;
    return newton ? mix_fn<K, 1>(ti, mfma) : mix_fn<K, 0>(ti, mfma);
  });
}
PackFn pack_fn(int ker) {
  return with_kernel(ker, [](auto kc) -> PackFn { return k_pack_tiles<decltype(kc)::value>; });
}
int layout_q(int ker) {
  return with_kernel(ker, [](auto kc) { return MixLayout<decltype(kc)::value>::Q; });
}
int max_tpl_index(int ker) {
  return with_kernel(ker, [](auto kc) { return tpl_index(max_tpl<decltype(kc)::value>()); });
}

}  // namespace

// Measured on MI355X, uniform cubes, us, FP64 kernels with the rsqrt estimate /
// mixed path:
//                    dense plan apply                     Eval
//   Laplace FxU      8000^2 34 / 39, 12000^2 59 / 62      8000^2 36 / 67, 17000^2 109 / 125
//   Laplace DxU      8000^2 44 / 59, 12000^2 83 / 92      8000^2 47 / 87, 17000^2 160 / 166
//   Stokes FxU       5000^2 30 / 35, 6500^2 44 / 43       5000^2 33 / 63, 8000^2 64 / 80
//   Helmholtz FxU    6500^2 104 / 118, 8000^2 147 / 141   8000^2 150 / 169
//   BiotSavart FxdU  2000 x 3000 22 / 39, 5000^2 53 / 50  5000^2 56 / 77
// The line is where an apply, which keeps its orders, is even, so that a plan
// and an Eval of one size run the same kernels (their results are equal bit
// for bit).  The estimate is good to 2^-24 and all else is FP64: errors are a
// tenth to a half of the mixed path's.
bool mixed_runs_f64(int ker, int64_t nt, int64_t ns) {
  int K0, K1, ND;
  kernel_dims(ker, &K0, &K1, &ND);
  const double pairs = (double)nt * (double)ns;
  if (ker == LAP_FXU || ker == LAP_DXU) return pairs <= 1.5e8;
  return pairs <= (needs_ctx(ker) ? 6e7 : (K1 > 4 ? 2e7 : 4.2e7));
}

// Whether a mixed Eval of this size takes the matrix-core kernel.  The Laplace
// single and double layer always do.  The kernels with three outputs run three
// waves per SIMD in it, which their near pairs pay for: a gain only where far
// tiles prevail.  Dense plan applies, FP32 form / matrix cores, us:
//                    20000^2 cube   50000^2 cube  90000^2 cube  131072 x 150001  262144^2
//                                                               clusters         sphere
//   Stokes FxU       195 / 203      1013 / 979    3124 / 2911   7682 / 6612      26421 / 22086
//   Stokes DxU       219 / 216      1170 / 1038   3650 / 3043   8828 / 6840      30768 / 22346
//   Laplace FxdU     151 / 157      757 / 730     2302 / 2129   5505 / 4696      19090 / 15338
// Few sources make large tiles, near to more targets: cubes of 400003 x 5000
// 906 / 1000, 1027 / 1076 and 697 / 763; x 20003 3195 / 3183, 3675 / 3392 and
// 2353 / 2348; 1500001 x 7001 4991 / 4750, 5411 / 5189 and 4090 / 3559; the
// other way round, 5000 x 400003, 843 / 789, 978 / 832 and 625 / 590.
bool far_mfma_at(int ker, int64_t nt, int64_t ns) {
  const double pairs = (double)nt * (double)ns;
  switch (ker) {
    case LAP_FXU:
    case LAP_DXU: return true;
    case STK_DXU: return pairs >= 1e10 || (ns >= 20000 && pairs >= 1e9);
    case STK_FXU:
    case LAP_FXDU: return pairs >= 1e10 || (ns >= 20000 && pairs >= 2e9);
    default: return false;
  }
}

bool mixed_runs_mfma(int ker, int64_t nt, int64_t ns) {
  return !mixed_runs_f64(ker, nt, ns) && far_mfma_at(ker, nt, ns);
}

// Launch geometry of one mixed Eval: target blocks and the source splits.
// Split the sources over gridDim.y when the target blocks cannot fill the
// device (each split one tile at the least), and so that no split exceeds
// SPLIT_TILES tiles: workgroups are dispatched in order of
// their linear index (blockIdx.x fastest), so the ones resident at a time
// share one split's records (2 MiB for Laplace FxU) in their XCD's 4 MiB L2
// instead of drifting apart over the whole source array.  The splits' partial
// sums stay within part_budget bytes (split_group).
int mixed_geometry(int ker, int64_t nt, int64_t ns, const DenseShape& shape, MixedGeometry* g, size_t part_budget) {
  DeviceInfo dev;
  SCTL_TRY(device_info(&dev));
  SCTL_CHECK_ARG(ns <= 0xffffffffLL && nt <= 0xffffffffLL, "mixed precision supports at most 2^32-1 points");
  g->mfma = far_mfma_at(ker, nt, ns);
  g->ti = g->mfma ? 0 : std::min(tpl_index(shape.tpl), max_tpl_index(ker));
  const int tpl = TPLS[g->ti];
  g->tb = (nt + (int64_t)WG * tpl - 1) / ((int64_t)WG * tpl);
  SCTL_CHECK_ARG(g->tb <= 0x7fffffffLL, "too many targets for one launch");
  g->ntiles = (ns + TILE - 1) / TILE;
  SCTL_CHECK_ARG(g->ntiles <= 0x7fffffffLL, "too many sources for one launch");
  g->Q = layout_q(ker);
  // Enough workgroups for 32 per CU (one tile per split at the least): a
  // small problem (a few hundred tiles) still fills the GPU.  The matrix-core
  // kernel's, shorter and four or three to a CU, take 96, so that the last ones
  // to run leave fewer CUs idle: Laplace FxU 50000^2 461 -> 448 us, 131072 x
  // 150001 2452 -> 2408, 524288^2 28.96 -> 28.41 ms; Stokes FxU 131072 x 150001
  // 6885 -> 6784 us.
  constexpr int64_t SPLIT_TILES = 256;
  const int64_t want = (g->mfma ? 96LL : 32LL) * std::max(dev.num_cus, 1);
  int64_t nsplit = g->tb < want ? (want + g->tb - 1) / g->tb : 1;
  nsplit = std::min<int64_t>(std::min<int64_t>(nsplit, g->ntiles), 65535);
  nsplit = std::min<int64_t>(std::max<int64_t>(nsplit, (g->ntiles + SPLIT_TILES - 1) / SPLIT_TILES), 65535);
  g->tps = (g->ntiles + nsplit - 1) / nsplit;
  g->nsplit = (g->ntiles + g->tps - 1) / g->tps;
  int K0, K1, ND;
  kernel_dims(ker, &K0, &K1, &ND);
  g->packed_bytes = sizeof(float4) * g->Q * TILE * g->ntiles;
  // tile centres, then sub-tiles, then the targets in their order
  g->meta_bytes = (sizeof(double4) + sizeof(float4) * (WG / 64)) * g->ntiles + sizeof(double) * 3 * nt;
  const size_t split_bytes = sizeof(double) * (size_t)nt * K1;
  g->group = split_group(g->nsplit, split_bytes, part_budget);
  g->part_bytes = g->group > 1 ? split_bytes * g->group : 0;
  return SCTL_AMD_SUCCESS;
}

size_t mixed_order_bytes(int64_t nt, int64_t ns) { return hilbert_order_bytes(ns, nt); }

int mixed_order(const double* r_trg, int64_t nt, const double* r_src, int64_t ns, uint32_t* tperm, uint32_t* sperm,
                void* work, hipStream_t stream) {
  Scratch own;
  if (!work) {
    SCTL_TRY(own.alloc(mixed_order_bytes(nt, ns), stream));
    work = own.as<void>();
  }
  return hilbert_order(r_src, ns, sperm, r_trg, nt, tperm, work, stream);
}

int mixed_apply(int ker, int newton, const MixedGeometry& g, const DenseShape& shape, const double* r_trg, int64_t nt,
                const uint32_t* tperm, const double* r_src, const double* n_src, const double* v_src, int64_t ns,
                const uint32_t* sperm, float4* packed, double4* meta, double* part, double* v_trg, double ctx,
                hipStream_t stream) {
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  SCTL_CHECK_ARG(g.group <= 1 || part, "no buffer for the split partial sums");
  int K0, K1, ND;
  kernel_dims(ker, &K0, &K1, &ND);
  // The sub-tile records follow the tile centres in the same buffer, then
  // the targets in the order tperm (written by the pack launch's last
  // workgroups), which the pairwise kernel reads once per split.
  float4* sub = reinterpret_cast<float4*>(meta + g.ntiles);
  double* xt_sorted = reinterpret_cast<double*>(sub + g.ntiles * (WG / 64));
  hipLaunchKernelGGL(pack_fn(ker), dim3((unsigned)(g.ntiles + (nt + WG - 1) / WG)), dim3(WG), 0, stream, r_src, n_src,
                     v_src, ns, sperm, packed, meta, sub, g.ntiles, r_trg, nt, tperm, xt_sorted);
  SCTL_HIP_TRY(hipGetLastError());
  const double scale = (double)(kernel_scale(ker) * fold_factor(ker, newton ? 1 : 0));
  const EvalMixFn fn = mix_fn(ker, newton, g.ti, g.mfma);
  size_t dyn = 0;
  SCTL_TRY(occupancy_lds((const void*)fn, shape.occ, sizeof(float4) * TILE * g.Q, &dyn));
  if (!stream_capturing(stream)) profile_count(ker, nt * ns);
  // Groups of g.group splits: tiles [y0*tps, (y0+gy)*tps) per launch.
  for (int64_t y0 = 0; y0 < g.nsplit; y0 += g.group) {
    const int64_t gy = std::min(g.group, g.nsplit - y0);
    const int64_t tile0 = y0 * g.tps, ntiles = std::min(g.ntiles - tile0, gy * g.tps);
    const bool direct = gy == 1;
    {
      ProfileScope prof(stream);
      hipLaunchKernelGGL(fn, split_grid(g.tb, gy, WG), dim3(WG), dyn, stream, xt_sorted, nt, tperm,
                         packed + tile0 * (int64_t)(TILE * g.Q), meta + tile0, sub + tile0 * (WG / 64), ntiles, g.tps,
                         direct ? v_trg : part,
                         direct ? 1 : 0, scale, ctx);
    }
    SCTL_HIP_TRY(hipGetLastError());
    if (!direct) {
      const int64_t n = nt * K1;
      hipLaunchKernelGGL(k_reduce_splits_perm, dim3((unsigned)((4 * n + WG - 1) / WG)), dim3(WG), 0, stream, part, nt, K1,
                         (int)gy, tperm, v_trg, scale);
      SCTL_HIP_TRY(hipGetLastError());
    }
  }
  return SCTL_AMD_SUCCESS;
}

namespace {
// Workspace of one mixed Eval: orders, packed tiles, tile centres and the
// sorts' workspace, then the split partial sums last.
struct MixedCarve {
  size_t sperm, tperm, packed, meta, work, part, fixed_bytes;
};
MixedCarve mixed_carve(const MixedGeometry& g, int64_t nt, int64_t ns) {
  MixedCarve m;
  Carve c;
  m.sperm = c.take(sizeof(uint32_t) * ns);
  m.tperm = c.take(sizeof(uint32_t) * nt);
  m.packed = c.take(g.packed_bytes);
  m.meta = c.take(g.meta_bytes);
  m.work = c.take(mixed_order_bytes(nt, ns));
  m.part = c.take(0);
  m.fixed_bytes = m.part;
  return m;
}
}  // namespace

size_t mixed_fixed_bytes(const MixedGeometry& g, int64_t nt, int64_t ns) { return mixed_carve(g, nt, ns).fixed_bytes; }

int mixed_eval_in(int ker, int newton, const MixedGeometry& g, const DenseShape& shape, const double* r_trg,
                  int64_t nt, const double* r_src, const double* n_src, const double* v_src, int64_t ns,
                  double* v_trg, double ctx, char* w, hipStream_t stream) {
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  const MixedCarve m = mixed_carve(g, nt, ns);
  uint32_t* sperm = reinterpret_cast<uint32_t*>(w + m.sperm);
  uint32_t* tperm = reinterpret_cast<uint32_t*>(w + m.tperm);
  SCTL_TRY(mixed_order(r_trg, nt, r_src, ns, tperm, sperm, w + m.work, stream));
  return mixed_apply(ker, newton, g, shape, r_trg, nt, tperm, r_src, n_src, v_src, ns, sperm,
                     reinterpret_cast<float4*>(w + m.packed), reinterpret_cast<double4*>(w + m.meta),
                     g.part_bytes ? reinterpret_cast<double*>(w + m.part) : nullptr, v_trg, ctx, stream);
}

int launch_eval_mixed(int ker, int newton, const double* r_trg, int64_t nt, const double* r_src,
                      const double* n_src, const double* v_src, int64_t ns, double* v_trg, const DenseShape& shape,
                      double ctx, hipStream_t stream) {
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  if (mixed_runs_f64(ker, nt, ns))
    return launch_eval_f64(ker, newton, r_trg, nt, r_src, n_src, v_src, ns, v_trg, shape, ctx, stream);
  MixedGeometry g;
  SCTL_TRY(mixed_geometry(ker, nt, ns, shape, &g));
  // One allocation for the call: orders, packed tiles, the sorts' workspace
  // and the partial sums.
  Scratch buf;
  SCTL_TRY(buf.alloc(mixed_fixed_bytes(g, nt, ns) + g.part_bytes, stream));
  return mixed_eval_in(ker, newton, g, shape, r_trg, nt, r_src, n_src, v_src, ns, v_trg, ctx, buf.as<char>(),
                       stream);
}

}  // namespace sctl_amd
