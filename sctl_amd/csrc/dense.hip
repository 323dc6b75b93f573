// Dense direct summation on gfx950: FP64 Eval and KernelMatrix.
//
// FP64 Eval (reference: generic-kernel.txx:102-211).  A workgroup of 256 lanes
// owns 256*TPL targets (TPL targets per lane, held in registers) and walks a
// contiguous range of sources in tiles of TILE sources staged through LDS;
// every lane of a wave reads the same source record (an LDS broadcast).  When
// there are too few target blocks to fill the 256 CUs, the source range is
// split over the grid, down to a fraction of a tile per workgroup
// (split_sources), and the per-split sums are reduced in split order by a
// second kernel.  No matrix cores: their FP64 rate is the vector rate.
//
// FP64 path: each tile is summed over its sources in index order, and the
// tiles' sums in order (shorter sums than one running accumulator's, so less
// rounding: Laplace DxU 100003 x 130001, error against 64 bits 2.9e-15 ->
// 1.0e-15).  A tile whose sum is not finite (some r2 == 0 in that tile) is
// redone with the r2 > 0 mask.
//
// The mixed-precision Eval is in mixed.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "internal.hpp"
#include "kernels.hpp"

namespace sctl_amd {

constexpr int WG = 256;
constexpr int TILE = 256;
constexpr int UNROLL = 2;  // sources per step of the pair loop; divides TILE

// Far-away padding for the unused slots of a partial tile: the contribution is
// a finite, vanishing kernel value times a zero density.
constexpr double PAD_F64 = 1e100;


// ------------------------------------------------------------------ FP64 Eval
template <int KER, int TPL, int NEWTON>
__global__ void __launch_bounds__(WG)
k_eval_f64(const double* __restrict__ xt, int64_t nt, const double* __restrict__ xs, const double* __restrict__ xn,
           const double* __restrict__ fs, int64_t ns, int64_t chunk, double* __restrict__ out, int direct,
           double scale, double mu) {
  using K = Ker<KER>;
  // The double layer stages f n, one multiplication per pair fewer, but for the
  // full-precision sums of few sources (FOLD_SOURCES): f n is rounded, which
  // n.r near 0 enlarges.
  constexpr bool FN = KER == LAP_DXU && NEWTON != 2;
  constexpr int K0 = K::K0, K1 = K::K1, ND = K::ND, R = rec_f64<KER, FN>();
  // Sources per tile.  The Helmholtz kernels' loop runs whole tiles (below), so
  // theirs are as long as the shortest split.
  constexpr int TS = needs_ctx(KER) ? 64 : TILE;
  __shared__ double lds[TILE * R];

  const int tid = threadIdx.x;
  const SplitCoord wg = split_coord((nt + WG * TPL - 1) / (WG * TPL));
  const int64_t s_begin = wg.split * chunk;
  const int64_t s_end = s_begin + chunk < ns ? s_begin + chunk : ns;
  const int64_t t0 = wg.block * (WG * TPL) + tid;

  double tx[TPL], ty[TPL], tz[TPL], tot[TPL][K1];
#pragma unroll
  for (int j = 0; j < TPL; j++) {
    const int64_t t = t0 + (int64_t)j * WG;
    const bool ok = t < nt;
    tx[j] = ok ? xt[t * 3 + 0] : 0.0;
    ty[j] = ok ? xt[t * 3 + 1] : 0.0;
    tz[j] = ok ? xt[t * 3 + 2] : 0.0;
#pragma unroll
    for (int k = 0; k < K1; k++) tot[j][k] = 0.0;
  }

  for (int64_t sb = s_begin; sb < s_end; sb += TS) {
    const int len = (int)(s_end - sb < TS ? s_end - sb : TS);
    __syncthreads();
    for (int i = tid; i < TS; i += WG) {
      double* rec = lds + i * R;
      if (i < len) {
        const int64_t s = sb + i;
        rec[0] = xs[s * 3 + 0];
        rec[1] = xs[s * 3 + 1];
        rec[2] = xs[s * 3 + 2];
        if constexpr (FN) {
          const double f = fs[s];
#pragma unroll
          for (int k = 0; k < 3; k++) rec[3 + k] = f * xn[s * 3 + k];
        } else {
#pragma unroll
          for (int k = 0; k < ND; k++) rec[3 + k] = xn[s * 3 + k];
#pragma unroll
          for (int k = 0; k < K0; k++) rec[3 + ND + k] = fs[s * K0 + k];
        }
      } else {
        rec[0] = rec[1] = rec[2] = PAD_F64;
#pragma unroll
        for (int k = 3; k < R; k++) rec[k] = 0.0;
      }
    }
    __syncthreads();

    double acc[TPL][K1];  // this tile's sums
#pragma unroll
    for (int j = 0; j < TPL; j++)
#pragma unroll
      for (int k = 0; k < K1; k++) acc[j][k] = 0.0;

    // One source of the tile; `masked`: r2 == 0 contributes 0.  The masked
    // double layer takes n and f from memory, not f n: a non-finite density
    // (which sends its tile there) then gives what n.r z^3 f gives.
    auto source = [&](int i, auto masked) {
      constexpr bool MASK = decltype(masked)::value;
      const double* rec = lds + i * R;
      const double sx = rec[0], sy = rec[1], sz = rec[2];
      double n[3] = {0, 0, 0}, f[K0];
#pragma unroll
      for (int k = 0; k < ND; k++) n[k] = rec[3 + k];
#pragma unroll
      for (int k = 0; k < (FN ? 0 : K0); k++) f[k] = rec[3 + ND + k];
      if constexpr (FN && MASK) {
#pragma unroll
        for (int k = 0; k < 3; k++) n[k] = xn[(sb + i) * 3 + k];
        f[0] = fs[sb + i];
      }
#pragma unroll
      for (int j = 0; j < TPL; j++) {
        if constexpr (FN && !MASK)
          lap_dxu_fn<NEWTON, false>(acc[j][0], tx[j] - sx, ty[j] - sy, tz[j] - sz, n);
        else interact<KER, NEWTON, MASK>(acc[j], tx[j] - sx, ty[j] - sy, tz[j] - sz, n, f, mu);
      }
    };
    if constexpr (needs_ctx(KER)) {
      // The whole tile, written out: from a loop of variable length, or through
      // the lambda, the compiler does not keep the sine's and cosine's constants
      // in registers (Helmholtz FxU 70 -> 83 instructions per pair, 32768^2 2.04
      // -> 2.28 ms).
#pragma unroll 2
      for (int i = 0; i < TS; i++) {
        const double* rec = lds + i * R;
        double n[3] = {0, 0, 0}, f[K0];
#pragma unroll
        for (int k = 0; k < ND; k++) n[k] = rec[3 + k];
#pragma unroll
        for (int k = 0; k < K0; k++) f[k] = rec[3 + ND + k];
#pragma unroll
        for (int j = 0; j < TPL; j++)
          interact<KER, NEWTON, false>(acc[j], tx[j] - rec[0], ty[j] - rec[1], tz[j] - rec[2], n, f, mu);
      }
    } else {
      // up to the first multiple of UNROLL at or past the tile's last source
      // (the staged padding covers the rest)
      for (int i = 0; i < len; i += UNROLL) {
#pragma unroll
        for (int u = 0; u < UNROLL; u++) source(i + u, std::false_type());
      }
    }

    bool bad = false;
#pragma unroll
    for (int j = 0; j < TPL; j++)
#pragma unroll
      for (int k = 0; k < K1; k++) bad |= !__builtin_isfinite(acc[j][k]);
    if (bad) {  // some r2 == 0 in this tile (or non-finite input): redo it masked
#pragma unroll
      for (int j = 0; j < TPL; j++)
#pragma unroll
        for (int k = 0; k < K1; k++) acc[j][k] = 0.0;
      for (int i = 0; i < len; i++) source(i, std::true_type());
    }
#pragma unroll
    for (int j = 0; j < TPL; j++)
#pragma unroll
      for (int k = 0; k < K1; k++) tot[j][k] += acc[j][k];
  }

#pragma unroll
  for (int j = 0; j < TPL; j++) {
    const int64_t t = t0 + (int64_t)j * WG;
    if (t < nt) {
#pragma unroll
      for (int k = 0; k < K1; k++) {
        if (direct) out[t * K1 + k] += tot[j][k] * scale;
        else out[wg.split * nt * K1 + t * K1 + k] = tot[j][k];
      }
    }
  }
}

// v_trg[i] += scale * sum_{y < nsplit} part[y][i]; one lane quad per element
// (sum_splits_quad).
__global__ void __launch_bounds__(WG)
k_reduce_splits(const double* __restrict__ part, int64_t n, int nsplit, double* __restrict__ out, double scale) {
  const int64_t i = ((int64_t)blockIdx.x * WG + threadIdx.x) >> 2;
  const double s = sum_splits_quad(part, n, nsplit, i, i < n);
  if (i < n && (threadIdx.x & 3) == 0) out[i] += s * scale;
}

// ------------------------------------------------------------- KernelMatrix
// M[(s*K0+k0)*ld + t*K1+k1] = scale * u[k0][k1]; one lane per target, the
// workgroup's gridDim.y slices stride over the sources.  HBM-write bound: the
// rows leave through LDS as consecutive words, so that a wave's store covers
// four whole 128-byte lines where a lane's own K1 words would leave lines to
// be merged.  A row starts anywhere within a line, so each workgroup writes the
// whole lines that start within its columns, and computes HALO targets of its
// predecessor's for the words of the first; only a row's first and last line
// is shared with its neighbours.  Where a source gives one word per target,
// four sources go under one barrier and the stores are nontemporal (wider rows
// were 10-25 % slower with them).  Two words per target are one 16-byte store
// and stay as they are.  MI355X, TB/s written, lane by lane / through LDS:
//   Laplace FxU 10001 x 9000 3.0 / 5.4, 8192 x 8192 3.3 / 5.5
//   Stokes FxU 2003 x 3001 4.5 / 5.3; Laplace FxdU 3658 x 1056 4.8 / 5.8
//   Laplace Fxd2U 2001 x 2000 2.7 / 6.5; Stokes FxT 1000 x 1003 2.7 / 6.5
// (a fill of 2 GiB: 6.8; Helmholtz FxU, left alone, 5.4-5.9).
template <int K1> constexpr int kmat_halo() { return (15 + K1 - 1) / K1; }  // targets that cover 15 words
template <int KER> constexpr int kmat_sources() { return Ker<KER>::K0 * Ker<KER>::K1 == 1 ? 4 : 1; }

template <int KER, int NEWTON>
__global__ void __launch_bounds__(WG)
k_kernel_matrix(const double* __restrict__ xt, int64_t nt, const double* __restrict__ xs,
                const double* __restrict__ xn, int64_t ns, double* __restrict__ M, double scale, double mu) {
  using K = Ker<KER>;
  constexpr int K0 = K::K0, K1 = K::K1, ND = K::ND, SB = kmat_sources<KER>();
  constexpr bool DIRECT = K1 == 2;
  constexpr int HALO = DIRECT ? 0 : kmat_halo<K1>(), TB = WG - HALO;
  const int tid = threadIdx.x;
  const int64_t first = (int64_t)blockIdx.x * TB, t = first - HALO + tid, ld = nt * K1;
  const int64_t tc = t < 0 ? 0 : (t < nt ? t : nt - 1);  // the targets past either end are not written
  const double tx = xt[tc * 3 + 0], ty = xt[tc * 3 + 1], tz = xt[tc * 3 + 2];
  auto values = [&](int64_t s, double(&u)[K0][K1]) {
    double n[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < ND; k++) n[k] = xn[s * 3 + k];
    kmatrix<KER, NEWTON>(u, tx - xs[s * 3 + 0], ty - xs[s * 3 + 1], tz - xs[s * 3 + 2], n, mu);
  };
  if constexpr (DIRECT) {
    for (int64_t s = blockIdx.y; s < ns; s += gridDim.y) {
      double u[K0][K1];
      values(s, u);
      if (t < nt) {
#pragma unroll
        for (int k0 = 0; k0 < K0; k0++)
#pragma unroll
          for (int k1 = 0; k1 < K1; k1++) M[(s * K0 + k0) * ld + t * K1 + k1] = u[k0][k1] * scale;
      }
    }
  } else {
    __shared__ double rows[2][SB][WG * K1];
    const int64_t base = (first - HALO) * K1, c_lo = first * K1, c_hi = (first + TB) * K1;
    // Row r of M from a buffer.
    auto write = [&](int64_t r, const double* row) {
      double* Mr = M + r * ld;
      const int64_t a = (int64_t)((reinterpret_cast<uintptr_t>(Mr) >> 3) & 15);
      const int64_t c0 = blockIdx.x ? c_lo - ((c_lo + a) & 15) : 0;
      const int64_t c1 = c_hi < ld ? c_hi - ((c_hi + a) & 15) : ld;
#pragma unroll
      for (int i = 0; i < K1 + 1; i++) {  // c1 - c0 <= TB * K1 + 15 <= (K1 + 1) * WG
        const int64_t c = c0 + tid + (int64_t)i * WG;
        if (c < c1) {
          if constexpr (K1 == 1) __builtin_nontemporal_store(row[c - base], Mr + c);
          else Mr[c] = row[c - base];
        }
      }
    };
    // Two buffers, one barrier each time one is filled: a thread fills a buffer
    // again only after every thread has passed the other's barrier, and so has
    // read this one.
    int buf = 0;
    for (int64_t s = (int64_t)blockIdx.y * SB; s < ns; s += (int64_t)gridDim.y * SB) {
      double u[SB][K0][K1];
#pragma unroll
      for (int j = 0; j < SB; j++) values(s + j < ns ? s + j : ns - 1, u[j]);
#pragma unroll
      for (int k0 = 0; k0 < K0; k0++) {
#pragma unroll
        for (int j = 0; j < SB; j++)
#pragma unroll
          for (int k1 = 0; k1 < K1; k1++) rows[buf][j][tid * K1 + k1] = u[j][k0][k1] * scale;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SB; j++)
          if (s + j < ns) write((s + j) * K0 + k0, rows[buf][j]);
        buf ^= 1;
      }
    }
  }
}

// --------------------------------------------------------------- dispatch
namespace {

using EvalF64Fn = void (*)(const double*, int64_t, const double*, const double*, const double*, int64_t, int64_t,
                           double*, int, double, double);
using KMatFn = void (*)(const double*, int64_t, const double*, const double*, int64_t, double*, double, double);

constexpr int TPLS[3] = {1, 2, 4};
int tpl_index(int tpl) { return tpl >= 4 ? 2 : (tpl >= 2 ? 1 : 0); }

template <int KER, int NEWTON> EvalF64Fn f64_fn(int ti) {
  constexpr int MT = max_tpl<KER>();
  if (ti >= 2 && MT >= 4) return k_eval_f64<KER, (MT >= 4 ? 4 : 1), NEWTON>;
  if (ti >= 1 && MT >= 2) return k_eval_f64<KER, (MT >= 2 ? 2 : 1), NEWTON>;
  return k_eval_f64<KER, 1, NEWTON>;
}
EvalF64Fn f64_fn(int ker, int newton, int ti) {
  return with_kernel(ker, [&](auto kc) {
    constexpr int K = decltype(kc)::value;
    if constexpr (Ker<K>::POW != 0) {
      if (newton == FOLDED) return f64_fn<K, FOLDED>(ti);
    }
    return newton == 0 ? f64_fn<K, 0>(ti) : (newton == 1 ? f64_fn<K, 1>(ti) : f64_fn<K, 2>(ti));
  });
}
int f64_step(int ker, int newton, int64_t ns) {
  return newton == 2 && one_power(ker) && ns >= FOLD_SOURCES ? FOLDED : newton;
}
int max_tpl_index(int ker) {
  return with_kernel(ker, [](auto kc) { return tpl_index(max_tpl<decltype(kc)::value>()); });
}
KMatFn kmat_fn(int ker, int newton) {
  return with_kernel(ker, [&](auto kc) -> KMatFn {
    constexpr int K = decltype(kc)::value;
    return newton == 0 ? k_kernel_matrix<K, 0> : (newton == 1 ? k_kernel_matrix<K, 1> : k_kernel_matrix<K, 2>);
  });
}

// Splits the source range over the grid: *nsplit chunks of *chunk sources
// (the last may be shorter), for about 32 workgroups per CU.  A chunk longer
// than a tile is a whole number of tiles; a shorter one is a multiple of 64
// sources.  Device time of one apply on MI355X, before and after small
// problems were cut below four tiles per workgroup and large ones finer than
// eight workgroups per CU (whose last ones left CUs idle):
//   Laplace FxU 2000 x 3000     57.1 -> 11.2 us (8 target blocks: 24 -> 376 workgroups)
//   Laplace DxU 2503 x 3001     74.2 -> 12.7 us
//   Stokes FxU 5000 x 7000      79.4 -> 43 us
//   Laplace DxU 100003 x 130001 8.84 -> 8.29 ms
// At 16 workgroups per CU 20 000 x 20 000 took 4 % longer and nothing else
// more than 1 % less; 32 instead of 64 sources gave nothing from 2000 points
// on, where the per-workgroup latency and the reduction of more splits weigh
// as much as the shorter loop.  No split is longer than SPLIT_TILES tiles
// (2 MiB of Laplace sources): the workgroups resident at a time (dispatched in
// linear-index order) then share one split in L2 rather than each streaming
// the whole source array.
void split_sources(int64_t target_blocks, int64_t ns, int num_cus, int64_t* nsplit, int64_t* chunk) {
  constexpr int64_t SPLIT_TILES = 256, MIN_CHUNK = 64;
  const int64_t want = 32LL * std::max(num_cus, 1);
  int64_t n = target_blocks < want ? (want + target_blocks - 1) / target_blocks : 1;
  n = std::max<int64_t>(n, (ns + SPLIT_TILES * TILE - 1) / (SPLIT_TILES * TILE));
  n = std::min<int64_t>(n, 65535);
  int64_t c = (ns + n - 1) / n;
  const int64_t step = c > TILE ? TILE : MIN_CHUNK;
  c = (c + step - 1) / step * step;
  *chunk = c;
  *nsplit = (ns + c - 1) / c;
}

}  // namespace

// Bytes of the per-split partial sums an FP64 Eval of this size and shape
// needs, bounded by part_budget (split_group).
int f64_part_bytes(int ker, int64_t nt, int64_t ns, const DenseShape& shape, size_t* bytes, size_t part_budget) {
  *bytes = 0;
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  DeviceInfo dev;
  SCTL_TRY(device_info(&dev));
  int K0, K1, ND;
  kernel_dims(ker, &K0, &K1, &ND);
  const int tpl = TPLS[std::min(tpl_index(shape.tpl), max_tpl_index(ker))];
  const int64_t tb = (nt + (int64_t)WG * tpl - 1) / ((int64_t)WG * tpl);
  int64_t nsplit, chunk;
  split_sources(tb, ns, dev.num_cus, &nsplit, &chunk);
  const size_t split_bytes = sizeof(double) * (size_t)nt * K1;
  const int64_t group = split_group(nsplit, split_bytes, part_budget);
  *bytes = group > 1 ? split_bytes * group : 0;
  return SCTL_AMD_SUCCESS;
}

int f64_apply(int ker, int newton, const double* r_trg, int64_t nt, const double* r_src, const double* n_src,
              const double* v_src, int64_t ns, double* v_trg, const DenseShape& shape, double ctx, double* part,
              hipStream_t stream, size_t part_budget) {
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  DeviceInfo dev;
  SCTL_TRY(device_info(&dev));
  int K0, K1, ND;
  kernel_dims(ker, &K0, &K1, &ND);
  const int ti = std::min(tpl_index(shape.tpl), max_tpl_index(ker)), tpl = TPLS[ti];
  const int64_t tb = (nt + (int64_t)WG * tpl - 1) / ((int64_t)WG * tpl);
  SCTL_CHECK_ARG(tb <= 0x7fffffffLL, "too many targets for one launch");
  int64_t nsplit, chunk;
  split_sources(tb, ns, dev.num_cus, &nsplit, &chunk);
  const int64_t group = split_group(nsplit, sizeof(double) * (size_t)nt * K1, part_budget);
  SCTL_CHECK_ARG(group <= 1 || part, "no buffer for the split partial sums");
  const int step = f64_step(ker, newton, ns);
  const double scale = (double)(kernel_scale(ker) * fold_factor(ker, step));
  const EvalF64Fn fn = f64_fn(ker, step, ti);
  size_t dyn = 0;
  SCTL_TRY(occupancy_lds((const void*)fn, shape.occ, 0, &dyn));
  if (!stream_capturing(stream)) profile_count(ker, nt * ns);
  // Groups of `group` splits: sources [y0*chunk, (y0+gy)*chunk) per launch.
  for (int64_t y0 = 0; y0 < nsplit; y0 += group) {
    const int64_t gy = std::min(group, nsplit - y0);
    const int64_t s0 = y0 * chunk, ns_g = std::min(ns - s0, gy * chunk);
    const bool direct = gy == 1;
    {
      ProfileScope prof(stream);
      hipLaunchKernelGGL(fn, split_grid(tb, gy, WG), dim3(WG), dyn, stream, r_trg, nt, r_src + s0 * 3,
                         ND ? n_src + s0 * 3 : n_src, v_src + s0 * K0, ns_g, chunk, direct ? v_trg : part,
                         direct ? 1 : 0, scale, ctx);
    }
    SCTL_HIP_TRY(hipGetLastError());
    if (!direct) {
      const int64_t n = nt * K1;
      hipLaunchKernelGGL(k_reduce_splits, dim3((unsigned)((4 * n + WG - 1) / WG)), dim3(WG), 0, stream, part, n,
                         (int)gy, v_trg, scale);
      SCTL_HIP_TRY(hipGetLastError());
    }
  }
  return SCTL_AMD_SUCCESS;
}

int launch_eval_f64(int ker, int newton, const double* r_trg, int64_t nt, const double* r_src, const double* n_src,
                    const double* v_src, int64_t ns, double* v_trg, const DenseShape& shape, double ctx,
                    hipStream_t stream) {
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  size_t bytes = 0;
  SCTL_TRY(f64_part_bytes(ker, nt, ns, shape, &bytes));
  Scratch part;
  SCTL_TRY(part.alloc(bytes, stream));
  return f64_apply(ker, newton, r_trg, nt, r_src, n_src, v_src, ns, v_trg, shape, ctx, part.as<double>(), stream);
}

int launch_kernel_matrix(int ker, int newton, const double* r_trg, int64_t nt, const double* r_src,
                         const double* n_src, int64_t ns, double* M, double ctx, hipStream_t stream) {
  if (nt <= 0 || ns <= 0) return SCTL_AMD_SUCCESS;
  DeviceInfo dev;
  SCTL_TRY(device_info(&dev));
  int K0, K1, ND;
  kernel_dims(ker, &K0, &K1, &ND);
  const int64_t per = K1 == 2 ? WG : WG - (15 + K1 - 1) / K1;  // targets per workgroup (kmat_halo)
  const int64_t tb = (nt + per - 1) / per;
  SCTL_CHECK_ARG(tb <= 0x7fffffffLL, "too many targets for one launch");
  // About 32 workgroups per CU, each with several rows to its targets (8 to 64
  // are within 3 %); the 16-byte stores run best with a source to a workgroup
  // (3501 x 3000: 5.9 against 5.3 TB/s).
  const int64_t want = 32LL * std::max(dev.num_cus, 1);
  const int64_t gy = K1 == 2 ? std::min<int64_t>(ns, 8192)
                             : std::min<int64_t>(ns, std::min<int64_t>(65535, (want + tb - 1) / tb));
  const double scale = kernel_scale(ker);
  profile_count(ker, nt * ns);
  ProfileScope prof(stream);
  hipLaunchKernelGGL(kmat_fn(ker, newton), dim3((unsigned)tb, (unsigned)gy), dim3(WG), 0, stream, r_trg, nt, r_src,
                     n_src, ns, M, scale, ctx);
  SCTL_HIP_TRY(hipGetLastError());
  return SCTL_AMD_SUCCESS;
}

}  // namespace sctl_amd
