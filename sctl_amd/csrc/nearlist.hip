// Near-interaction lists of BoundaryIntegralOp on the device: the
// single-process output of BuildNearList (boundary_integral.txx:50-520).
//
// Definition (the reference's, :390-401): target t is near element e when
// some node s of e has |x_t - x_s|^2 < r_s^2.  The near pairs are listed by
// element, then target index (:418-428 sort by (elem_idx, idx)); per pair the
// target's coordinates (and normal) are gathered (:430-447); near_elem_cnt /
// near_elem_dsp count pairs per element (:449-476); near_scatter_index orders
// the pairs by target (SortScatterIndex, :483, comm.txx:1393) and
// near_trg_cnt / near_trg_dsp count them per target, with dsp 0 for a target
// without pairs (:485-514).  The reference sorts the pairs of one target by
// key only with std::sort, which leaves their order unspecified; here they
// follow element order.
//
// The reference finds candidates through a Morton tree of the nodes.  Here:
//   1. targets get 63-bit Morton keys over the reference's bounding cube
//      (all points, grown by 5 % per side, :104-154), are radix sorted and
//      copied into that order;
//   2. one workgroup per element takes the bounding boxes of its nodes, 64 at a
//      time, and of all of them grown by the largest radius, picks the finest
//      Morton depth at which that box spans at most 64 cells, finds the cells'
//      targets by binary search in the sorted keys (one cell per lane), and
//      its four waves take the cells' targets 64 at a time as one list: those
//      inside the grown box are queued and tested in batches (k_nl_elements);
//   3. the near ones go out as (element, target) keys, gathered in LDS and
//      appended through an atomic counter once per element (one atomic per
//      batch of 64 tests was most of this kernel's time: a single address
//      takes ~75 per microsecond); the buffer holds 24 pairs per target (fewer from
//      256 MiB on), and a list that has more is filled again into one of the
//      size then known;
//   4. the keys are radix sorted (so the list does not depend on the order of
//      the appends), in 32 bits where an element and a target number fit; each
//      element's range is found by binary search, and a stable sort of the
//      pairs by target gives the scatter index.
// Every target within a node's radius lies in the grown box, hence in one of
// the cells (the cell range is computed with the same quantisation as the
// target keys), so the list is exact.
//
// Build, get and destroy for 2048 elements (0.9 M nodes) and 500 009 targets on
// MI355X: 5.53 -> 0.87 ms; the passes over the elements, two of them before
// (candidates counted, then tested), 1.78 -> 0.35 ms, the sorts of the pairs 0.38
// -> 0.19.  Scratch and results are one block each of memory kept between
// builds (block_take): seven hipMalloc and hipFree each for the results, and
// their waits, were half of the time.
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "internal.hpp"
#include "wave.hpp"

namespace sctl_amd {
namespace {

// Device memory of near lists (a build's scratch, a list's results) kept for
// the next build: up to KEEP_BLOCKS blocks and KEEP_BYTES per device, the
// oldest given back beyond that, all of them where an allocation of the library
// fails (blocks_release).  A block carries an event recorded after its
// last use; whoever takes it makes its stream wait for that event, so threads
// and streams share the blocks freely.  (The stream-ordered pool, asked for
// such buffers again while the last read of the previous ones was under way,
// mapped new memory instead, and past its threshold did so on every call: 5.4
// instead of 1.3 ms, or 1.3, from one run to the next.)
struct Block {
  char* p = nullptr;
  size_t bytes = 0;
  int device = 0;
  hipEvent_t used = nullptr;
};
constexpr size_t KEEP_BYTES = (size_t)2 << 30;
constexpr int KEEP_BLOCKS = 8;
std::mutex g_blocks_mutex;
std::vector<Block>& free_blocks() {  // oldest first; never destroyed (the runtime may be gone by then)
  static auto* v = new std::vector<Block>();
  return *v;
}

void block_drop(Block b) {  // hipFree waits for the device
  int cur = -1;
  (void)hipGetDevice(&cur);
  if (cur != b.device) (void)hipSetDevice(b.device);
  if (b.p) (void)hipFree(b.p);
  if (b.used) (void)hipEventDestroy(b.used);
  if (cur >= 0 && cur != b.device) (void)hipSetDevice(cur);
}

}  // namespace

void blocks_release() {
  std::vector<Block> all;
  {
    std::lock_guard<std::mutex> lock(g_blocks_mutex);
    all.swap(free_blocks());
  }
  for (Block& b : all) block_drop(b);
}

namespace {

// A block of at least `bytes` on the current device, usable on stream s.
int block_take(size_t bytes, hipStream_t s, Block* out) {
  DeviceInfo dev;
  SCTL_TRY(device_info(&dev));
  {
    std::lock_guard<std::mutex> lock(g_blocks_mutex);
    auto& v = free_blocks();
    size_t best = v.size();
    for (size_t i = 0; i < v.size(); i++)
      if (v[i].device == dev.device && v[i].bytes >= bytes && v[i].bytes / 4 <= bytes + ((size_t)16 << 20) &&
          (best == v.size() || v[i].bytes < v[best].bytes))
        best = i;
    if (best < v.size()) {
      *out = v[best];
      v.erase(v.begin() + best);
    }
  }
  if (out->p) {
    const hipError_t e = hipStreamWaitEvent(s, out->used, 0);
    if (e == hipSuccess) return SCTL_AMD_SUCCESS;
    block_drop(*out);  // uses that stream s does not wait for
    *out = Block();
    SCTL_HIP_TRY(e);
  }
  size_t step = (size_t)1 << 16;  // an eighth of the size's power of two, so that sizes that differ a little reuse
  while (step * 16 <= bytes) step *= 2;
  out->device = dev.device;
  out->bytes = (bytes + step - 1) / step * step;
  if (hipMalloc(reinterpret_cast<void**>(&out->p), out->bytes) != hipSuccess) {
    (void)hipGetLastError();
    blocks_release();
    out->p = nullptr;
    const hipError_t e = hipMalloc(reinterpret_cast<void**>(&out->p), out->bytes);
    if (e != hipSuccess) {
      (void)hipGetLastError();  // the caller may ask for less
      *out = Block();
      SCTL_HIP_TRY(e);
    }
  }
  const hipError_t e = hipEventCreateWithFlags(&out->used, hipEventDisableTiming);
  if (e != hipSuccess) {
    out->used = nullptr;
    block_drop(*out);
    *out = Block();
  }
  SCTL_HIP_TRY(e);
  return SCTL_AMD_SUCCESS;
}

// Returns a block whose `used` event has been recorded after its last use.
void block_give(Block b) {
  if (!b.p || !b.used) {
    block_drop(b);
    return;
  }
  std::vector<Block> drop;
  {
    std::lock_guard<std::mutex> lock(g_blocks_mutex);
    auto& v = free_blocks();
    v.push_back(b);
    size_t bytes = 0, count = 0;
    for (const Block& x : v)
      if (x.device == b.device) {
        bytes += x.bytes;
        count++;
      }
    for (size_t i = 0; i < v.size() && (bytes > KEEP_BYTES || count > KEEP_BLOCKS);) {
      if (v[i].device != b.device) {
        i++;
        continue;
      }
      bytes -= v[i].bytes;
      count--;
      drop.push_back(v[i]);
      v.erase(v.begin() + i);
    }
  }
  for (Block& x : drop) block_drop(x);
}

// A build's scratch: given back in stream order when it goes out of scope.
struct BlockScratch {
  Block b;
  hipStream_t s = nullptr;
  int alloc(size_t bytes, hipStream_t stream) {
    s = stream;
    return block_take(bytes, s, &b);
  }
  ~BlockScratch() {
    if (!b.p) return;
    if (hipEventRecord(b.used, s) != hipSuccess) {  // no order known: free it, which waits
      (void)hipGetLastError();
      block_drop(b);
      return;
    }
    block_give(b);
  }
};

}  // namespace
}  // namespace sctl_amd

struct sctl_amd_near_list_s {
  int device = 0;
  int64_t ntrg = 0, nelem = 0, n_near = 0;
  bool has_normal = false;
  sctl_amd::Block buf;  // all results; its event: after every read so far, whichever their streams
  std::mutex read;      // a read's wait, launch and record are one step
  // Some use is not behind buf's event: a captured read (its graph's launches
  // have none), kernels of a build that failed, a read that failed half-way.
  bool loose = false;
  double *d_xtn = nullptr, *d_xntn = nullptr;
  int64_t *d_ecnt = nullptr, *d_edsp = nullptr, *d_scatter = nullptr, *d_tcnt = nullptr, *d_tdsp = nullptr;
  ~sctl_amd_near_list_s() {
    if (loose) sctl_amd::block_drop(buf);  // hipFree waits for what is under way
    else sctl_amd::block_give(buf);
  }
};

namespace sctl_amd {
namespace {

constexpr int NL_WG = 256;
constexpr int MAX_DEPTH = 21;    // 21 bits per axis, 63-bit keys
constexpr int MAX_CELLS = 64;    // cells per element at the chosen depth

__device__ __forceinline__ uint64_t spread21(uint64_t v) {  // 21 bits -> every third bit
  v &= 0x1fffffULL;
  v = (v | (v << 32)) & 0x001f00000000ffffULL;
  v = (v | (v << 16)) & 0x001f0000ff0000ffULL;
  v = (v | (v << 8)) & 0x100f00f00f00f00fULL;
  v = (v | (v << 4)) & 0x10c30c30c30c30c3ULL;
  v = (v | (v << 2)) & 0x1249249249249249ULL;
  return v;
}
__device__ __forceinline__ uint64_t interleave(uint64_t x, uint64_t y, uint64_t z) {
  return spread21(x) | (spread21(y) << 1) | (spread21(z) << 2);
}

// The reference's bounding cube (:104-154), computed once so that the key
// and the search kernels quantise with the same bits: cube = {origin x, y,
// z, 2^21 / edge length}.
__global__ void k_nl_cube(const double* box, double* cube) {  // in place: cube may alias box
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double bl = 0;
  for (int k = 0; k < 3; k++) bl = fmax(bl, box[3 + k] - box[k]);
  const double L = bl > 0 ? bl : 1.0;
  for (int k = 0; k < 3; k++) cube[k] = box[k] - 0.05 * L;
  cube[3] = 2097152.0 / (1.1 * L);
}
__device__ __forceinline__ uint32_t quant(double x, double x0, double scale) {
  double u = (x - x0) * scale;
  u = fmin(fmax(u, 0.0), 2097151.0);  // fmax returns 0 for a NaN u
  return (uint32_t)u;
}

__global__ void __launch_bounds__(NL_WG)
k_nl_keys(const double* __restrict__ xt, int64_t nt, const double* __restrict__ box, uint64_t* __restrict__ keys,
          uint32_t* __restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * NL_WG + threadIdx.x;
  if (i >= nt) return;
  const double scale = box[3];
  keys[i] = interleave(quant(xt[i * 3 + 0], box[0], scale), quant(xt[i * 3 + 1], box[1], scale),
                       quant(xt[i * 3 + 2], box[2], scale));
  idx[i] = (uint32_t)i;
}

__device__ __forceinline__ int64_t lower_bound_u64(const uint64_t* __restrict__ a, int64_t n, uint64_t key) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (a[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// |d|^2 rounded as node_dist2 sums it (boundary_integral.txx:72-79), without
// fused multiply-adds, so the radius test matches the reference's bit for bit.
__device__ __forceinline__ double dist2(double dx, double dy, double dz) {
#pragma clang fp contract(off)
  return (dx * dx + dy * dy) + dz * dz;
}

constexpr int QCAP = 128;          // per-wave queue of candidates inside the grown box
constexpr int NWAVE = NL_WG / 64;  // waves sharing one element's candidates
constexpr int MAX_BOXES = 64;      // node boxes of an element: one per 64 nodes up to 4096 nodes, larger ones beyond
constexpr int HITS = 512;          // near targets a wave gathers before it appends them

struct Cand {
  double x, y, z;
  uint32_t t;
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}
__device__ __forceinline__ uint64_t uniform64(uint64_t v, int lane) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
}

// One workgroup per element: appends the key (e << tbits | t) of each near
// target at out[atomicAdd(counter)], cap entries at most (the counter goes on
// counting).
//
// A candidate inside the grown box is near when it is within some node's
// radius.  Each batch of 64 is decided in three steps, cheapest first:
//   lane per candidate   the node boxes within reach: a box whose nearest point
//                        is not within its largest radius holds no node that
//                        is (dist2 is monotone in each |difference|, so this
//                        is exact).  No box: not near.
//   wave per candidate   64 of the element's nodes, spread over it, one per
//                        lane, one ballot.  Radii of several node spacings
//                        decide nearly every near candidate here.
//   wave per candidate   box by box, those left with the box within reach, 64
//                        nodes a ballot.
// Testing every candidate against the element's nodes chunk by chunk took ~8
// ballots each.
template <class Key>
__global__ void __launch_bounds__(NL_WG)
k_nl_elements(const int64_t* __restrict__ ecnt, const int64_t* __restrict__ edsp, int64_t nsrc,
              const double* __restrict__ xs, const double* __restrict__ rad, int64_t nt,
              const double* __restrict__ xsorted, const uint64_t* __restrict__ skeys,
              const uint32_t* __restrict__ sidx, const double* __restrict__ cube, int tbits,
              unsigned long long* __restrict__ counter, int64_t cap, Key* __restrict__ out) {
  __shared__ Cand queue_all[NWAVE][QCAP];
  __shared__ uint32_t hits_all[NWAVE][HITS];
  __shared__ double box[7][MAX_BOXES];  // lo, hi, largest radius^2
  __shared__ int64_t cell_first[MAX_CELLS];
  __shared__ uint64_t cell_before[MAX_CELLS + 1];
  __shared__ int nhits[NWAVE];
  __shared__ unsigned long long out_base;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  Cand* queue = queue_all[w];
  uint32_t* hits = hits_all[w];
  const int64_t e = blockIdx.x;
  const int64_t s0 = edsp[e], sc = ecnt[e];
  if (!(s0 >= 0 && sc > 0 && s0 <= nsrc && sc <= nsrc - s0 && nt > 0)) return;  // the whole workgroup

  // Node boxes: per_box nodes each, a whole number of 64-node chunks.
  const int64_t nch = (sc + 63) / 64, per_box = (nch + MAX_BOXES - 1) / MAX_BOXES * 64;
  const int nbox = (int)((sc + per_box - 1) / per_box);
  for (int b = w; b < nbox; b += NWAVE) {
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY}, rmax = 0;
    const int64_t end = (b + 1) * per_box < sc ? (b + 1) * per_box : sc;
    for (int64_t s = b * per_box + lane; s < end; s += 64) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double x = xs[(s0 + s) * 3 + k];
        lo[k] = fmin(lo[k], x);
        hi[k] = fmax(hi[k], x);
      }
      rmax = fmax(rmax, fabs(rad[s0 + s]));
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      lo[k] = sctl_amd::wave_min(lo[k]);
      hi[k] = sctl_amd::wave_max(hi[k]);
    }
    rmax = sctl_amd::wave_max(rmax);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        box[k][b] = lo[k];
        box[3 + k][b] = hi[k];
      }
      box[6][b] = rmax * rmax;
    }
  }
  __syncthreads();
  // The element's own box and largest radius.
  double glo[3], ghi[3];
  double rmax = sctl_amd::wave_max(lane < nbox ? box[6][lane] : 0.0);
  if (!(rmax > 0)) return;  // uniform over the workgroup
  rmax = sqrt(rmax);
  const double grow = rmax * (1.0 + 1e-9);  // a margin above the rounding of the additions and of sqrt(r^2)
  uint32_t qlo[3], qhi[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double lo = sctl_amd::wave_min(lane < nbox ? box[k][lane] : INFINITY);
    const double hi = sctl_amd::wave_max(lane < nbox ? box[3 + k][lane] : -INFINITY);
    glo[k] = lo - grow - 1e-14 * fabs(lo);
    ghi[k] = hi + grow + 1e-14 * fabs(hi);
    qlo[k] = quant(glo[k], cube[k], cube[3]);
    qhi[k] = quant(ghi[k], cube[k], cube[3]);
  }
  int shift = 0;
  int64_t cells = 1;
  for (int d = MAX_DEPTH; d >= 0; d--) {
    shift = MAX_DEPTH - d;
    auto span = [&](int k) { return (int64_t)(qhi[k] >> shift) - (qlo[k] >> shift) + 1; };
    cells = span(0) * span(1);
    if (cells > MAX_CELLS) continue;  // times span(2) it may wrap: 2^63 for a box that spans the cube
    cells *= span(2);
    if (cells <= MAX_CELLS) break;
  }
  // Targets of the cells, one cell per lane of wave 0: two binary searches.
  if (w == 0) {
    int64_t i0 = 0, i1 = 0;
    if (lane < cells) {
      const uint32_t nx = (qhi[0] >> shift) - (qlo[0] >> shift) + 1, ny = (qhi[1] >> shift) - (qlo[1] >> shift) + 1;
      const uint32_t c = lane, bx = (qlo[0] >> shift) + c % nx, by = (qlo[1] >> shift) + c / nx % ny,
                     bz = (qlo[2] >> shift) + c / nx / ny;
      const uint64_t klo = interleave(bx, by, bz) << (3 * shift);
      i0 = lower_bound_u64(skeys, nt, klo);
      i1 = lower_bound_u64(skeys, nt, klo + (1ULL << (3 * shift)));
    }
    uint64_t inc = (uint64_t)(i1 - i0);
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const uint64_t o = __shfl_up(inc, m, 64);
      if (lane >= m) inc += o;
    }
    cell_first[lane] = i0;
    cell_before[lane + 1] = inc;
    if (lane == 0) cell_before[0] = 0;
  }
  // Sample nodes, one per lane; r2 = -1 marks a lane without one.
  double px = 0, py = 0, pz = 0, pr2 = -1.0;
  {
    const int64_t s = sc >= 64 ? (2 * lane + 1) * sc / 128 : lane;
    if (s < sc) {
      px = xs[(s0 + s) * 3 + 0];
      py = xs[(s0 + s) * 3 + 1];
      pz = xs[(s0 + s) * 3 + 2];
      const double r = rad[s0 + s];
      pr2 = r * r;
    }
  }
  __syncthreads();

  int nh = 0;  // near targets gathered by this wave (uniform)
  auto flush = [&]() {
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(counter, (unsigned long long)nh);
    base = uniform64(base, 0);
    for (int i = lane; i < nh; i += 64)
      if ((int64_t)base + i < cap) out[base + i] = ((Key)e << tbits) | (Key)hits[i];
    nh = 0;
  };
  // Which of the queue entries in `mask` are within a node's radius, one node
  // per lane; four at a time, so that their LDS reads and ballots overlap.
  auto tested = [&](uint64_t mask, double x, double y, double z, double r2) -> uint64_t {
    uint64_t hit = 0;
    while (mask) {
      int j[4];
      double d2[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {  // fewer than four left: the last one again
        j[k] = mask ? __builtin_ctzll(mask) : j[k - 1];
        mask &= mask - 1;
      }
#pragma unroll
      for (int k = 0; k < 4; k++) d2[k] = dist2(x - queue[j[k]].x, y - queue[j[k]].y, z - queue[j[k]].z);
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (__builtin_amdgcn_ballot_w64(d2[k] < r2) != 0) hit |= 1ULL << j[k];
    }
    return hit;
  };
  // Tests queue entries [0, n) (n <= 64).
  auto batch = [&](int n) {
    const Cand q = queue[lane < n ? lane : 0];
    uint64_t reach = 0;
    for (int b = 0; b < nbox; b++) {
      const double dx = fmax(fmax(box[0][b] - q.x, q.x - box[3][b]), 0.0);
      const double dy = fmax(fmax(box[1][b] - q.y, q.y - box[4][b]), 0.0);
      const double dz = fmax(fmax(box[2][b] - q.z, q.z - box[5][b]), 0.0);
      if (dist2(dx, dy, dz) < box[6][b]) reach |= 1ULL << b;
    }
    if (lane >= n) reach = 0;
    uint64_t rem = __builtin_amdgcn_ballot_w64(reach != 0), nearm = 0;
    nearm = tested(rem, px, py, pz, pr2);
    rem &= ~nearm;
    if (sc > 64 && rem) {  // the samples were not all nodes
      for (int b = 0; b < nbox && rem; b++) {
        const uint64_t mine = __builtin_amdgcn_ballot_w64((reach >> b) & 1ULL) & rem;
        if (!mine) continue;
        const int64_t first = b * per_box, end = first + per_box < sc ? first + per_box : sc;
        uint64_t left = mine;
        for (int64_t s1 = first; s1 < end && left; s1 += 64) {
          const int64_t s = s1 + lane < end ? s1 + lane : end - 1;  // the last node again past the end
          const double r = rad[s0 + s];
          left &= ~tested(left, xs[(s0 + s) * 3 + 0], xs[(s0 + s) * 3 + 1], xs[(s0 + s) * 3 + 2], r * r);
        }
        nearm |= mine & ~left;
        rem &= ~(mine & ~left);
      }
    }
    if (nh + 64 > HITS) {
      wave_sync();
      flush();
    }
    if ((nearm >> lane) & 1ULL) hits[nh + lanes_below(nearm)] = q.t;
    nh += __builtin_popcountll(nearm);
    wave_sync();
  };

  const uint64_t total = cell_before[MAX_CELLS];
  int qn = 0;  // queued candidates (< 64 between batches)
  for (uint64_t base = (uint64_t)w * 64; base < total; base += NL_WG) {
    const uint64_t c = base + lane;
    bool inside = false;
    Cand v{0, 0, 0, 0};
    if (c < total) {
      int cell = 0;  // the cell of the c-th target: the last with cell_before <= c
#pragma unroll
      for (int step = MAX_CELLS / 2; step > 0; step >>= 1)
        if (cell_before[cell + step] <= c) cell += step;
      const int64_t i = cell_first[cell] + (int64_t)(c - cell_before[cell]);
      v.x = xsorted[i * 3 + 0];
      v.y = xsorted[i * 3 + 1];
      v.z = xsorted[i * 3 + 2];
      v.t = sidx[i];
      inside = v.x >= glo[0] && v.x <= ghi[0] && v.y >= glo[1] && v.y <= ghi[1] && v.z >= glo[2] && v.z <= ghi[2];
    }
    const uint64_t in = __builtin_amdgcn_ballot_w64(inside);
    if (inside) queue[qn + lanes_below(in)] = v;  // qn < 64, so the entry is below QCAP
    qn += __builtin_popcountll(in);
    wave_sync();
    if (qn >= 64) {
      batch(64);
      const Cand rest = queue[64 + (lane < qn - 64 ? lane : 0)];
      wave_sync();
      if (lane < qn - 64) queue[lane] = rest;
      qn -= 64;
      wave_sync();
    }
  }
  if (qn > 0) batch(qn);
  // What is left of the four waves' hits goes out together.
  if (lane == 0) nhits[w] = nh;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < NWAVE; k++) {
    before += k < w ? nhits[k] : 0;
    all += nhits[k];
  }
  if (threadIdx.x == 0 && all) out_base = atomicAdd(counter, (unsigned long long)all);
  __syncthreads();
  for (int i = lane; i < nh; i += 64) {
    const int64_t pos = (int64_t)out_base + before + i;
    if (pos < cap) out[pos] = ((Key)e << tbits) | (Key)hits[i];
  }
}

// near_elem_dsp[e] / near_elem_cnt[e]: the range of element e in the sorted
// keys (e << tbits | t), found by binary search (dsp = the pairs of the
// elements before e, also for an element without pairs).
template <class Key>
__global__ void __launch_bounds__(NL_WG)
k_nl_elem_ranges(int64_t nelem, const Key* __restrict__ keys, int64_t n, int tbits, int64_t* __restrict__ ecnt_out,
                 int64_t* __restrict__ edsp_out) {
  const int64_t e = (int64_t)blockIdx.x * NL_WG + threadIdx.x;
  if (e >= nelem) return;
  int64_t at[2];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if ((int64_t)(keys[mid] >> tbits) < e + k) lo = mid + 1;
      else hi = mid;
    }
    at[k] = lo;
  }
  ecnt_out[e] = at[1] - at[0];
  edsp_out[e] = at[0];
}

__global__ void __launch_bounds__(NL_WG) k_nl_zero(int64_t* __restrict__ a, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * NL_WG + threadIdx.x;
  if (i < n) a[i] = 0;
}

// The targets in the order of their keys.
__global__ void __launch_bounds__(NL_WG) k_nl_gather(const double* __restrict__ xt, int64_t nt,
                                                     const uint32_t* __restrict__ sidx, double* __restrict__ xsorted) {
  const int64_t i = (int64_t)blockIdx.x * NL_WG + threadIdx.x;
  if (i >= nt) return;
  const int64_t t = sidx[i];
#pragma unroll
  for (int k = 0; k < 3; k++) xsorted[i * 3 + k] = xt[t * 3 + k];
}

// Pair i (element-major): gather the target's coordinates / normal, and its
// key (the target) and value (the pair) for the target-major sort.
template <class Key>
__global__ void __launch_bounds__(NL_WG)
k_nl_unpack(int64_t n, const Key* __restrict__ pairs, int tbits, const double* __restrict__ xt,
            const double* __restrict__ xn, double* __restrict__ xtn, double* __restrict__ xntn,
            uint32_t* __restrict__ trg, uint32_t* __restrict__ pair) {
  const int64_t i = (int64_t)blockIdx.x * NL_WG + threadIdx.x;
  if (i >= n) return;
  const uint64_t t = (uint64_t)pairs[i] & ((1ULL << tbits) - 1);
#pragma unroll
  for (int k = 0; k < 3; k++) xtn[i * 3 + k] = xt[t * 3 + k];
  if (xn) {
#pragma unroll
    for (int k = 0; k < 3; k++) xntn[i * 3 + k] = xn[t * 3 + k];
  }
  trg[i] = (uint32_t)t;
  pair[i] = (uint32_t)i;
}

// Target-major position q: scatter_index[q] = the pair; near_trg_dsp of a
// target = its first position, near_trg_cnt the length of its run (its end
// minus its start, added to 0 by the run's two ends).
__global__ void __launch_bounds__(NL_WG)
k_nl_scatter(int64_t n, const uint32_t* __restrict__ trg, const uint32_t* __restrict__ pair,
             int64_t* __restrict__ scatter, unsigned long long* __restrict__ tcnt, int64_t* __restrict__ tdsp) {
  const int64_t q = (int64_t)blockIdx.x * NL_WG + threadIdx.x;
  if (q >= n) return;
  const uint32_t t = trg[q];
  scatter[q] = (int64_t)pair[q];
  if (q == 0 || trg[q - 1] != t) {
    tdsp[t] = q;
    if (q) atomicAdd(&tcnt[t], 0ULL - (unsigned long long)q);
  }
  if (q == n - 1 || trg[q + 1] != t) atomicAdd(&tcnt[t], (unsigned long long)(q + 1));
}

// Up to seven arrays of 8-byte words copied by one launch.
struct CopyList {
  const uint64_t* src[7];
  uint64_t* dst[7];
  int64_t end[7];  // words of the arrays up to and including this one
};
__global__ void __launch_bounds__(NL_WG) k_nl_copy(CopyList c) {
  for (int64_t i = (int64_t)blockIdx.x * NL_WG + threadIdx.x; i < c.end[6]; i += (int64_t)gridDim.x * NL_WG) {
    int64_t begin = 0;
#pragma unroll
    for (int k = 0; k < 7; k++) {
      if (i >= begin && i < c.end[k]) c.dst[k][i - begin] = c.src[k][i - begin];
      begin = c.end[k];
    }
  }
}

// Whether kernels on `device` may write p: memory of another GPU may not be mapped there.
bool on_device(const void* p, int device) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeDevice && a.device == device;
}

unsigned grid_of(int64_t n) { return (unsigned)((n + NL_WG - 1) / NL_WG); }

int bits_for(int64_t n) {
  int b = 0;
  while (b < 63 && ((int64_t)1 << b) < n) b++;
  return b;
}

// The buffer of a list of n pairs, its count and offset arrays zeroed.
int list_alloc(sctl_amd_near_list_s* L, int64_t n, hipStream_t s) {
  Carve c;
  const size_t xtn = c.take(sizeof(double) * 3 * n), xntn = c.take(L->has_normal ? sizeof(double) * 3 * n : 0),
               scatter = c.take(sizeof(int64_t) * n), ecnt = c.take(sizeof(int64_t) * L->nelem),
               edsp = c.take(sizeof(int64_t) * L->nelem), tcnt = c.take(sizeof(int64_t) * L->ntrg),
               tdsp = c.take(sizeof(int64_t) * L->ntrg);
  L->n_near = n;
  if (!c.bytes) return SCTL_AMD_SUCCESS;
  SCTL_TRY(block_take(c.bytes, s, &L->buf));
  L->d_xtn = reinterpret_cast<double*>(L->buf.p + xtn);
  if (L->has_normal) L->d_xntn = reinterpret_cast<double*>(L->buf.p + xntn);
  L->d_scatter = reinterpret_cast<int64_t*>(L->buf.p + scatter);
  L->d_ecnt = reinterpret_cast<int64_t*>(L->buf.p + ecnt);
  L->d_edsp = reinterpret_cast<int64_t*>(L->buf.p + edsp);
  L->d_tcnt = reinterpret_cast<int64_t*>(L->buf.p + tcnt);
  L->d_tdsp = reinterpret_cast<int64_t*>(L->buf.p + tdsp);
  const int64_t words = (int64_t)(c.bytes - ecnt) / 8;
  if (words > 0) {
    hipLaunchKernelGGL(k_nl_zero, dim3(grid_of(words)), dim3(NL_WG), 0, s, L->d_ecnt, words);
    SCTL_HIP_TRY(hipGetLastError());
  }
  return SCTL_AMD_SUCCESS;
}

// Scratch of the steps that follow once the number of pairs n is known.
template <class Key> struct PairScratch {
  size_t pairs, trg, pair, trg_s, pair_s, tmp, tmp1 = 0, tmp2 = 0, bytes;
  int tbits, bits;
};
template <class Key> int pair_scratch(int64_t nt, int64_t nelem, int64_t n, PairScratch<Key>* p) {
  p->tbits = bits_for(nt);
  p->bits = p->tbits + bits_for(nelem);
  SCTL_HIP_TRY(rocprim::radix_sort_keys(nullptr, p->tmp1, (Key*)nullptr, (Key*)nullptr, (size_t)n, 0,
                                        std::max(p->bits, 1), nullptr));
  SCTL_HIP_TRY(rocprim::radix_sort_pairs(nullptr, p->tmp2, (uint32_t*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                         (uint32_t*)nullptr, (size_t)n, 0, std::max(p->tbits, 1), nullptr));
  Carve c;
  p->pairs = c.take(sizeof(Key) * n);
  p->trg = c.take(4 * n);
  p->pair = c.take(4 * n);
  p->trg_s = c.take(4 * n);
  p->pair_s = c.take(4 * n);
  p->tmp = c.take(std::max(p->tmp1, p->tmp2));
  p->bytes = c.bytes;
  return SCTL_AMD_SUCCESS;
}

// The build on device arrays of at least one target, node and element.  One
// scratch allocation holds the targets' sort, the pairs found and the steps that
// follow, as long as the list has at most ROOM and USUAL pairs per target; their
// shares are bounded (ROOM_BYTES, at least LEAST pairs per target, and
// USUAL_BYTES).  !reserve (the device's memory did not suffice): no such shares;
// the first pass over the elements only counts, and what is needed is allocated
// by size.  The later steps reuse the memory of the targets' sort.
template <class Key>
int build_pairs(sctl_amd_near_list_s* L, const double* xt, int64_t nt, const double* xn, const double* xs, int64_t ns,
                const double* rad, int64_t nelem, const int64_t* ecnt, const int64_t* edsp, bool reserve,
                hipStream_t s) {
  constexpr double ROOM = 24, LEAST = 4, USUAL = 8;  // pairs per target
  constexpr int64_t ROOM_BYTES = (int64_t)256 << 20, USUAL_BYTES = (int64_t)256 << 20;
  auto at_most = [&](double per_target) {
    return (int64_t)std::min<double>((double)nt * (double)nelem, std::max(per_target * (double)nt, 65536.0));
  };
  size_t sort_bytes = 0;
  SCTL_HIP_TRY(rocprim::radix_sort_pairs(nullptr, sort_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                         (uint32_t*)nullptr, (uint32_t*)nullptr, (size_t)nt, 0, 63, s));
  // The sort of the targets, then their sorted coordinates in place of its inputs.
  Carve sort;
  const size_t o_keys_in = sort.take(8 * nt), o_idx_in = sort.take(4 * nt), o_tmp = sort.take(sort_bytes);
  const size_t sort_region = std::max<size_t>(sort.bytes, 24 * nt);
  int64_t cap = std::min(at_most(ROOM), std::max<int64_t>(at_most(LEAST), ROOM_BYTES / (int64_t)sizeof(Key))), n = 0;
  int64_t usual = std::min<int64_t>(at_most(USUAL), USUAL_BYTES / (2 * sizeof(Key) + 24));
  if (!reserve) cap = usual = 1;
  PairScratch<Key> ps;
  SCTL_TRY(pair_scratch(nt, nelem, usual, &ps));
  Carve c;
  const size_t o_cube = c.take(sizeof(double) * 6), o_part = c.take(bounding_box_bytes(nt, ns)),
               o_counter = c.take(sizeof(int64_t)), o_found = c.take(sizeof(Key) * cap),
               o_keys = c.take(8 * nt),  // from here on the later steps'
               o_idx = c.take(4 * nt), o_sort = c.take(sort_region);
  const size_t later_bytes = std::max(ps.bytes, c.bytes - o_keys);
  BlockScratch work, more, later;
  SCTL_TRY(work.alloc(o_keys + later_bytes, s));
  char *w = work.b.p, *a = w + o_sort;
  double *cube = reinterpret_cast<double*>(w + o_cube), *xsorted = reinterpret_cast<double*>(a);
  uint64_t *keys_in = reinterpret_cast<uint64_t*>(a + o_keys_in), *keys = reinterpret_cast<uint64_t*>(w + o_keys);
  uint32_t *idx_in = reinterpret_cast<uint32_t*>(a + o_idx_in), *idx = reinterpret_cast<uint32_t*>(w + o_idx);
  int64_t* counter = reinterpret_cast<int64_t*>(w + o_counter);
  Key* found = reinterpret_cast<Key*>(w + o_found);
  SCTL_TRY(bounding_box(xt, nt, xs, ns, cube, w + o_part, s));
  hipLaunchKernelGGL(k_nl_cube, dim3(1), dim3(64), 0, s, cube, cube);
  hipLaunchKernelGGL(k_nl_keys, dim3(grid_of(nt)), dim3(NL_WG), 0, s, xt, nt, cube, keys_in, idx_in);
  SCTL_HIP_TRY(hipGetLastError());
  SCTL_HIP_TRY(rocprim::radix_sort_pairs(a + o_tmp, sort_bytes, keys_in, keys, idx_in, idx, (size_t)nt, 0, 63, s));
  hipLaunchKernelGGL(k_nl_gather, dim3(grid_of(nt)), dim3(NL_WG), 0, s, xt, nt, idx, xsorted);
  SCTL_HIP_TRY(hipGetLastError());
  for (int pass = 0; pass < 2; pass++) {
    hipLaunchKernelGGL(k_nl_zero, dim3(1), dim3(NL_WG), 0, s, counter, (int64_t)1);
    hipLaunchKernelGGL((k_nl_elements<Key>), dim3((unsigned)nelem), dim3(NL_WG), 0, s, ecnt, edsp, ns, xs, rad, nt,
                       xsorted, keys, idx, cube, ps.tbits, reinterpret_cast<unsigned long long*>(counter), cap, found);
    SCTL_HIP_TRY(hipGetLastError());
    SCTL_HIP_TRY(hipMemcpyAsync(&n, counter, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    SCTL_HIP_TRY(hipStreamSynchronize(s));
    if (n <= cap) break;
    SCTL_CHECK_ARG(pass == 0, "near-pair count exceeds its bound (internal error)");
    cap = n;
    SCTL_TRY(more.alloc(sizeof(Key) * cap, s));
    found = reinterpret_cast<Key*>(more.b.p);
  }
  SCTL_CHECK_ARG(n < ((int64_t)1 << 32), "more than 2^32-1 near pairs");
  SCTL_TRY(list_alloc(L, n, s));
  if (n == 0) {
    SCTL_HIP_TRY(hipStreamSynchronize(s));
    return SCTL_AMD_SUCCESS;
  }
  char* l = w + o_keys;
  SCTL_TRY(pair_scratch(nt, nelem, n, &ps));
  if (ps.bytes > later_bytes) {  // not n > usual: the sorts' shares need not grow with n
    SCTL_TRY(later.alloc(ps.bytes, s));
    l = later.b.p;
  }
  Key* pairs = reinterpret_cast<Key*>(l + ps.pairs);
  uint32_t *trg = reinterpret_cast<uint32_t*>(l + ps.trg), *pair = reinterpret_cast<uint32_t*>(l + ps.pair);
  uint32_t *trg_s = reinterpret_cast<uint32_t*>(l + ps.trg_s), *pair_s = reinterpret_cast<uint32_t*>(l + ps.pair_s);
  SCTL_HIP_TRY(rocprim::radix_sort_keys(l + ps.tmp, ps.tmp1, found, pairs, (size_t)n, 0, std::max(ps.bits, 1), s));
  hipLaunchKernelGGL((k_nl_elem_ranges<Key>), dim3(grid_of(nelem)), dim3(NL_WG), 0, s, nelem, pairs, n, ps.tbits,
                     L->d_ecnt, L->d_edsp);
  SCTL_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL((k_nl_unpack<Key>), dim3(grid_of(n)), dim3(NL_WG), 0, s, n, pairs, ps.tbits, xt, xn, L->d_xtn,
                     L->d_xntn, trg, pair);
  SCTL_HIP_TRY(hipGetLastError());
  SCTL_HIP_TRY(rocprim::radix_sort_pairs(l + ps.tmp, ps.tmp2, trg, trg_s, pair, pair_s, (size_t)n, 0,
                                         std::max(ps.tbits, 1), s));
  hipLaunchKernelGGL(k_nl_scatter, dim3(grid_of(n)), dim3(NL_WG), 0, s, n, trg_s, pair_s, L->d_scatter,
                     reinterpret_cast<unsigned long long*>(L->d_tcnt), L->d_tdsp);
  SCTL_HIP_TRY(hipGetLastError());
  SCTL_HIP_TRY(hipStreamSynchronize(s));
  return SCTL_AMD_SUCCESS;
}

int build_list(sctl_amd_near_list_s* L, const double* xt, int64_t nt, const double* xn, const double* xs, int64_t ns,
               const double* rad, int64_t nelem, const int64_t* ecnt, const int64_t* edsp, hipStream_t s) {
  if (nt == 0 || ns == 0 || nelem == 0) {
    SCTL_TRY(list_alloc(L, 0, s));
    SCTL_HIP_TRY(hipStreamSynchronize(s));
    return SCTL_AMD_SUCCESS;
  }
  auto build = bits_for(nt) < 32 && bits_for(nt) + bits_for(nelem) <= 32 ? build_pairs<uint32_t> : build_pairs<uint64_t>;
  const int rc = build(L, xt, nt, xn, xs, ns, rad, nelem, ecnt, edsp, true, s);
  if (rc != SCTL_AMD_ERROR_OUT_OF_MEMORY) return rc;
  block_drop(L->buf);  // hipFree waits for what is under way
  L->buf = Block();
  blocks_release();
  return build(L, xt, nt, xn, xs, ns, rad, nelem, ecnt, edsp, false, s);
}

}  // namespace
}  // namespace sctl_amd

using namespace sctl_amd;

extern "C" {

int sctl_amd_near_list_build(sctl_amd_near_list* list, const double* Xtrg, int64_t ntrg, const double* Xn_trg,
                             const double* Xsrc, int64_t nsrc, const double* src_radius, int64_t nelem,
                             const int64_t* elem_nds_cnt, const int64_t* elem_nds_dsp, uint32_t flags,
                             void* stream) {
  SCTL_CHECK_ARG(list, "list is NULL");
  *list = nullptr;
  SCTL_CHECK_ARG((flags & ~SCTL_AMD_HOST_PTRS) == 0, "unknown flag bits");
  SCTL_CHECK_ARG(ntrg >= 0 && nsrc >= 0 && nelem >= 0, "negative size");
  SCTL_CHECK_ARG(ntrg < ((int64_t)1 << 32) && nelem < ((int64_t)1 << 31), "too many targets or elements");
  SCTL_CHECK_ARG(ntrg == 0 || Xtrg, "Xtrg is NULL");
  SCTL_CHECK_ARG(nsrc == 0 || (Xsrc && src_radius), "Xsrc or src_radius is NULL");
  SCTL_CHECK_ARG(nelem == 0 || (elem_nds_cnt && elem_nds_dsp), "NULL element array");
  const bool host = flags & SCTL_AMD_HOST_PTRS;
  if (host) {
    for (int64_t e = 0; e < nelem; e++)
      SCTL_CHECK_ARG(elem_nds_cnt[e] >= 0 && elem_nds_dsp[e] >= 0 && elem_nds_dsp[e] + elem_nds_cnt[e] <= nsrc,
                     "element node range outside the sources (element " + std::to_string(e) + ")");
  }
  DeviceInfo dev;
  SCTL_TRY(device_info(&dev));
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : hipStreamPerThread;
  auto* L = new sctl_amd_near_list_s();
  L->device = dev.device;
  L->ntrg = ntrg;
  L->nelem = nelem;
  L->has_normal = Xn_trg != nullptr;
  int rc = SCTL_AMD_SUCCESS;
  if (!host) {
    rc = build_list(L, Xtrg, ntrg, Xn_trg, Xsrc, nsrc, src_radius, nelem, elem_nds_cnt, elem_nds_dsp, s);
  } else {
    Scratch a, b, c, d, e, f;
    auto up = [&](Scratch& buf, const void* src, size_t bytes) -> int {
      if (!src || !bytes) return SCTL_AMD_SUCCESS;
      SCTL_TRY(buf.alloc(bytes, s));
      SCTL_HIP_TRY(hipMemcpyAsync(buf.as<void>(), src, bytes, hipMemcpyHostToDevice, s));
      return SCTL_AMD_SUCCESS;
    };
    if (!rc) rc = up(a, Xtrg, sizeof(double) * 3 * ntrg);
    if (!rc) rc = up(b, Xn_trg, sizeof(double) * 3 * ntrg);
    if (!rc) rc = up(c, Xsrc, sizeof(double) * 3 * nsrc);
    if (!rc) rc = up(d, src_radius, sizeof(double) * nsrc);
    if (!rc) rc = up(e, elem_nds_cnt, sizeof(int64_t) * nelem);
    if (!rc) rc = up(f, elem_nds_dsp, sizeof(int64_t) * nelem);
    if (!rc)
      rc = build_list(L, a.as<double>(), ntrg, Xn_trg ? b.as<double>() : nullptr, c.as<double>(), nsrc,
                      d.as<double>(), nelem, e.as<int64_t>(), f.as<int64_t>(), s);
    if (!rc && hipStreamSynchronize(s) != hipSuccess) rc = SCTL_AMD_ERROR_HIP;
  }
  if (!rc && L->buf.used && hipEventRecord(L->buf.used, s) != hipSuccess) {
    set_error("hipEventRecord failed after a near-list build");
    rc = SCTL_AMD_ERROR_HIP;
  }
  if (rc) {
    L->loose = true;
    delete L;
    return rc;
  }
  *list = L;
  return SCTL_AMD_SUCCESS;
}

int sctl_amd_near_list_size(sctl_amd_near_list list, int64_t* n_near) {
  SCTL_CHECK_ARG(list && n_near, "NULL argument");
  *n_near = list->n_near;
  return SCTL_AMD_SUCCESS;
}

int sctl_amd_near_list_get(sctl_amd_near_list list, double* Xtrg_near, double* Xn_trg_near, int64_t* near_elem_cnt,
                           int64_t* near_elem_dsp, int64_t* near_scatter_index, int64_t* near_trg_cnt,
                           int64_t* near_trg_dsp, uint32_t flags, void* stream) {
  SCTL_CHECK_ARG(list, "list is NULL");
  SCTL_CHECK_ARG((flags & ~SCTL_AMD_HOST_PTRS) == 0, "unknown flag bits");
  SCTL_CHECK_ARG(!Xn_trg_near || list->has_normal || list->n_near == 0, "the list was built without target normals");
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : hipStreamPerThread;
  const int64_t n = list->n_near, ne = list->nelem, nt = list->ntrg;
  const struct {
    void* dst;
    const void* src;
    int64_t words;
  } a[7] = {{Xtrg_near, list->d_xtn, 3 * n},          {Xn_trg_near, list->d_xntn, 3 * n},
            {near_elem_cnt, list->d_ecnt, ne},        {near_elem_dsp, list->d_edsp, ne},
            {near_scatter_index, list->d_scatter, n}, {near_trg_cnt, list->d_tcnt, nt},
            {near_trg_dsp, list->d_tdsp, nt}};
  if (flags & SCTL_AMD_HOST_PTRS) {  // done on return: nothing to order
    hipError_t e = hipSuccess;
    for (const auto& x : a)
      if (e == hipSuccess && x.dst && x.src && x.words)
        e = hipMemcpyAsync(x.dst, x.src, 8 * (size_t)x.words, hipMemcpyDeviceToHost, s);
    const hipError_t done = hipStreamSynchronize(s);  // also after a failure: copies may be in flight
    if (done != hipSuccess) {
      std::lock_guard<std::mutex> lock(list->read);
      list->loose = true;
    }
    SCTL_HIP_TRY(e);
    SCTL_HIP_TRY(done);
    return SCTL_AMD_SUCCESS;
  }
  // One launch copies all that lies on the list's GPU; outputs elsewhere (another
  // GPU's memory) take the runtime's copies.
  int cur = -1;
  (void)hipGetDevice(&cur);
  bool here = cur == list->device;
  CopyList c;
  int64_t words = 0;
  for (int k = 0; k < 7; k++) {
    if (here && a[k].dst && a[k].src && a[k].words) here = on_device(a[k].dst, list->device);
    words += a[k].dst && a[k].src ? a[k].words : 0;
    c.src[k] = static_cast<const uint64_t*>(a[k].src);
    c.dst[k] = static_cast<uint64_t*>(a[k].dst);
    c.end[k] = words;
  }
  if (!words) return SCTL_AMD_SUCCESS;
  // Reads of the results follow each other whatever their streams and threads, so
  // that the list's event, recorded after the latest, is after all of them: a
  // list destroyed then gives its buffer to the next build behind that event.  A
  // captured read runs when its graph does, as often as that is launched, so the
  // buffer of such a list is freed and not given on (destroy waits for launches
  // under way; the graph needs the list for others, as any graph its buffers).
  std::lock_guard<std::mutex> lock(list->read);
  const bool capturing = stream_capturing(s);
  if (!capturing) SCTL_HIP_TRY(hipStreamWaitEvent(s, list->buf.used, 0));
  const bool loose = list->loose;
  list->loose = true;
  if (here) {
    hipLaunchKernelGGL(k_nl_copy, dim3(std::min<unsigned>(grid_of(words), 4096)), dim3(NL_WG), 0, s, c);
    SCTL_HIP_TRY(hipGetLastError());
  } else {
    for (const auto& x : a)
      if (x.dst && x.src && x.words)
        SCTL_HIP_TRY(hipMemcpyAsync(x.dst, x.src, 8 * (size_t)x.words, hipMemcpyDeviceToDevice, s));
  }
  if (capturing) return SCTL_AMD_SUCCESS;
  SCTL_HIP_TRY(hipEventRecord(list->buf.used, s));
  list->loose = loose;
  return SCTL_AMD_SUCCESS;
}

int sctl_amd_near_list_destroy(sctl_amd_near_list list) {
  delete list;
  return SCTL_AMD_SUCCESS;
}

}  // extern "C"
