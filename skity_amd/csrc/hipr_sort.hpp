// hipr_sort.hpp -- per-job edge ordering for the walk.
//
// SortEdges (src/render/sw/sw_raster.cc:679-704) orders edges by
// (upper_y, x, dx).  The walk only needs them grouped by upper_y in emission
// order (it orders each group of newly active edges by (x, dx, position)
// itself), so the key is (upper_y, emission index): a bitonic sort of 64-bit
// keys in LDS, followed by a gather of the records into a work copy that the
// walk may mutate (quad edges advance their forward differences in place).
#ifndef SKITY_HIP_SORT_HPP_
#define SKITY_HIP_SORT_HPP_

#include "hipr_common.hpp"

namespace hipr {

constexpr int kSortThreads = 256;
constexpr int kSortLdsKeys = 8192;  // 64 KiB of keys

// A job of at most this many edges, over rows that leave the histogram of its
// keys' LDS one row per bin, is sorted by one wave in 8 KiB of LDS.  A block of
// the general form holds 64 KiB, so that two fit a compute unit, and its four
// waves idle on such a job: the page of 16,900 glyphs (20 to 60 edges each)
// took 0.315 ms by the general form and takes 0.037; curves + strokes, 4,096
// paths of 900 edges on average, 1.0 and 0.60 ms.  Longer jobs have work for
// four waves in every stage, and their keys would not leave the LDS to others.
constexpr int kSortSmallKeys = 1024;
constexpr int kSortSmallRows = kSortSmallKeys * 2 - 2;

// Pixel rows of a job's bounds, the same on the host and the device for any
// bounds (none, NaN and out of range included).
__host__ __device__ inline int SortRows(const JobGeo& g) {
  if (!(g.t < g.b)) return 1;
  const float limit = 8388608.f;
  const int top = (int)floorf(g.t > -limit ? (g.t < limit ? g.t : limit) : -limit);
  const int bottom = (int)ceilf(g.b > -limit ? (g.b < limit ? g.b : limit) : -limit);
  return bottom > top ? bottom - top : 1;
}
__host__ __device__ inline bool SortIsSmall(const JobGeo& g) {
  return g.edges <= kSortSmallKeys && SortRows(g) <= kSortSmallRows;
}

__device__ __forceinline__ uint64_t EdgeKey(const EdgeRec& e, int idx) {
  // upper_y is a 16.16 multiple of 1/4; bias to make it unsigned.
  return ((uint64_t)((uint32_t)e.upper_y ^ 0x80000000u) << 32) | (uint32_t)idx;
}

// keys: per-job scratch of next_pow2(n) entries (used when n exceeds LDS).
// active_bound (may be null) receives an upper bound of the job's active
// edge list: the largest number of edges whose row range (upper_y to lower_y,
// or to the last step's y for a quad edge) meets one bin of rows (a bin is one pixel row when the job spans at most
// 16384 rows).  The walk keeps exactly the edges with upper_y <= y < lower_y
// active, so this bounds every sub-step's list.
//
// Two instantiations share the jobs by SortIsSmall: one wave with
// kSortSmallKeys, four waves with kSortLdsKeys (a block whose job is the
// other's ends at once).
template <int kThreads, int kKeys>
__global__ void __launch_bounds__(kThreads)
    SortGatherKernel(const int32_t* __restrict__ job_list, int n_list,
                     const JobGeo* __restrict__ geo, const int64_t* __restrict__ edge_base,
                     const EdgeRec* __restrict__ edges, EdgeRec* __restrict__ wedges,
                     uint64_t* __restrict__ gkeys, int32_t* __restrict__ active_bound) {
  constexpr bool kSmall = kThreads == kWave;
  __shared__ uint64_t skeys[kKeys];
  int li = blockIdx.x;
  if (li >= n_list) return;
  int j = job_list[li];
  const JobGeo g = geo[j];
  const int n = g.edges;
  if (SortIsSmall(g) != kSmall) return;
  if (n <= 0) {
    if (active_bound && threadIdx.x == 0) active_bound[j] = 0;
    return;
  }
  int64_t base = edge_base[j];
  const EdgeRec* src = edges + base;
  EdgeRec* dst = wedges + base;
  auto sync = [] {
    if (kSmall) {
      WaveSync();
    } else {
      __syncthreads();
    }
  };
  if (kSmall && n <= kWave) {
    // one edge per lane: its place is the number of smaller keys
    const int lane = threadIdx.x;
    uint64_t key = ~0ull;
    if (lane < n) key = EdgeKey(src[lane], lane);
    int place = 0;
    for (int i = 0; i < n; i++) {
      const uint64_t other =
          ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(key >> 32), i) << 32) |
          (uint32_t)i;
      place += other < key;
    }
    if (lane < n) dst[place] = src[lane];
  } else {
    int np2 = 1;
    while (np2 < n) np2 <<= 1;
    bool in_lds = kSmall || np2 <= kKeys;
    uint64_t* keys = in_lds ? skeys : gkeys + base * 2;  // scratch sized 2n >= np2
    for (int i = threadIdx.x; i < np2; i += kThreads) {
      keys[i] = i < n ? EdgeKey(src[i], i) : ~0ull;
    }
    sync();
    for (int k = 2; k <= np2; k <<= 1) {
      for (int jj = k >> 1; jj > 0; jj >>= 1) {
        // pair p of the stage: elements i and i + jj
        for (int p = threadIdx.x; p < np2 / 2; p += kThreads) {
          const int i = ((p & ~(jj - 1)) << 1) | (p & (jj - 1));
          uint64_t a = keys[i], b = keys[i + jj];
          bool up = (i & k) == 0;
          if ((a > b) == up) {
            keys[i] = b;
            keys[i + jj] = a;
          }
        }
        if (!in_lds) __threadfence_block();
        sync();
      }
    }
    for (int i = threadIdx.x; i < n; i += kThreads) {
      int idx = (int)(uint32_t)(keys[i] & 0xFFFFFFFFu);
      dst[i] = src[idx];
    }
  }
  if (!active_bound) return;
  // ---- row-overlap bound (LDS reused as a histogram of row bins) ----
  sync();
  constexpr int kBins = kKeys * 2;
  int32_t* hist = (int32_t*)skeys;
  const int top = (int)floorf(g.t);
  const int H = SortRows(g);
  const int bin = kSmall ? 1 : (H + kBins - 3) / (kBins - 2);  // rows per bin, >= 1
  const int nb = H / bin + 2;                                  // <= kBins
  for (int i = threadIdx.x; i < nb; i += kThreads) hist[i] = 0;
  sync();
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const EdgeRec& e = src[i];
    // a quad edge stays in the list until its last step (q_last_y)
    Fixed last = EdgeIsQuad(e.packed) && e.q_last_y > e.lower_y ? e.q_last_y : e.lower_y;
    int r0 = (e.upper_y >> 16) - top, r1 = ((last - 1) >> 16) - top;
    r0 = r0 < 0 ? 0 : (r0 >= H ? H - 1 : r0);
    r1 = r1 < r0 ? r0 : (r1 >= H ? H - 1 : r1);
    atomicAdd(&hist[kSmall ? r0 : r0 / bin], 1);
    atomicAdd(&hist[kSmall ? r1 + 1 : r1 / bin + 1], -1);
  }
  sync();
  // chunked scan: each thread owns a contiguous chunk of bins, the chunks are
  // summed by wave scans
  __shared__ int32_t part[2 * kThreads / kWave];
  const int wave = threadIdx.x / kWave;
  const int chunk = (nb + kThreads - 1) / kThreads;
  const int c0 = threadIdx.x * chunk, c1 = c0 + chunk < nb ? c0 + chunk : nb;
  int sum = 0;
  for (int i = c0; i < c1; i++) sum += hist[i];
  const int upto = WaveInclusiveSum(sum);
  int run = upto - sum;
  if (!kSmall) {
    if (Lane() == kWave - 1) part[wave] = upto;
    sync();
    for (int w = 0; w < wave; w++) run += part[w];
  }
  int mx = 0;
  for (int i = c0; i < c1; i++) {
    run += hist[i];
    mx = run > mx ? run : mx;
  }
  mx = WaveMax(mx);
  if (!kSmall) {
    if (Lane() == 0) part[kThreads / kWave + wave] = mx;
    sync();
    for (int w = 0; w < kThreads / kWave; w++) mx = max(mx, part[kThreads / kWave + w]);
  }
  if (threadIdx.x == 0) active_bound[j] = mx;
}

}  // namespace hipr

#endif  // SKITY_HIP_SORT_HPP_
