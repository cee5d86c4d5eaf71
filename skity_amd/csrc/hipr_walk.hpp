// hipr_walk.hpp -- stage (b): the analytic-AA scanline walk of one path per
// wavefront, producing 16x16 coverage tiles.
//
// This is WalkEdges (src/render/sw/sw_raster.cc:546-677) with
// insert_new_edges / backward_insert_edge_based_on_x / check_intersection
// (sw_raster.cc:159-247) re-expressed for a 64-lane wave.  The active edge
// list lives in registers (element p in lane p % 64, slot p / 64) and every
// sequential list operation of the reference is replaced by the parallel
// operation with the same result, and rows without an event are taken up to 16
// at a time:
//   * winding sums and interval roles: wave prefix sums in list order;
//   * the left edge of an interval / the previous right edge: max-scans;
//   * the per-edge x re-insertion after a step keeps the survivors stably
//     sorted by x (backward_insert_edge_based_on_x moves an edge behind the
//     processed edges with larger x), and check_intersection compares each
//     survivor with its predecessor among the already processed survivors;
//   * insert_new_edges places the first new edge after the last active edge
//     with x <= its x and every later one before the first following active
//     edge with x >= its x; new edges arrive sorted by (upper_y, x, dx, index)
//     (SortEdges, sw_raster.cc:679-704, with emission order breaking ties).
// Coverage of a pixel row is collected as LDS deltas (hipr_blit.hpp) and, when
// the row is complete, resolved into at most two covers per pixel (the
// directly emitted span first, then the accumulated one), which are written
// into the plane(s) of the 16x16 tile holding the pixel.  A tile whose every
// pixel is covered by 255 gets no plane, only a map entry.
#ifndef SKITY_HIP_WALK_HPP_
#define SKITY_HIP_WALK_HPP_

#include "hipr_blit.hpp"
#include "hipr_common.hpp"

namespace hipr {

constexpr int kTilePlaneBytes = kTile * kTile;
// Tile slot of an allocation that found no plane (capacity and pool spent).
constexpr int32_t kNoPlane = 0x7FFFFFFF;
// Planes the bands of a job take at a time (a multiple of three).
constexpr int kPlaneChunk = 48;
// Map entries: a plane number, or no coverage, or a tile whose every pixel
// has the first cover 255, which needs no plane.
constexpr int32_t kNoTile = -1;
constexpr int32_t kSolidTile = -2;

// Walk modes: count the tile planes, write them, or only follow the step
// schedule (no coverage) to record the row-band snapshots.
enum WalkMode : int { kWalkCount = 0, kWalkWrite = 1, kWalkSchedule = 2 };

// Row bands.  A path taller than `band_rows` is walked by several wavefronts
// at once, each over a range of rows.  A sequential pass (count or schedule)
// records the complete walk state at the start of every band after the
// first: the first loop iteration that begins on a pixel row that is a
// multiple of 16 (a tile row boundary) at or below the band's nominal start
// row.  Restarted from that state, the walk of a band is the same computation
// as the sequential walk over those rows, and every tile row belongs to one
// band.
// Widest walk: 64 slots x 64 lanes, an active list of 4096 edges.
constexpr int kMaxSlots = 64;
constexpr int kBandBits = 5;  // work items are job << kBandBits | band
constexpr int kMaxBands = 1 << kBandBits;
struct SnapHeader {
  int32_t y, nny, pp, n;  // y = kMaxS32: the band has no rows
  int32_t pad[12];
};
static_assert(sizeof(SnapHeader) == 64, "snapshot header is 64 bytes");
// header, then X, DX, DY, LY, M [cap] and the quad edge state [cap]
__host__ __device__ inline int64_t SnapStride(int cap) {
  return (int64_t)sizeof(SnapHeader) + (int64_t)cap * (5 * 4 + (int64_t)sizeof(EdgeRec));
}

struct WalkParams {
  const Job* jobs;
  const int32_t* walk_list;  // work items: job << kBandBits | band
  int32_t n_walk;
  const JobGeo* geo;
  const int64_t* edge_base;
  const EdgeRec* wedges;    // per job, sorted by (upper_y, index); read only
  EdgeRec* qstate;          // quad edge state: nE records per job and band
  const int64_t* q_base;    // per job: first qstate record of band 0
  uint8_t* snaps;           // band snapshots
  const int64_t* snap_base; // per job: byte offset of band 1's snapshot
  const int32_t* band_count;  // per job: row bands (1 = one sequential walk)
  const Canvas* canvases;
  const int64_t* plane_base;  // per job: first plane of its estimated range
  const int32_t* plane_cap;
  uint8_t* planes;
  // Shared overflow pool (estimate modes): a job's planes beyond its
  // capacity come from planes [pool_base, pool_base + pool_cap), taken with
  // an atomic counter (starts at 0).  Maps hold absolute plane numbers.
  int32_t* pool_ctr;
  int32_t pool_base, pool_cap;
  const int64_t* map_base;
  int32_t* map0;
  int32_t* map1;
  JobCov* cov;
  int32_t lds_width;        // widest row in pixels
  int32_t row_ints;         // row delta capacity (multiple of 16)
  int32_t* queue;           // persistent form: item counter (starts at 0), else null
};

// Job pixel bounds as RastePath computes them (sw_raster.cc:741-754).
// Device-space coordinates beyond +-kCoordLimit are refused before any walk
// (the reference's float -> 26.6 conversion overflows there); the clamp keeps
// every width and height of a refused job within int32.
constexpr float kCoordLimit = 8388608.f;  // 2^23 px
// Source coordinates are refused far beyond it (a canvas matrix could bring
// them back into range, so the device-space check is the one that counts).
constexpr float kSourceCoordLimit = 1073741824.f;  // 2^30
struct PixBounds {
  int l, t, r, b;
  bool empty;
};
__host__ __device__ inline float ClampCoord(float v) {
  return v < -kCoordLimit ? -kCoordLimit : (v > kCoordLimit ? kCoordLimit : v);
}
__host__ __device__ inline PixBounds JobPixBounds(const JobGeo& g) {
  PixBounds pb;
  bool ok = g.l < g.r && g.t < g.b;
  float l = ok ? floorf(ClampCoord(g.l)) : 0.f, t = ok ? floorf(ClampCoord(g.t)) : 0.f;
  float r = ok ? ceilf(ClampCoord(g.r)) : 0.f, b = ok ? ceilf(ClampCoord(g.b)) : 0.f;
  pb.empty = !(l < r && t < b);
  pb.l = (int)l;
  pb.t = (int)t;
  pb.r = (int)r;
  pb.b = (int)b;
  return pb;
}
// Scan bounds of a job (sw_raster.cc:741-754): the quad path's bounds
// intersected with the job's clip bounds (Rect::Intersect, rect.cc:160-172:
// empty unless l < r and t < b), floored / ceiled.  Without a clip they are
// the path's own pixel bounds.  The walk starts at the path's top row
// (JobPixBounds) and clips everything else to these.
__host__ __device__ inline PixBounds JobScanBounds(const JobGeo& g) {
  float l = g.l > g.cl ? g.l : g.cl, r = g.r < g.cr ? g.r : g.cr;
  float t = g.t > g.ct ? g.t : g.ct, b = g.b < g.cb ? g.b : g.cb;
  if (!(l < r && t < b)) {
    PixBounds e{0, 0, 0, 0, true};
    return e;
  }
  JobGeo h = g;
  h.l = l;
  h.t = t;
  h.r = r;
  h.b = b;
  return JobPixBounds(h);
}
// Visible tile range of a job on its canvas (inclusive); ntc = 0 if none.
struct TileRange {
  int tc0, tr0, ntc, ntr;
};
__host__ __device__ inline TileRange JobTiles(const PixBounds& pb, int cw, int ch) {
  TileRange tr{0, 0, 0, 0};
  if (pb.empty) return tr;
  int x0 = pb.l > 0 ? pb.l : 0, x1 = pb.r < cw ? pb.r : cw;
  int y0 = pb.t > 0 ? pb.t : 0, y1 = pb.b < ch ? pb.b : ch;
  if (x0 >= x1 || y0 >= y1) return tr;
  tr.tc0 = x0 >> 4;
  tr.tr0 = y0 >> 4;
  tr.ntc = ((x1 - 1) >> 4) - tr.tc0 + 1;
  tr.ntr = ((y1 - 1) >> 4) - tr.tr0 + 1;
  return tr;
}

// Number of row bands of a job and the nominal first row of band b >= 1,
// rounded up to a tile row.
__host__ __device__ inline int BandCount(const PixBounds& pb, int band_rows) {
  if (pb.empty || band_rows <= 0) return 1;
  int nb = (pb.b - pb.t) / band_rows;
  return nb < 1 ? 1 : (nb > kMaxBands ? kMaxBands : nb);
}
__host__ __device__ inline int BandStartRow(const PixBounds& pb, int nb, int b) {
  int v = pb.t + (int)((int64_t)(pb.b - pb.t) * b / nb);
  return (v + kTile - 1) & ~(kTile - 1);
}

// meta word of an active edge: bit 0 winding < 0, bit 1 quad, bit 2 the quad's
// state has moved on (it lives in qstate; before that it is the sorted edge
// record's), bits 3.. index
__device__ __forceinline__ bool MetaQuad(int m) { return (m & 2) != 0; }
__device__ __forceinline__ bool MetaMoved(int m) { return (m & 4) != 0; }
__device__ __forceinline__ int MetaIndex(int m) { return (int)((uint32_t)m >> 3); }
__device__ __forceinline__ int MakeMeta(int winding, bool quad, bool moved, int idx) {
  return (winding < 0 ? 1 : 0) | (quad ? 2 : 0) | (moved ? 4 : 0) | (idx << 3);
}

struct WalkLds {
  int32_t* d;      // packed row deltas (RowSink), from the first tile column's left edge
  uint32_t* touch; // a bit per tile column: the row has deltas there
  int32_t* slot0;  // per tile column of the current band
  int32_t* slot1;
  int32_t* rows;   // per tile column: rows written, plane 0 (bits 0-15), plane 1 (16-31)
  int32_t* full;   // per tile column 16 bits: rows whose 16 pixels all have the cover 255
  int32_t* sX;     // permutation scratch (CAP entries each)
  int32_t* sDX;
  int32_t* sDY;
  int32_t* sLY;
  int32_t* sM;
  // left and right edges of the step's intervals; they share the permutation
  // scratch, which is free while the intervals are drawn
  int4* iL;        // {x, step, dy, -}; CAP / 2 entries each
  int4* iR;        // {x, step, dy, kNext*}
  int2* iN;        // the next edge's {x, dx}
  BlitScratch blit;
  // row flush (in the blit scratch): the touched tile columns of a group of
  // 64, and each one's value at its last pixel
  int32_t* list;
  int32_t* vend;
};
// LDS words of a K-slot walk whose rows are up to `w` pixels wide (w a
// multiple of 16), the rows starting and ending anywhere in their tiles, with
// room for `row_ints` row deltas (at least one row's, WalkRowInts).
__host__ __device__ inline int WalkRowInts(int w) { return w + 3 * kTile; }
__host__ __device__ inline int WalkTouchInts(int row_ints) {
  return 2 * ((row_ints / kTile + kWave) / kWave);
}
// The 32- and 64-slot walks take one row at a time and keep no next edges
// (iN), so their blit scratch fits into the permutation scratch: a 64-slot
// walk of a 16,384-pixel row just fits the 160 KB of a CU.
constexpr int kWideSlots = 32;
__host__ __device__ inline int WalkLdsInts(int K, int w, int row_ints) {
  return (K >= kWideSlots ? 0 : kBlitScratchInts) + 5 * K * kWave + row_ints +
         WalkTouchInts(row_ints) + 3 * (w / kTile + 2) + (w / kTile + 3) / 2;
}
// What follows a closing edge in the list: nothing, an edge whose distance
// the interval checks, or one that is known to be too close.
enum : int32_t { kNextNone = 0, kNextCheck = 1, kNextClose = 2 };

// Bitonic sort (ascending) of N = 64 * 2^j keys held as element
// p = slot * 64 + lane; keys at p >= N are not touched (N <= 64 * K).
template <int K, int SS>
__device__ __forceinline__ void SlotExchange(int64_t (&key)[K], int size, int lane) {
#pragma unroll
  for (int s = 0; s < K; s++) {
    const int t = s ^ SS;
    if (t > s && t < K) {
      int p = s * kWave + lane;
      bool asc = (p & size) == 0;
      int64_t a = key[s], b = key[t];
      bool sw = asc ? (a > b) : (a < b);
      key[s] = sw ? b : a;
      key[t] = sw ? a : b;
    }
  }
}
template <int K>
__device__ void BitonicSortSlots(int64_t (&key)[K], int N, int lane) {
  for (int size = 2; size <= N; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= kWave) {
        int ss = stride / kWave;
        if (ss == 1) SlotExchange<K, 1>(key, size, lane);
        else if (ss == 2) SlotExchange<K, 2>(key, size, lane);
        else if (ss == 4) SlotExchange<K, 4>(key, size, lane);
        else if (ss == 8) SlotExchange<K, 8>(key, size, lane);
        else if (ss == 16) SlotExchange<K, 16>(key, size, lane);
        else if (ss == 32) SlotExchange<K, 32>(key, size, lane);
      } else {
        bool lower = (lane & stride) == 0;
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s * kWave >= N) break;
          int64_t o = __shfl_xor(key[s], stride, kWave);
          int p = s * kWave + lane;
          bool asc = (p & size) == 0;
          int64_t mn = key[s] < o ? key[s] : o, mx = key[s] < o ? o : key[s];
          key[s] = (lower == asc) ? mn : mx;
        }
      }
    }
  }
}

// Write pass (kWalkWrite): one wave per (job, band) item; the job's map
// starts at kNoTile (filled before the launch), its JobCov at zero, and the
// bands of a job, which run concurrently, take planes from the job's counter
// (JobCov::alloc).  Count and schedule passes: one wave per job, band
// 0, walking every row and recording the band snapshots.
template <int K, int kMode>
__device__ __forceinline__ void WalkItem(const WalkParams& P, int wi, int32_t* lds) {
  constexpr int CAP = K * kWave;
  constexpr bool kWrite = kMode == kWalkWrite;
  constexpr bool kBlit = kMode != kWalkSchedule;
  const int lane = Lane();
  const uint64_t t_start = wall_clock64();
  const int item = P.walk_list[wi];
  const int j = item >> kBandBits;
  const int rband = kWrite ? (item & (kMaxBands - 1)) : 0;
  const Job job = P.jobs[j];
  const JobGeo geo = P.geo[j];
  const Canvas cv = P.canvases[job.canvas];
  const int path_top = JobPixBounds(geo).t;  // RastePath's start_y
  PixBounds pb = JobScanBounds(geo);
  TileRange tr = JobTiles(pb, cv.width, cv.height);
  // The LDS row holds the visible columns [ox, ox + W) of the canvas
  // (RowSink folds the deltas of off-canvas pixels), so its width is bounded
  // by the canvas, not by the path.
  const int ox = pb.l > 0 ? pb.l : 0;
  const int W = (pb.r < cv.width ? pb.r : cv.width) - ox;
  int flags = 0;
  int n_tiles = 0, max_active = 0;
  int nE = geo.edges;
  int32_t* map0 = kWrite ? P.map0 + P.map_base[j] : nullptr;
  int32_t* map1 = kWrite ? P.map1 + P.map_base[j] : nullptr;
  if (pb.empty || tr.ntc == 0 || nE == 0 || W > P.lds_width) {
    if (!pb.empty && W > P.lds_width) flags |= 16;
    if (lane == 0 && rband == 0) {
      // field by field: a struct copy would go through scratch memory
      JobCov* c = &P.cov[j];
      c->left = pb.l;
      c->top = pb.t;
      c->right = pb.r;
      c->bottom = pb.b;
      c->tiles = 0;
      c->planes = 0;
      c->alloc = 0;
      c->max_active = 0;
      c->flags = flags;
      c->steps = 0;
      c->time_10ns = 0;
#pragma unroll
      for (int k = 0; k < 5; k++) c->phase[k] = 0;
    }
    return;
  }
  const int nb = P.band_count[j];
  uint8_t* sbase = nb > 1 ? P.snaps + P.snap_base[j] : nullptr;
  auto snap_at = [&](int b) -> SnapHeader* {
    return (SnapHeader*)(sbase + (int64_t)(b - 1) * SnapStride(CAP));
  };
  // the band ends where the next band's snapshot was taken
  const Fixed stop_y = (kWrite && rband + 1 < nb) ? snap_at(rband + 1)->y : kMaxS32;
  WalkLds L;
  constexpr bool kWide = K >= kWideSlots;
  L.sX = lds + (kWide ? 0 : kBlitScratchInts);
  L.sDX = L.sX + CAP;
  L.sDY = L.sDX + CAP;
  L.sLY = L.sDY + CAP;
  L.sM = L.sLY + CAP;
  L.iL = (int4*)L.sX;
  L.iR = L.iL + CAP / 2;
  L.iN = (int2*)(L.iR + CAP / 2);
  L.d = L.sM + CAP;
  L.touch = (uint32_t*)(L.d + P.row_ints);
  L.slot0 = (int32_t*)L.touch + WalkTouchInts(P.row_ints);
  L.slot1 = L.slot0 + (P.lds_width / kTile + 2);
  L.rows = L.slot1 + (P.lds_width / kTile + 2);
  L.full = L.rows + (P.lds_width / kTile + 2);
  int32_t* blit = kWide ? L.sM : lds;
  L.blit.items = (int4*)blit;
  L.blit.mark = blit + 2 * kWave * 4;
  L.list = blit;
  L.vend = blit + kWave;
  // Delta rows: a row takes its tile columns and one more, which holds the
  // end-of-row entry when the row ends on a tile boundary; up to 16 rows.
  const int ncol = tr.ntc + 1;
  const int row_cap = kWide ? 1 : Min32(P.row_ints / (ncol * kTile), kTile);
  for (int i = lane; i < row_cap * ncol * (kTile / 4); i += kWave)
    ((int4*)L.d)[i] = make_int4(0, 0, 0, 0);
  for (int i = lane; i < tr.ntc; i += kWave) {
    L.slot0[i] = -1;
    L.slot1[i] = -1;
    L.rows[i] = 0;
  }
  for (int i = lane; i < (tr.ntc + 1) / 2; i += kWave) L.full[i] = 0;
  for (int i = lane; i < WalkTouchInts(P.row_ints); i += kWave) L.touch[i] = 0;
  WaveSync();

  const EdgeRec* E = P.wedges + P.edge_base[j];
  EdgeRec* Q = P.qstate + P.q_base[j] + (int64_t)rband * nE;
  const int64_t pbase = kWrite ? P.plane_base[j] : 0;
  const int pcap = kWrite ? P.plane_cap[j] : 0;
  uint8_t* planes = P.planes;

  const Fixed left_clip = (Fixed)((uint32_t)pb.l << 16);
  const Fixed right_clip = (Fixed)((uint32_t)pb.r << 16);
  const int winding_mask = job.fill == HIPR_FILL_EVEN_ODD ? 1 : -1;
  const int cy0 = pb.t > 0 ? pb.t : 0, cy1 = pb.b < cv.height ? pb.b : cv.height;
  // A job whose blend mode is not a no-op for a transparent source keeps the
  // reference's zero-cover direct spans: its tiles take three planes (direct
  // covers, accumulated covers, and a byte per pixel marking a direct span).
  const bool triple = (job.flags & kJobKeepZero) != 0;
  RowSink sink{L.d + (ox & (kTile - 1)), L.touch, ncol * kTile, ox, W, triple};

  // Active list registers.
  Fixed X[K], DX[K], DY[K], LY[K];
  int M[K];
#pragma unroll
  for (int t = 0; t < K; t++) X[t] = DX[t] = DY[t] = LY[t] = M[t] = 0;
  int n = 0;
  int n_planes = 0;   // planes of this lane's tiles (a solid tile counts one)
  int next_slot = 0;  // next plane of the job's range
  int chunk_end = 0;  // end of the chunk taken (several bands)
  int band = -1;      // current 16-row band

  // ---- helpers ---------------------------------------------------------------
  // Write the active list (m elements in lane/slot layout) from scratch.
  auto load_from_scratch = [&](int m) {
#pragma unroll
    for (int s = 0; s < K; s++) {
      int p = s * kWave + lane;
      if (p < m) {
        X[s] = L.sX[p];
        DX[s] = L.sDX[p];
        DY[s] = L.sDY[p];
        LY[s] = L.sLY[p];
        M[s] = L.sM[p];
      }
    }
  };

  // Takes planes for the tile columns `c` of the lanes that need one: plane 0
  // (three of them for a keep-zero job) and / or plane 1 of the column.
  // Count pass: nothing to take, the slots are only marked as held.
  // A job walked by one wave counts its planes itself; the bands of a job
  // share its range and take it kPlaneChunk planes at a time (the host adds
  // that much per band), so that a flush hardly ever waits for an atomic's
  // answer.
  auto take_planes = [&](bool need0, bool need1, int c) {
    int a0 = 0, a1 = 0;
    if (kWrite) {
      const int req = triple ? (need0 ? 3 : 0) : (need0 ? 1 : 0) + (need1 ? 1 : 0);
      const int rincl = ScanSum(req);
      const int rtot = __builtin_amdgcn_readlane(rincl, kWave - 1);
      const int at = rincl - req;
      a0 = next_slot + at;
      a1 = a0 + (need0 ? 1 : 0);
      if (nb > 1 && next_slot + rtot > chunk_end) {
        // the rest of the chunk, then a new one (chunks and triples are both
        // multiples of three)
        const int more = next_slot + rtot - chunk_end;
        const int grab = (more + kPlaneChunk - 1) / kPlaneChunk * kPlaneChunk;
        int got = 0;
        if (lane == 0) got = atomicAdd(&P.cov[j].alloc, grab);
        got = __builtin_amdgcn_readlane(got, 0);
        if (a0 >= chunk_end) a0 += got - chunk_end;
        if (a1 >= chunk_end) a1 += got - chunk_end;
        next_slot = got + more;
        chunk_end = got + grab;
      } else {
        next_slot += rtot;
      }
      // absolute plane numbers, from the job's range or (past its capacity)
      // from the pool
      const bool over0 = need0 && a0 + (triple ? 2 : 0) >= pcap, over1 = need1 && a1 >= pcap;
      int p0 = (int)(pbase + a0), p1 = (int)(pbase + a1);
      if (__ballot(over0 || over1) != 0) {
        // a triple must be contiguous: it never comes from the pool (a
        // job that outgrows its range that way is walked again exactly)
        const int ov = triple ? 0 : (over0 ? 1 : 0) + (over1 ? 1 : 0);
        const int oincl = ScanSum(ov);
        const int otot = __builtin_amdgcn_readlane(oincl, kWave - 1);
        int pg = 0;
        if (lane == 0 && otot > 0) pg = atomicAdd(P.pool_ctr, otot);
        int pi = __builtin_amdgcn_readlane(pg, 0) + oincl - ov;
        if (over0) {
          p0 = !triple && pi < P.pool_cap ? P.pool_base + pi : kNoPlane;
          pi++;
        }
        if (over1) p1 = pi < P.pool_cap ? P.pool_base + pi : kNoPlane;
        if ((over0 && p0 == kNoPlane) || (over1 && p1 == kNoPlane)) flags |= 1;
      }
      a0 = p0;
      a1 = p1;
    }
    if (need0) L.slot0[c] = a0;
    if (need1) L.slot1[c] = a1;
    WaveSync();
  };

  // Finish a band: publish the tile slots of every column to the job map.
  // Each plane row is written once: by the row flush, or here, with zeros
  // for the rows the band never wrote and with 255 for the full rows (which
  // the flush only notes, so that a tile of 16 full rows, most tiles of a
  // large fill, costs neither a plane nor its 256 bytes written and read).
  auto finish_band = [&]() {
    if (band < 0) return;
    const int trow = band - tr.tr0;
    // rows of this band on the canvas
    const int brows = cv.height - band * kTile;
    const int all_rows = brows >= kTile ? 0xFFFF : (1 << brows) - 1;
    for (int c0 = 0; c0 < tr.ntc; c0 += kWave) {
      const int c = c0 + lane;
      const bool ok = c < tr.ntc;
      uint32_t written = 0;
      int fm = 0;
      if (ok) {
        written = (uint32_t)L.rows[c];
        fm = (L.full[c >> 1] >> (16 * (c & 1))) & 0xFFFF;
      }
      const bool has0 = (written & 0xFFFF) != 0 || fm != 0, has1 = (written >> 16) != 0;
      n_tiles += has0 ? 1 : 0;
      n_planes += triple ? (has0 ? 3 : 0) : (has0 ? 1 : 0) + (has1 ? 1 : 0);
      if (kWrite) {
        const bool solid = fm == all_rows && (written & 0xFFFF) == 0;
        const bool need = fm != 0 && !solid && L.slot0[ok ? c : 0] < 0;
        if (__ballot(need) != 0) take_planes(need, false, c);
        const int s0 = ok ? L.slot0[c] : -1, s1 = ok ? L.slot1[c] : -1;
        // Only planes that were found are published; a job that found none is
        // reported through flags and redone by the exact path.
        if (solid || (s0 >= 0 && s0 != kNoPlane)) {
          map0[(int64_t)trow * tr.ntc + c] = solid ? kSolidTile : s0;
          map1[(int64_t)trow * tr.ntc + c] = (s1 >= 0 && s1 != kNoPlane) ? s1 : kNoTile;
        }
        const int4 zero = {0, 0, 0, 0}, ones = {-1, -1, -1, -1};
        if (s0 >= 0 && s0 != kNoPlane) {
          for (int t = 0; t < (triple ? 3 : 1); t++) {
            int4* pl = (int4*)(planes + (int64_t)(s0 + t) * kTilePlaneBytes);
            for (int k = 0; k < kTile; k++)
              if (!((written >> k) & 1)) pl[k] = (fm >> k) & 1 ? ones : zero;
          }
        }
        if (s1 >= 0 && s1 != kNoPlane) {
          int4* pl = (int4*)(planes + (int64_t)s1 * kTilePlaneBytes);
          for (int k = 0; k < kTile; k++)
            if (!((written >> (16 + k)) & 1)) pl[k] = zero;
        }
      }
      if (ok) {
        L.slot0[c] = -1;
        L.slot1[c] = -1;
        L.rows[c] = 0;
        if ((c & 1) == 0) L.full[c >> 1] = 0;  // (c + 1 was read with c)
      }
    }
    WaveSync();
  };

  // The covers of a pixel whose deltas sum to S: the directly emitted span
  // (or the accumulated one where there is none), then the accumulated one;
  // for a keep-zero job the direct cover, the accumulated one, and whether
  // there is a direct span.
  auto covers = [&](int S, uint32_t* first, uint32_t* second, uint32_t* third) {
    const int a = S & 0xFFFF, d = S >> 16;
    const int av = a > 255 ? 255 : a;
    const int cnt = d >> 12;  // direct spans
    const bool dir = cnt != 0;
    const int dv = d & (kDirectCount - 1);
    if (triple) {
      *first = dir ? dv & 0xFF : 0;
      *second = av;
      *third = dir ? 1 : 0;
    } else {
      *first = (dir ? dv : av) & 0xFF;
      *second = dir ? av : 0;
      *third = 0;
    }
    if (cnt >= 2) flags |= 4;
  };

  // Resolve the `rows` pixel rows from r on (delta rows 0 .. rows - 1, all in
  // one band) and emit their tile rows.  Only the tile columns that hold
  // deltas are summed, 16 of them at a time (four lanes of four pixels each,
  // in column order, so one prefix sum runs through them); the columns
  // between take the value at the end of the touched column before them, one
  // lane per column.  The rows lie end to end: a row's deltas add up to zero,
  // so the sum starts each row at zero.
  auto flush_rows = [&](int r, int rows) {
    WaveSync();
    const int rb = r >> 4;
    if (rb != band) {
      finish_band();
      band = rb;
    }
    const int rowk0 = r & 15;
    const int cols = rows * ncol;
    // column -> row and tile column (col < 2^11, and the quotient is at least
    // 1 / (2 ncol) away from an integer)
    const float inv = rows > 1 ? __builtin_amdgcn_rcpf((float)ncol) : 0.f;
    auto place = [&](int col, int* row, int* tcol) {
      *row = 0;
      *tcol = col;
      if (rows > 1) {
        const int q = (int)(((float)col + 0.5f) * inv);
        *row = q;
        *tcol = col - __mul24(q, ncol);
      }
    };
    int carry = 0;
    for (int g = 0; g < cols; g += kWave) {
      const uint32_t* tw = L.touch + 2 * (g / kWave);
      const uint64_t T = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)tw[0]) |
                         (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)tw[1]) << 32;
      if (T == 0 && carry == 0) continue;
      const int v_in = carry;
      if (T != 0) {
        if (lane < 2) L.touch[2 * (g / kWave) + lane] = 0;
        if (__builtin_amdgcn_inverse_ballot_w64(T)) L.list[CountBelow(T)] = lane;
        WaveSync();
        const int nt = __popcll(T);
        for (int b = 0; b < nt; b += kWave / 4) {
          const int ti = b + (lane >> 2), sub = lane & 3;
          const bool held = ti < nt;
          const int col = held ? L.list[ti] : 0;
          int jrow, tcol;
          place(g + col, &jrow, &tcol);
          const bool ok = held && tcol < tr.ntc;  // not the end-of-row column
          const int rowk = rowk0 + jrow;
          int4 dv = make_int4(0, 0, 0, 0);
          if (held) {
            int4* dp = (int4*)(L.d + (g + col) * kTile + 4 * sub);
            dv = *dp;
            *dp = make_int4(0, 0, 0, 0);
          }
          const int t1 = dv.x + dv.y, t2 = t1 + dv.z, t3 = t2 + dv.w;
          const int incl = ScanSum(t3);
          const int e = incl - t3 + carry;
          carry += __builtin_amdgcn_readlane(incl, kWave - 1);
          if (held && sub == 3) L.vend[col] = e + t3;
          // Most rows have only one kind of span in 16 columns: steps of less
          // than a row accumulate, and a step of a whole row sends its spans
          // directly unless edges are close.
          const int v0 = e + dv.x, v1 = e + t1, v2 = e + t2, v3 = e + t3;
          const uint32_t any = (uint32_t)(v0 | v1 | v2 | v3);
          uint32_t c0 = 0, c1 = 0, c2 = 0;
          if (!triple && __ballot((any >> 16) != 0) == 0) {
            c0 = (uint32_t)Min32(v0, 255) | (uint32_t)Min32(v1, 255) << 8 |
                 (uint32_t)Min32(v2, 255) << 16 | (uint32_t)Min32(v3, 255) << 24;
          } else if (!triple && __ballot((any & 0xEF00FFFFu) != 0) == 0) {
            // direct covers up to 255, one span at a pixel
            c0 = ((uint32_t)v0 >> 16 & 0xFF) | ((uint32_t)v1 >> 8 & 0xFF00) |
                 ((uint32_t)v2 & 0xFF0000) | ((uint32_t)v3 << 8 & 0xFF000000);
          } else {
            uint32_t f, s2, t;
            covers(v0, &f, &s2, &t);
            c0 = f, c1 = s2, c2 = t;
            covers(v1, &f, &s2, &t);
            c0 |= f << 8, c1 |= s2 << 8, c2 |= t << 8;
            covers(v2, &f, &s2, &t);
            c0 |= f << 16, c1 |= s2 << 16, c2 |= t << 16;
            covers(v3, &f, &s2, &t);
            c0 |= f << 24, c1 |= s2 << 24, c2 |= t << 24;
          }
          // the tile row's state over its four lanes: bit 0 a cover in plane
          // 0, bit 1 one in plane 1, bit 2 not full
          int st = 0;
          if (ok) {
            st = triple ? ((c0 | c1 | c2) != 0 ? 5 : 4)
                        : (c0 != 0 ? 1 : 0) | (c1 != 0 ? 2 : 0) |
                              (c0 != 0xFFFFFFFFu || c1 != 0 ? 4 : 0);
          }
          st |= DppSwapPairs(st);
          st |= DppSwapHalves(st);
          const bool plane0 = (st & 5) == 5, plane1 = (st & 2) != 0;
          const int cc = ok ? tcol : 0;
          if (sub == 0 && ok) {
            if ((st & 5) == 1) atomicOr(&L.full[cc >> 1], 1 << (16 * (cc & 1) + rowk));
            const int wr = (plane0 ? 1 << rowk : 0) | (plane1 ? 1 << (16 + rowk) : 0);
            if (wr) atomicOr(&L.rows[cc], wr);
          }
          int cur0 = L.slot0[cc], cur1 = L.slot1[cc];
          bool need0 = sub == 0 && plane0 && cur0 < 0;
          bool need1 = sub == 0 && plane1 && cur1 < 0;
          // most columns already hold their planes: allocate only when needed
          if (__ballot(need0 || need1) != 0) {
            // several rows may meet the same column here: one of them asks
            if (rows > 1) {
              if (need0) need0 = atomicCAS(&L.slot0[cc], -1, -2) == -1;
              if (need1) need1 = atomicCAS(&L.slot1[cc], -1, -2) == -1;
            }
            take_planes(need0, need1, cc);
            cur0 = L.slot0[cc];
            cur1 = L.slot1[cc];
          }
          if (kWrite) {
            if (plane0 && cur0 != kNoPlane) {
              uint32_t* pl = (uint32_t*)(planes + (int64_t)cur0 * kTilePlaneBytes);
              pl[rowk * 4 + sub] = c0;
              if (triple) {
                pl[kTilePlaneBytes / 4 + rowk * 4 + sub] = c1;
                pl[2 * kTilePlaneBytes / 4 + rowk * 4 + sub] = c2;
              }
            }
            if (plane1 && cur1 != kNoPlane) {
              uint32_t* pl = (uint32_t*)(planes + (int64_t)cur1 * kTilePlaneBytes);
              pl[rowk * 4 + sub] = c1;
            }
          }
        }
        WaveSync();
      }
      // the other columns of the group
      const uint64_t below = T & ((1ull << lane) - 1);
      int v = v_in;
      if (below) v = L.vend[kWave - 1 - __builtin_clzll(below)];
      int jrow, c;
      place(g + lane, &jrow, &c);
      const int rowk = rowk0 + jrow;
      const bool rest = g + lane < cols && c < tr.ntc && ((T >> lane) & 1) == 0 && v != 0;
      if (__ballot(rest) == 0) continue;
      uint32_t f = 0, s2 = 0, t = 0;
      if (rest) covers(v, &f, &s2, &t);
      const bool is_full = !triple && f == 255 && s2 == 0;
      const bool plane0 = rest && !is_full && (triple ? (f | s2 | t) != 0 : f != 0);
      const bool plane1 = rest && !triple && s2 != 0;
      if (rest && is_full) atomicOr(&L.full[c >> 1], 1 << (16 * (c & 1) + rowk));
      if (__ballot(plane0 || plane1) == 0) continue;
      const int cc = rest ? c : 0;
      const int wr = (plane0 ? 1 << rowk : 0) | (plane1 ? 1 << (16 + rowk) : 0);
      if (wr) atomicOr(&L.rows[cc], wr);
      bool need0 = plane0 && L.slot0[cc] < 0, need1 = plane1 && L.slot1[cc] < 0;
      if (__ballot(need0 || need1) != 0) {
        if (rows > 1) {
          if (need0) need0 = atomicCAS(&L.slot0[cc], -1, -2) == -1;
          if (need1) need1 = atomicCAS(&L.slot1[cc], -1, -2) == -1;
        }
        take_planes(need0, need1, cc);
      }
      if (kWrite) {
        const int cur0 = L.slot0[cc], cur1 = L.slot1[cc];
        auto put = [&](int slot, uint32_t b) {
          const int w = (int)(b * 0x01010101u);
          ((int4*)(planes + (int64_t)slot * kTilePlaneBytes))[rowk] = make_int4(w, w, w, w);
        };
        if (plane0 && cur0 != kNoPlane) {
          put(cur0, f);
          if (triple) {
            put(cur0 + 1, s2);
            put(cur0 + 2, t);
          }
        }
        if (plane1 && cur1 != kNoPlane) put(cur1, s2);
      }
    }
    WaveSync();
  };

  // ---- pending edges ---------------------------------------------------------
  // The next 64 pending edges are kept in registers, lane i holding sorted
  // edge w_base + i, so that looking at the next one and activating edges
  // takes no memory access.
  int pp = 0;  // next pending edge (sorted position)
  int w_base = 0;
  Fixed w_x = 0, w_dx = 0, w_dy = 0, w_uy = kMaxS32, w_ly = 0;
  int w_pk = 0;
  auto load_window = [&](int base) {
    w_base = base;
    const int idx = base + lane;
    w_uy = kMaxS32;
    if (idx < nE) {
      const int4* e = (const int4*)&E[idx];
      const int4 a = e[0], b = e[1];
      w_x = a.x;
      w_dx = a.z;
      w_dy = a.w;
      w_uy = b.y;
      w_ly = b.z;
      w_pk = b.w;
    }
  };
  // upper_y of the next pending edge (kMaxS32 after the last)
  auto pending_upper = [&]() -> Fixed {
    if (pp - w_base >= kWave) load_window(pp);
    return __builtin_amdgcn_readlane(w_uy, pp - w_base);
  };
  Fixed nny = kMaxS32;
  Fixed min_ly = kMaxS32;  // smallest lower_y of the active list

  // Takes the pending edges with upper_y <= y into the active list
  // (insert_new_edges; with an empty list, the initial activation).  Returns
  // false when the list outgrows the walk.
  auto insert_new = [&](Fixed y, bool initial) -> bool {
    if (pp - w_base >= kWave) load_window(pp);
    int off = pp - w_base;
    uint64_t ready = __ballot(lane >= off && w_uy <= y);
    if ((ready >> (kWave - 1)) != 0 && off > 0) {
      // the run may go on past the window
      load_window(pp);
      off = 0;
      ready = __ballot(w_uy <= y);
    }
    int k = __popcll(ready);
    if (k == kWave) {
      // 64 or more at once: count them all
      for (;;) {
        const int idx = pp + k + lane;
        const int cnt = __popcll(__ballot(idx < nE && E[idx < nE ? idx : 0].upper_y <= y));
        k += cnt;
        if (n + k > CAP) return false;
        if (cnt < kWave) break;
      }
    }
    if (n + k > CAP) return false;
    WaveSync();
    if (k <= kWave) {
      // lane i takes new edge i
      const bool mine = lane < k;
      Fixed nX = w_x, nDX = w_dx, nDY = w_dy, nLY = w_ly;
      int nM = MakeMeta(EdgeWinding(w_pk), EdgeIsQuad(w_pk), false, w_base + lane);
      if (off != 0) {
        const int src = (lane + off) & (kWave - 1);
        nX = __shfl(nX, src, kWave);
        nDX = __shfl(nDX, src, kWave);
        nDY = __shfl(nDY, src, kWave);
        nLY = __shfl(nLY, src, kWave);
        nM = __shfl(nM, src, kWave);
      }
      if (k > 1) {
        // sorted by (x, dx, sorted position): rank by counting
        int r = 0;
        for (int q = 0; q < k; q++) {
          const Fixed xq = __builtin_amdgcn_readlane(nX, q);
          const Fixed dxq = __builtin_amdgcn_readlane(nDX, q);
          r += (xq < nX || (xq == nX && (dxq < nDX || (dxq == nDX && q < lane)))) ? 1 : 0;
        }
        if (!mine) r = lane;
        if (__ballot(r != lane) != 0) {
          nX = __builtin_amdgcn_ds_permute(4 * r, nX);
          nDX = __builtin_amdgcn_ds_permute(4 * r, nDX);
          nDY = __builtin_amdgcn_ds_permute(4 * r, nDY);
          nLY = __builtin_amdgcn_ds_permute(4 * r, nLY);
          nM = __builtin_amdgcn_ds_permute(4 * r, nM);
        }
      }
      const int least = DppWaveMin(mine ? nLY : kMaxS32);
      min_ly = Min32(min_ly, least);
      const int mn = initial ? DppWaveMin(mine && nLY > y ? nLY : kMaxS32) : least;
      // insertion positions: P0 = #{a : x_a <= x_N0};
      // Pi = max(P(i-1), #{a : x_a < x_Ni}); list element q moves to
      // q + #{i : Pi <= q}, new edge i goes to Pi + i
      int my_pos = 0, p_cur = 0, first_pos = 0;
      int shift[K];
#pragma unroll
      for (int s = 0; s < K; s++) shift[s] = 0;
      const int S0 = (n + kWave - 1) / kWave;
      if (n > 0) {
        for (int i = 0; i < k; i++) {
          const Fixed xi = __builtin_amdgcn_readlane(nX, i);
          int cnt = 0;
#pragma unroll
          for (int s = 0; s < K; s++) {
            if (s >= S0) break;
            const int p = s * kWave + lane;
            cnt += __popcll(__ballot(p < n && (i == 0 ? X[s] <= xi : X[s] < xi)));
          }
          if (i == 0) first_pos = cnt;
          p_cur = Max32(p_cur, cnt);
          my_pos = lane == i ? p_cur : my_pos;
#pragma unroll
          for (int s = 0; s < K; s++) {
            if (s >= S0) break;
            shift[s] += (s * kWave + lane >= p_cur) ? 1 : 0;
          }
        }
      }
      if (!initial) {
        // check_intersection with the predecessor at insertion: the new edge
        // before it if that sits right there, else the list element before
        bool crosses = false;
        if (n > 0) {
#pragma unroll
          for (int s = 0; s < K; s++) {
            if (s >= S0) break;
            L.sM[s * kWave + lane] = X[s] + DX[s];
          }
          WaveSync();
        }
        const Fixed v = nX + nDX;
        const Fixed pv = ShiftUp(v, 0);
        const int ppos = ShiftUp(my_pos, -1);
        if (mine) {
          if (lane > 0 && ppos == my_pos) {
            crosses = pv > v;
          } else if (my_pos > 0) {
            crosses = L.sM[my_pos - 1] > v;
          }
        }
        if (__ballot(crosses) != 0) nny = y + (kFixed1 >> kAcc);
        WaveSync();
      }
      if (mn > y && mn < nny) nny = mn;
      // merge through scratch, from the slot of the first new edge on
      const int s_from = first_pos / kWave;
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s >= S0) break;
        if (s < s_from) continue;
        const int q = s * kWave + lane;
        if (q < n) {
          const int d = q + shift[s];
          L.sX[d] = X[s];
          L.sDX[d] = DX[s];
          L.sDY[d] = DY[s];
          L.sLY[d] = LY[s];
          L.sM[d] = M[s];
        }
      }
      if (mine) {
        const int d = my_pos + lane;
        L.sX[d] = nX;
        L.sDX[d] = nDX;
        L.sDY[d] = nDY;
        L.sLY[d] = nLY;
        L.sM[d] = nM;
      }
      WaveSync();
      n += k;
      pp += k;
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s < s_from) continue;
        const int p = s * kWave + lane;
        if (p < n) {
          X[s] = L.sX[p];
          DX[s] = L.sDX[p];
          DY[s] = L.sDY[p];
          LY[s] = L.sLY[p];
          M[s] = L.sM[p];
        }
      }
      WaveSync();
      return true;
    }
    if (K == 1) return false;
    // More than 64 at once (K > 1): the same through scratch.
    for (int p = lane; p < k; p += kWave) {
      const EdgeRec* er = &E[pp + p];
      const int32_t packed = er->packed;
      L.sX[p] = er->x;
      L.sDX[p] = er->dx;
      L.sDY[p] = er->dy;
      L.sLY[p] = er->lower_y;
      L.sM[p] = MakeMeta(EdgeWinding(packed), EdgeIsQuad(packed), false, pp + p);
    }
    WaveSync();
    int rk[K];
    Fixed nX[K], nDX[K], nDY[K], nLY[K];
    int nM[K];
    int mn = kMaxS32, least = kMaxS32;
#pragma unroll
    for (int s = 0; s < K; s++) {
      const int p = s * kWave + lane;
      rk[s] = 0;
      if (p < k) {
        const Fixed xi = L.sX[p], dxi = L.sDX[p];
        int r = 0;
        for (int q = 0; q < k; q++) {
          const Fixed xq = L.sX[q], dxq = L.sDX[q];
          r += (xq < xi || (xq == xi && (dxq < dxi || (dxq == dxi && q < p)))) ? 1 : 0;
        }
        rk[s] = r;
        nX[s] = xi;
        nDX[s] = dxi;
        nDY[s] = L.sDY[p];
        nLY[s] = L.sLY[p];
        nM[s] = L.sM[p];
        least = Min32(least, nLY[s]);
        if (!initial || nLY[s] > y) mn = Min32(mn, nLY[s]);
      }
    }
    mn = DppWaveMin(mn);
    min_ly = Min32(min_ly, DppWaveMin(least));
    WaveSync();
#pragma unroll
    for (int s = 0; s < K; s++) {
      const int p = s * kWave + lane;
      if (p < k) {
        L.sX[rk[s]] = nX[s];
        L.sDX[rk[s]] = nDX[s];
      }
    }
    WaveSync();
    // positions of the new edges in sorted order, kept in sLY
    int p_cur = 0;
    bool crosses = false;
    int shift[K];
#pragma unroll
    for (int s = 0; s < K; s++) shift[s] = 0;
    for (int i = 0; i < k; i++) {
      const Fixed xi = L.sX[i];
      int cnt = 0;
#pragma unroll
      for (int s = 0; s < K; s++) {
        const int p = s * kWave + lane;
        cnt += __popcll(__ballot(p < n && (i == 0 ? X[s] <= xi : X[s] < xi)));
      }
      const int prev = p_cur;
      p_cur = Max32(p_cur, cnt);
      Fixed pred = 0;
      bool has_pred = false;
      if (i > 0 && p_cur == prev) {
        pred = L.sX[i - 1] + L.sDX[i - 1];
        has_pred = true;
      } else if (p_cur > 0) {
        const int q = __builtin_amdgcn_readfirstlane(p_cur - 1);
#pragma unroll
        for (int t = 0; t < K; t++)
          if (t == q / kWave) pred = __builtin_amdgcn_readlane(X[t] + DX[t], q % kWave);
        has_pred = true;
      }
      if (has_pred && pred > xi + L.sDX[i]) crosses = true;
      if (lane == 0) L.sLY[i] = p_cur;
#pragma unroll
      for (int s = 0; s < K; s++) shift[s] += (s * kWave + lane >= p_cur) ? 1 : 0;
    }
    if (!initial && crosses) nny = y + (kFixed1 >> kAcc);
    if (mn > y && mn < nny) nny = mn;
    WaveSync();
    int posN[K];
#pragma unroll
    for (int s = 0; s < K; s++) {
      const int p = s * kWave + lane;
      posN[s] = p < k ? L.sLY[rk[s]] + rk[s] : 0;
    }
    WaveSync();
#pragma unroll
    for (int s = 0; s < K; s++) {
      const int q = s * kWave + lane;
      if (q < n) {
        const int d = q + shift[s];
        L.sX[d] = X[s];
        L.sDX[d] = DX[s];
        L.sDY[d] = DY[s];
        L.sLY[d] = LY[s];
        L.sM[d] = M[s];
      }
      if (q < k) {
        const int d = posN[s];
        L.sX[d] = nX[s];
        L.sDX[d] = nDX[s];
        L.sDY[d] = nDY[s];
        L.sLY[d] = nLY[s];
        L.sM[d] = nM[s];
      }
    }
    WaveSync();
    n += k;
    pp += k;
    load_from_scratch(n);
    WaveSync();
    return true;
  };

  // ---- initial activation (sw_raster.cc:554-563) -------------------------------
  Fixed y = Max32(E[0].upper_y, IntToFixed(path_top));
  if (rband > 0) {
    // resume from the band's snapshot
    const SnapHeader* h = snap_at(rband);
    y = h->y;
    if (y == kMaxS32) return;  // the walk ended before this band
    nny = h->nny;
    pp = h->pp;
    n = h->n;
    const int32_t* a = (const int32_t*)(h + 1);
    const EdgeRec* qs = (const EdgeRec*)(a + 5 * CAP);
    int mn = kMaxS32;
#pragma unroll
    for (int s = 0; s < K; s++) {
      int p = s * kWave + lane;
      if (p < n) {
        X[s] = a[p];
        DX[s] = a[CAP + p];
        DY[s] = a[2 * CAP + p];
        LY[s] = a[3 * CAP + p];
        M[s] = a[4 * CAP + p];
        if (MetaMoved(M[s])) Q[MetaIndex(M[s])] = qs[p];
        mn = Min32(mn, LY[s]);
      }
    }
    min_ly = DppWaveMin(mn);
    load_window(pp);
  } else {
    load_window(0);
    if (!insert_new(y, true)) flags |= 2;
    const Fixed nu = pending_upper();
    if (nu > y && nu < nny) nny = nu;
  }

  const Fixed stop_fixed = IntToFixed(pb.b);
  int guard = 0;  // steps taken
  uint32_t turn = 0;
  // Phase times (10 ns units) of every 16th turn: reading the clock waits for
  // it and for the LDS operations in flight, which took a third of a small
  // step when every step did it five times.
  uint64_t ph[5] = {0, 0, 0, 0, 0};
  const uint64_t tp_loop = wall_clock64();
  int next_b = 1;  // next band snapshot to record (count / schedule passes)
  for (;;) {
    if (y >= stop_y) break;  // the next band starts here
    if (!kWrite && next_b < nb && (y & 0xFFFF) == 0 && ((y >> 16) & (kTile - 1)) == 0) {
      const int yrow = y >> 16;
      while (next_b < nb && yrow >= BandStartRow(pb, nb, next_b)) {
        SnapHeader* h = snap_at(next_b);
        if (lane == 0) {
          h->y = y;
          h->nny = nny;
          h->pp = pp;
          h->n = n;
        }
        int32_t* a = (int32_t*)(h + 1);
        EdgeRec* qs = (EdgeRec*)(a + 5 * CAP);
#pragma unroll
        for (int s = 0; s < K; s++) {
          int p = s * kWave + lane;
          if (p < n) {
            a[p] = X[s];
            a[CAP + p] = DX[s];
            a[2 * CAP + p] = DY[s];
            a[3 * CAP + p] = LY[s];
            a[4 * CAP + p] = M[s];
            if (MetaMoved(M[s])) qs[p] = Q[MetaIndex(M[s])];
          }
        }
        next_b++;
      }
    }
    if (++guard > (1 << 26)) {  // cannot happen: y strictly increases
      flags |= 32;
      break;
    }
    const bool sample = (turn++ & 15) == 0;
    max_active = Max32(max_active, n);
    Fixed next_y = Min32(nny, FixedCeilToFixed(y + 1));
    int y_shift = 0;
    if ((next_y - y) & (kFixed1 >> 2)) {
      y_shift = 2;
      next_y = y + (kFixed1 >> 2);
    } else if ((next_y - y) & (kFixed1 >> 1)) {
      y_shift = 1;
    }
    const Alpha full = (Alpha)FixedRoundToInt(0xFF * (next_y - y));
    const int row = y >> 16;
    const int S = (n + kWave - 1) / kWave;
    // rows off the canvas are stepped but not drawn
    const bool draw = kBlit && row >= cy0 && row < cy1;
    // ---- several rows at once ----------------------------------------------------
    // From a whole row on, until the first event (an edge ends or begins),
    // every step is one whole row as long as no two edges cross, and the list
    // stays as it is: row i is x + i dx.  Each neighbouring pair moves apart
    // or together linearly, so a list in order now and after `rows` rows is in
    // order on all rows between, and the steps up to there are taken as one.
    // A list of few edges, most of them, takes 16 rows (a band, as many delta
    // rows as fit) in little more than the time of one.  (The first row may hold
    // edges that have ended before it: a tall quad whose first piece runs
    // upward, by the rounding of its forward differences.  They take this row's
    // step and go on or end after it.)
    int rows = 1;
    if ((y & 0xFFFF) == 0 && min_ly > y) {
      int most = Min32((nny - 1) >> 16, stop_fixed >> 16) - row;
      if (kWrite && stop_y != kMaxS32) most = Min32(most, (stop_y >> 16) - row);
      if (!kWrite && next_b < nb) {
        // not past the row of the next snapshot
        const int at = Max32(BandStartRow(pb, nb, next_b), (row + kTile) & ~(kTile - 1));
        most = Min32(most, at - row);
      }
      if (draw) {
        most = Min32(most, Min32(row_cap, kTile - (row & (kTile - 1))));
        most = Min32(most, cy1 - row);
      } else {
        most = Min32(most, kWave - 1);
        if (kBlit && row < cy0) most = Min32(most, cy0 - row);
      }
      if (most > 1) {
        // no overflow on the way: |x| < 2^30, |63 dx| < 2^29
        bool off = false;
        Fixed cx = kMinS32, cj = kMinS32;
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s >= S) break;
          const bool valid = s * kWave + lane < n;
          const Fixed x0 = X[s], xj = x0 + __mul24(DX[s], most);
          const Fixed p0 = ShiftUp(x0, cx), pj = ShiftUp(xj, cj);
          off |= valid && (p0 > x0 || pj > xj || (uint32_t)(DX[s] + (1 << 23)) >= (1u << 24) ||
                           (uint32_t)(x0 + (1 << 30)) >= (1u << 31));
          cx = __builtin_amdgcn_readlane(x0, kWave - 1);
          cj = __builtin_amdgcn_readlane(xj, kWave - 1);
        }
        if (__ballot(off) == 0) {
          rows = most;
          next_y = y + rows * kFixed1;
          guard += rows - 1;
        }
      }
    }

    uint64_t tp0 = 0, tp1 = 0, tp2 = 0, tp3 = 0, tp4 = 0;
    if (sample) tp0 = wall_clock64();
    // ---- one pass over the list: interval edges, step, order checks -----------
    // An edge opens or closes an interval where the winding sum up to it
    // changes between inside and outside.  The k-th opening edge belongs to
    // the k-th closing one, so both kinds are packed into LDS in list order
    // and interval k reads entries k (and k - 1 for the interval before).
    // Windings are counted from ballots: no scan.  The step itself and the
    // two order checks (is the stepped list still sorted, does an edge cross
    // its predecessor within the next step) use the same registers; when no
    // edge ends and the order holds, which is most steps, the step is done.
    uint64_t ends = 0;
    bool bad = false, cross = false;
    int carry_w = 0, nl = 0, nr = 0;
    uint64_t carry_in = 0;
    {
      Fixed cx = kMinS32, cv = kMinS32;
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s >= S) break;
        const int rem = n - s * kWave;
        const uint64_t bval = rem >= kWave ? ~0ull : (1ull << rem) - 1;
        const bool valid = lane < rem;
        const Fixed xo = X[s], dx = DX[s], step = dx >> y_shift;
        const Fixed xn = rows > 1 ? xo + __mul24(dx, rows) : xo + step;
        if (draw) {
          const bool neg = (M[s] & 1) != 0;
          const uint64_t bneg = __ballot(neg) & bval, bpos = bval & ~bneg;
          const int incl = CountBelow(bpos, carry_w) - CountBelow(bneg) + (neg ? -1 : 1);
          const uint64_t bin = __ballot((incl & winding_mask) != 0) & bval;
          const uint64_t prev = (bin << 1) | carry_in;
          const uint64_t bl = bin & ~prev, br = bval & ~bin & prev;
          // the next element (old x, dx); lane 63's is lane 0 of slot s + 1
          Fixed nxo = ShiftDown(xo, xo), ndx = ShiftDown(dx, dx);
          if (s + 1 < K) {
            const Fixed n0x = __builtin_amdgcn_readlane(X[s + 1 < K ? s + 1 : s], 0);
            const Fixed n0dx = __builtin_amdgcn_readlane(DX[s + 1 < K ? s + 1 : s], 0);
            if (lane == kWave - 1) {
              nxo = n0x;
              ndx = n0dx;
            }
          }
          if (__builtin_amdgcn_inverse_ballot_w64(bl))
            L.iL[CountBelow(bl, nl)] = make_int4(xo, step, DY[s], 0);
          if (__builtin_amdgcn_inverse_ballot_w64(br)) {
            const int at = CountBelow(br, nr);
            int next = lane + 1 < rem ? kNextCheck : kNextNone;
            if (kWide) {
              if (next != kNextNone)
                next = xn + kFixed1 >= nxo - Abs32(ndx) ? kNextClose : kNextNone;
            } else {
              L.iN[at] = make_int2(nxo, ndx);
            }
            L.iR[at] = make_int4(xo, step, DY[s], next);
          }
          nl += __popcll(bl);
          nr += __popcll(br);
          carry_w += __popcll(bpos) - __popcll(bneg);
          carry_in = (bin >> ((rem >= kWave ? kWave : rem) - 1)) & 1;
        }
        ends |= __ballot(LY[s] <= next_y) & bval;
        X[s] = xn;
        const Fixed v = xn + dx;
        const Fixed px = ShiftUp(xn, cx), pv = ShiftUp(v, cv);
        bad |= valid && px > xn;
        cross |= valid && pv > v;
        cx = __builtin_amdgcn_readlane(xn, kWave - 1);
        cv = __builtin_amdgcn_readlane(v, kWave - 1);
      }
    }
    // ---- the step's trapezoids -------------------------------------------------
    if (draw) {
      if (carry_in) {
        // open interval at the end of the list (right edge culled away): it
        // runs to the right clip.  The reference tests
        // edges_too_close(left_edge->prev, left_edge); with a closed path the
        // winding sum is 0 here, so this is not reached on the parity scenes.
        // The left edge's list predecessor is not tracked; the span is
        // emitted as accumulated coverage.
        flags |= 8;
        if (lane == 0) {
          L.iR[nr] = make_int4(right_clip, 0, 0, kNextClose);
          if (!kWide) L.iN[nr] = make_int2(0, 0);
        }
        nr++;
      }
      WaveSync();
      // two lanes (left and right edge) per interval and row
      const int total = nr * rows;
      // (rows > 1: t / nr by a product; t < 2^13, and a quotient is at least
      // 1 / (2 nr) away from an integer)
      const float inv = rows > 1 ? __builtin_amdgcn_rcpf((float)nr) : 0.f;
      for (int t0 = 0; t0 < total; t0 += kWave / 2) {
        const int t = t0 + (lane >> 1);
        const bool act = t < total;
        int jr = 0, k = t;
        if (rows > 1) {
          jr = (int)(((float)t + 0.5f) * inv);
          k = t - __mul24(jr, nr);
        }
        int4 l = make_int4(0, 0, 0, 0), r = l, q = l;
        int2 nx = make_int2(0, 0);
        if (act) {
          l = L.iL[k];
          r = L.iR[k];
          if (!kWide) nx = L.iN[k];
          if (k > 0) q = L.iR[k - 1];
        }
        if (rows > 1) {
          l.x += __mul24(l.y, jr);
          r.x += __mul24(r.y, jr);
          q.x += __mul24(q.y, jr);
          nx.x += __mul24(nx.y, jr);
        }
        const Fixed lxn = l.x + l.y, rxn = r.x + r.y;
        const Fixed left = Max32(l.x, left_clip), next_left = Max32(left_clip, lxn);
        const Fixed right = Min32(right_clip, r.x), next_right = Min32(right_clip, rxn);
        const int prev_right = k > 0 ? FixedCeilToInt(Max32(Min32(right_clip, q.x), q.x + q.y))
                                     : FixedFloorToInt(left_clip);
        const bool close_prev =
            prev_right > FixedFloorToInt(left) || prev_right > FixedFloorToInt(lxn);
        const bool close_next =
            r.w == kNextClose ||
            (r.w == kNextCheck && (rxn + kFixed1 >= nx.x - Abs32(nx.y)));
        const bool no_real = full == 0xFF && (close_prev || close_next);
        BlitEdges(sink, L.blit, act, lane & 1, jr, left, right, next_left, next_right, l.z, r.z,
                  full, no_real);
      }
      WaveSync();
    }

    if (sample) {
      tp1 = wall_clock64();
      ph[0] += tp1 - tp0;
    }
    // ---- quad updates ------------------------------------------------------------
    int m = n;
    uint64_t dead = 0;
    if (ends != 0) {
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s >= S) break;
        int p = s * kWave + lane;
        if (p < n && LY[s] <= next_y && MetaQuad(M[s])) {
          // while (lower_y <= next_y) { KeepContinuous; UpdateQuad } with
          // KeepContinuous taking the edge's current x and y
          // (sw_raster.cc:628-638, sw_edge.cc:294-297).
          const int idx = MetaIndex(M[s]);
          EdgeRec e;
          {
            const int4* src = (const int4*)(MetaMoved(M[s]) ? (const EdgeRec*)&Q[idx] : &E[idx]);
            int4* dst = (int4*)&e;
            const int4 q0 = src[0], q1 = src[1], q2 = src[2], q3 = src[3];
            dst[0] = q0;
            dst[1] = q1;
            dst[2] = q2;
            dst[3] = q3;
          }
          Fixed sy = next_y;
          Fixed cx = X[s];
          while (LY[s] <= next_y && EdgeCurveCount(e.packed) > 0) {
            e.snapped_x = cx;
            if (!UpdateQuad(&e, sy)) break;
            cx = e.x;
            sy = e.upper_y;
            DX[s] = e.dx;
            DY[s] = e.dy;
            LY[s] = e.lower_y;
          }
          X[s] = cx;
          M[s] = MakeMeta(EdgeWinding(e.packed), true, true, idx);
          Q[idx] = e;
        }
        dead |= __ballot(p < n && LY[s] <= next_y);
      }
      if (dead == 0) {
        // every edge lives on: check the order in place
        bad = false;
        cross = false;
        Fixed cx = kMinS32, cv = kMinS32;
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s >= S) break;
          const bool valid = s * kWave + lane < n;
          const Fixed v = X[s] + DX[s];
          const Fixed px = ShiftUp(X[s], cx), pv = ShiftUp(v, cv);
          bad |= valid && px > X[s];
          cross |= valid && pv > v;
          cx = __builtin_amdgcn_readlane(X[s], kWave - 1);
          cv = __builtin_amdgcn_readlane(v, kWave - 1);
        }
      }
    }

    if (sample) {
      tp2 = wall_clock64();
      ph[1] += tp2 - tp1;
    }
    // ---- survivors, stable x order, intersection checks ------------------------
    bool flag_isect = false;
    if (dead == 0 && __ballot(bad) == 0) {
      flag_isect = __ballot(cross) != 0;
    } else {
      // write the survivors to scratch in list order
      m = 0;
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s >= S) break;
        int p = s * kWave + lane;
        const bool sv = p < n && LY[s] > next_y;
        const uint64_t b = __ballot(sv);
        if (sv) {
          const int c = CountBelow(b, m);
          L.sX[c] = X[s];
          L.sDX[c] = DX[s];
          L.sDY[c] = DY[s];
          L.sLY[c] = LY[s];
          L.sM[c] = M[s];
        }
        m += __popcll(b);
      }
      WaveSync();
      const int S2 = (m + kWave - 1) / kWave;
      bad = false;
      cross = false;
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s >= S2) break;
        const int c = s * kWave + lane;
        if (c < m) {
          X[s] = L.sX[c];
          DX[s] = L.sDX[c];
          if (c > 0) {
            const Fixed px = L.sX[c - 1], pdx = L.sDX[c - 1];
            bad |= px > X[s];
            cross |= px + pdx > X[s] + DX[s];
          }
        }
      }
      if (__ballot(bad) == 0) {
        flag_isect = __ballot(cross) != 0;
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s >= S2) break;
          const int c = s * kWave + lane;
          if (c < m) {
            DY[s] = L.sDY[c];
            LY[s] = L.sLY[c];
            M[s] = L.sM[c];
          }
        }
      } else {
        // Stable re-sort by x.  The survivors stay in scratch in list order;
        // only the keys (x, list position) are sorted in registers, by
        // odd-even transposition (a step only swaps edges that crossed, so
        // one or two passes usually do), with a bitonic network when eight
        // passes do not; then the other fields are gathered by position.
        int O[K];
#pragma unroll
        for (int s = 0; s < K; s++) O[s] = s * kWave + lane;
        auto gt_key = [](Fixed xa, int oa, Fixed xb, int ob) {
          return xa > xb || (xa == xb && oa > ob);
        };
        bool sorted = false;
        for (int pass = 0; pass < 8 && !sorted; pass++) {
          // even phase: pairs (2t, 2t+1) are lanes (2t, 2t+1) of one slot
#pragma unroll
          for (int s = 0; s < K; s++) {
            if (s >= S2) break;
            int p = s * kWave + lane;
            int q = p ^ 1;
            Fixed ox = DppSwapPairs(X[s]);
            int oo = DppSwapPairs(O[s]);
            bool both = p < m && q < m;
            bool left = (lane & 1) == 0;
            bool take = both && (left ? gt_key(X[s], O[s], ox, oo) : gt_key(ox, oo, X[s], O[s]));
            if (take) {
              X[s] = ox;
              O[s] = oo;
            }
          }
          // odd phase: pairs (2t+1, 2t+2); lane 63 of slot s pairs with
          // lane 0 of slot s+1.  Slot s+1 has not moved yet when slot s is
          // processed; lane 63 of slot s-1 is kept from before it moved.
          Fixed p63x = 0;
          int p63o = 0;
#pragma unroll
          for (int s = 0; s < K; s++) {
            if (s >= S2) break;
            int p = s * kWave + lane;
            bool left = (lane & 1) == 1;  // odd position = left of its pair
            int q = left ? p + 1 : p - 1;
            const Fixed c63x = __builtin_amdgcn_readlane(X[s], kWave - 1);
            const int c63o = __builtin_amdgcn_readlane(O[s], kWave - 1);
            Fixed dnx = ShiftDown(X[s], 0), upx = ShiftUp(X[s], p63x);
            int dno = ShiftDown(O[s], 0), upo = ShiftUp(O[s], p63o);
            if (s + 1 < K) {
              const int t = s + 1 < K ? s + 1 : s;
              const Fixed n0x = __builtin_amdgcn_readlane(X[t], 0);
              const int n0o = __builtin_amdgcn_readlane(O[t], 0);
              if (lane == kWave - 1) {
                dnx = n0x;
                dno = n0o;
              }
            }
            bool both = p < m && q >= 0 && q < m;
            bool take = both && (left ? gt_key(X[s], O[s], dnx, dno) : gt_key(upx, upo, X[s], O[s]));
            if (take) {
              X[s] = left ? dnx : upx;
              O[s] = left ? dno : upo;
            }
            p63x = c63x;
            p63o = c63o;
          }
          // sorted when every element exceeds its predecessor
          bool worse = false;
          Fixed cx = kMinS32;
          int co = 0;
#pragma unroll
          for (int s = 0; s < K; s++) {
            if (s >= S2) break;
            int p = s * kWave + lane;
            Fixed px = ShiftUp(X[s], cx);
            int po = ShiftUp(O[s], co);
            if (p >= 1 && p < m && gt_key(px, po, X[s], O[s])) worse = true;
            cx = __builtin_amdgcn_readlane(X[s], kWave - 1);
            co = __builtin_amdgcn_readlane(O[s], kWave - 1);
          }
          sorted = __ballot(worse) == 0;
        }
        if (!sorted) {
          // bitonic sort of the keys (x, list position)
          int64_t key[K];
#pragma unroll
          for (int s = 0; s < K; s++) {
            int c = s * kWave + lane;
            // signed x in the high word, list position (>= 0) in the low word
            key[s] = c < m ? (int64_t)(((uint64_t)(uint32_t)X[s] << 32) | (uint32_t)O[s])
                           : INT64_MAX;
          }
          int N = kWave;
          while (N < m) N <<= 1;
          BitonicSortSlots<K>(key, N, lane);
#pragma unroll
          for (int s = 0; s < K; s++) {
            int c = s * kWave + lane;
            if (c < m) {
              X[s] = (Fixed)(key[s] >> 32);
              O[s] = (int)(uint32_t)((uint64_t)key[s] & 0xFFFFFFFFull);
            }
          }
        }
        // the other fields, by list position
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s >= S2) break;
          int c = s * kWave + lane;
          if (c < m) {
            DX[s] = L.sDX[O[s]];
            DY[s] = L.sDY[O[s]];
            LY[s] = L.sLY[O[s]];
            M[s] = L.sM[O[s]];
          }
        }
        WaveSync();
        // check_intersection with the predecessor at insertion time: the
        // nearest earlier element of the sorted list whose list position is
        // smaller (edges that moved in front of it were processed later).
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s >= S2) break;
          int c = s * kWave + lane;
          if (c < m) {
            L.sX[c] = X[s] + DX[s];
            L.sLY[c] = O[s];
          }
        }
        WaveSync();
        bool f = false;
#pragma unroll
        for (int s = 0; s < K; s++) {
          if (s >= S2) break;
          int c = s * kWave + lane;
          if (c < m) {
            int q = c - 1;
            while (q >= 0 && L.sLY[q] > O[s]) q--;
            if (q >= 0 && L.sX[q] > X[s] + DX[s]) f = true;
          }
        }
        flag_isect = __ballot(f) != 0;
      }
      WaveSync();
    }
    n = m;
    if (ends != 0) {
      // the smallest lower_y changes only when an edge ends or moves on
      int mn = kMaxS32;
#pragma unroll
      for (int s = 0; s < K; s++) {
        if (s * kWave >= n) break;
        int p = s * kWave + lane;
        if (p < n) mn = Min32(mn, LY[s]);
      }
      min_ly = DppWaveMin(mn);
    }
    nny = flag_isect ? next_y + (kFixed1 >> kAcc) : min_ly;

    if (sample) {
      tp3 = wall_clock64();
      ph[2] += tp3 - tp2;
    }
    // ---- row completion ------------------------------------------------------
    y = next_y;
    if (draw && (y & 0xFFFF) == 0) flush_rows(row, rows);
    if (sample) {
      tp4 = wall_clock64();
      ph[3] += tp4 - tp3;
    }
    if (y >= stop_fixed) break;

    // ---- insert new edges (insert_new_edges) -----------------------------------
    Fixed nu = pending_upper();
    if (nu <= y) {
      if (!insert_new(y, false)) {
        flags |= 2;
        break;
      }
      nu = pending_upper();
    }
    if (nu > y && nu < nny) nny = nu;
    if (sample) ph[4] += wall_clock64() - tp4;
  }
  finish_band();
  if (!kWrite) {
    // bands the walk never reached are empty
    for (; next_b < nb; next_b++)
      if (lane == 0) snap_at(next_b)->y = kMaxS32;
  }
  n_tiles = WaveSum(n_tiles);
  n_planes = WaveSum(n_planes);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) flags |= __shfl_xor(flags, o, kWave);
  if (lane == 0) {
    uint64_t t_end = wall_clock64();
    uint64_t dt = t_end - t_start;
    // the sampled steps' split, scaled to the whole walk
    uint64_t sampled = 0;
    for (int k = 0; k < 5; k++) sampled += ph[k];
    if (sampled > 0) {
      const double scale = (double)(t_end - tp_loop) / (double)sampled;
      for (int k = 0; k < 5; k++) ph[k] = (uint64_t)((double)ph[k] * scale);
    } else {
      ph[4] = t_end - tp_loop;
    }
    int32_t dt32 = (int32_t)(dt < 0x7FFFFFFF ? dt : 0x7FFFFFFF);
    if (kWrite) {
      JobCov* c = &P.cov[j];
      c->left = pb.l;
      c->top = pb.t;
      c->right = pb.r;
      c->bottom = pb.b;
      atomicAdd(&c->tiles, n_tiles);
      atomicAdd(&c->planes, n_planes);
      atomicMax(&c->max_active, max_active);
      atomicOr(&c->flags, flags);
      atomicAdd(&c->steps, guard);
      atomicMax(&c->time_10ns, dt32);
#pragma unroll
      for (int k = 0; k < 5; k++)
        atomicAdd(&c->phase[k], (int32_t)(ph[k] < 0x7FFFFFFF ? ph[k] : 0x7FFFFFFF));
    } else {
      JobCov* c = &P.cov[j];
      c->left = pb.l;
      c->top = pb.t;
      c->right = pb.r;
      c->bottom = pb.b;
      c->tiles = n_tiles;
      c->planes = n_planes;
      c->max_active = max_active;
      c->flags = flags;
      c->steps = guard;
      c->time_10ns = dt32;
#pragma unroll
      for (int k = 0; k < 5; k++) c->phase[k] = (int32_t)(ph[k] < 0x7FFFFFFF ? ph[k] : 0x7FFFFFFF);
    }
  }
}

// The slot walk's kernel (paths of more than 64 active edges; up to 64 walk as
// a team of one wave, hipr_walk_team.hpp).  Without a queue, workgroup i walks
// item i (the dispatcher hands out items in list order).  With a queue
// (persistent form), a grid sized to the resident waves takes items from an
// atomic counter until the list is exhausted; every wave leaves when the
// counter passes n_walk.
// Bound by instruction issue and by the chain of a path's sub-steps; HBM is
// idle.  Curves + strokes, 4,096 paths at 2048^2: the write pass 144 ms with
// one trapezoid per lane and one row per turn, 88.5 ms now.  The 2-, 4- and
// 8-slot walks are held to 256 registers (two waves per SIMD); a tighter cap
// does not let more waves in, since a walk's LDS (17.6 KB at 2048 px) holds
// nine to a CU: capped to 168 and 128 registers the pass took 90.9 and 91.7
// ms.  The 16-, 32- and 64-slot walks take what they need.
template <int K, int kMode>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(K <= 8 ? 2 : 1)))
WalkKernel(WalkParams P) {
  extern __shared__ int32_t lds[];
  // The 8- and 16-slot walks hold the paths with the widest active lists,
  // the longest sequential walks of a frame: their waves take precedence in
  // instruction issue over the waves of shorter lists on their SIMD.
  if (K >= 8) __builtin_amdgcn_s_setprio(2);
  // one call site, so the item body is inlined once
  auto take = [&]() -> int {
    if (!P.queue) return (int)blockIdx.x;
    int got = 0;
    if (Lane() == 0) got = atomicAdd(P.queue, 1);
    return __builtin_amdgcn_readlane(got, 0);
  };
  for (int wi = take(); wi < P.n_walk; wi = take()) {
    WalkItem<K, kMode>(P, wi, lds);
    if (!P.queue) break;
    WaveSync();
  }
}

// The 32- and 64-slot walks (active lists of up to 2048 and 4096 edges) are
// instantiated in their own translation unit, hipr_walk_wide.hip, which
// compiles beside the main one; they walk unbanded jobs in the count and
// write modes only.  Launches WalkKernel<K, mode> for K = 32 or 64.
hipError_t LaunchWideWalk(int K, int mode, unsigned grid, size_t lds, hipStream_t st,
                          const WalkParams& P);

#ifndef HIPR_TEMPLATES_ONLY
// Grid-stride fill of n int32 words.
__global__ void FillKernel(int32_t* __restrict__ p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Before the write pass: both tile maps at kNoTile, the coverage records, the
// plane pool's counter and the composite's counters at zero.  One launch (four
// fills and a memset were 20 us of a small frame); bound by the maps' bytes,
// which go out 16 per lane (the maps begin at an allocation).
__global__ void PrepareWriteKernel(int32_t* __restrict__ map0, int32_t* __restrict__ map1,
                                   int64_t n_map, int32_t* __restrict__ cov, int64_t n_cov,
                                   int32_t* __restrict__ pool_ctr,
                                   unsigned long long* __restrict__ counters) {
  const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  const int64_t n4 = n_map / 4;
  const int4 none = make_int4(kNoTile, kNoTile, kNoTile, kNoTile);
  for (int64_t i = first; i < n4; i += step) {
    ((int4*)map0)[i] = none;
    ((int4*)map1)[i] = none;
  }
  if (first < n_map - 4 * n4) {
    map0[4 * n4 + first] = kNoTile;
    map1[4 * n4 + first] = kNoTile;
  }
  for (int64_t i = first; i < n_cov; i += step) cov[i] = 0;
  if (first == 0) *pool_ctr = 0;
  for (int64_t i = first; i < kCounterWords; i += step) counters[i] = 0;
}

// Zeroes the coverage records of the listed jobs (before a write pass redoes
// them).
__global__ void ResetCovKernel(const int32_t* __restrict__ list, int n, JobCov* __restrict__ cov) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cov[list[i]] = JobCov{};
}
#endif  // HIPR_TEMPLATES_ONLY

}  // namespace hipr

#endif  // SKITY_HIP_WALK_HPP_
