// hipr_walk_team.hpp -- the analytic-AA scanline walk of one path by a team of
// one wave per 64 active edges.
//
// The walk itself (what a step does, row bands, delta rows, tile planes) is
// described in hipr_walk.hpp, whose register-slot form holds longer lists in
// one wave.  Here element p of the active edge list lives in lane p % 64 of
// wave p / 64, so a list operation is one wave operation plus, in a team of
// several waves, an exchange of a few words per wave through LDS; y, the list
// length, the next event and the pending edges are the same in every wave.
//
// A team of one wave draws the paths of up to 64 active edges in every mode.
// It is the slot walk without slots: no loops over them, no carries between
// them, the edges that open and close intervals kept between list changes
// (64 polygons on 800x600: walk 1.28 -> 1.10 ms; a page of 16,900 glyphs: 1.15
// -> 0.83 ms; 4.7-5.3 us a step instead of 5.1-5.7 where the device is full).
// Teams of 8 and 16 waves run schedule passes only.  A schedule pass is as
// long as its longest path's steps; there the team's steps are shorter (lists
// of up to 400 edges: 4.5 us against 7 us a step), while drawing by teams
// costs more wave time than it saves: the waves wait at two to a dozen
// barriers a step.
#ifndef SKITY_HIP_WALK_TEAM_HPP_
#define SKITY_HIP_WALK_TEAM_HPP_

#include "hipr_walk.hpp"

namespace hipr {

constexpr int kMaxTeam = 16;  // waves of the largest team

// LDS words: per wave the blit scratch; per list entry five permutation words;
// the delta rows, their touched bits, the touched columns and their end
// values; the tile columns' state; the exchange buffers.
constexpr int kTeamShareInts = 8;  // words a wave shares at a time
__host__ __device__ inline int TeamLdsInts(int NW, int w, int row_ints) {
  return NW * kBlitScratchInts + 5 * NW * kWave + row_ints + WalkTouchInts(row_ints) +
         2 * (row_ints / kTile + 4) + 3 * (w / kTile + 2) + (w / kTile + 3) / 2 +
         2 * NW * kTeamShareInts + NW * kTile;
}

template <int NW, int kMode>
__device__ __forceinline__ void TeamWalkItem(const WalkParams& P, int wi, int32_t* lds) {
  constexpr int CAP = NW * kWave;
  constexpr int kThreads = NW * kWave;
  constexpr bool kWrite = kMode == kWalkWrite;
  constexpr bool kBlit = kMode != kWalkSchedule;
  static_assert(NW == 1 || !kBlit, "teams of several waves only schedule");
  const int lane = Lane();
  const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int me = w * kWave + lane;  // this thread's list element
  // Every wave of the team comes here.
  auto sync = [&]() {
    if (NW == 1) {
      WaveSync();
    } else {
      __syncthreads();
    }
  };
  const uint64_t t_start = wall_clock64();
  const int item = P.walk_list[wi];
  const int j = item >> kBandBits;
  const int rband = kWrite ? (item & (kMaxBands - 1)) : 0;
  const Job job = P.jobs[j];
  const JobGeo geo = P.geo[j];
  const Canvas cv = P.canvases[job.canvas];
  const int path_top = JobPixBounds(geo).t;  // RastePath's start_y
  const PixBounds pb = JobScanBounds(geo);
  const TileRange tr = JobTiles(pb, cv.width, cv.height);
  // a delta row holds the visible columns [ox, ox + W) of the canvas
  const int ox = pb.l > 0 ? pb.l : 0;
  const int W = (pb.r < cv.width ? pb.r : cv.width) - ox;
  int flags = 0;
  int n_tiles = 0, max_active = 0;
  const int nE = geo.edges;
  int32_t* map0 = kWrite ? P.map0 + P.map_base[j] : nullptr;
  int32_t* map1 = kWrite ? P.map1 + P.map_base[j] : nullptr;
  if (pb.empty || tr.ntc == 0 || nE == 0 || W > P.lds_width) {
    if (!pb.empty && W > P.lds_width) flags |= 16;
    if (me == 0 && rband == 0) {
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
  // ---- LDS -----------------------------------------------------------------------
  const int cols_cap = P.lds_width / kTile + 2;
  int32_t* at = lds;
  auto take = [&](int ints) {
    int32_t* p = at;
    at += ints;
    return p;
  };
  int32_t* const wide = take(NW * kBlitScratchInts);  // the waves' blit scratch, or 2 x CAP words
  const BlitScratch blit{(int4*)(wide + w * kBlitScratchInts),
                         wide + w * kBlitScratchInts + 2 * kWave * 4};
  int32_t* const sX = take(CAP);
  int32_t* const sDX = take(CAP);
  int32_t* const sDY = take(CAP);
  int32_t* const sLY = take(CAP);
  int32_t* const sM = take(CAP);
  int4* const iL = (int4*)sX;  // intervals, as in hipr_walk.hpp
  int4* const iR = iL + CAP / 2;
  int2* const iN = (int2*)(iR + CAP / 2);
  int32_t* const shareb = take(2 * NW * kTeamShareInts);
  int32_t* const d = take(P.row_ints);
  uint32_t* const touch = (uint32_t*)take(WalkTouchInts(P.row_ints));
  int32_t* const list = take(P.row_ints / kTile + 4);  // touched columns
  int32_t* const vend = take(P.row_ints / kTile + 4);  // per column: value at its end
  int32_t* const slot0 = take(cols_cap);
  int32_t* const slot1 = take(cols_cap);
  int32_t* const rowsw = take(cols_cap);
  int32_t* const fullw = take((cols_cap + 1) / 2);
  int32_t* const cntb = take(NW * kTile);
  const int ncol = tr.ntc + 1;
  const int row_cap = Min32(P.row_ints / (ncol * kTile), kTile);
  for (int i = me; i < row_cap * ncol * (kTile / 4); i += kThreads)
    ((int4*)d)[i] = make_int4(0, 0, 0, 0);
  for (int i = me; i < tr.ntc; i += kThreads) {
    slot0[i] = -1;
    slot1[i] = -1;
    rowsw[i] = 0;
  }
  for (int i = me; i < (tr.ntc + 1) / 2; i += kThreads) fullw[i] = 0;
  for (int i = me; i < WalkTouchInts(P.row_ints); i += kThreads) touch[i] = 0;
  sync();

  const EdgeRec* E = P.wedges + P.edge_base[j];
  EdgeRec* Q = P.qstate + P.q_base[j] + (int64_t)rband * nE;
  const int64_t pbase = kWrite ? P.plane_base[j] : 0;
  const int pcap = kWrite ? P.plane_cap[j] : 0;
  uint8_t* planes = P.planes;
  const Fixed left_clip = (Fixed)((uint32_t)pb.l << 16);
  const Fixed right_clip = (Fixed)((uint32_t)pb.r << 16);
  const int winding_mask = job.fill == HIPR_FILL_EVEN_ODD ? 1 : -1;
  const int cy0 = pb.t > 0 ? pb.t : 0, cy1 = pb.b < cv.height ? pb.b : cv.height;
  const bool triple = (job.flags & kJobKeepZero) != 0;
  RowSink sink{d + (ox & (kTile - 1)), touch, ncol * kTile, ox, W, triple};

  Fixed X = 0, DX = 0, DY = 0, LY = 0;
  int M = 0;
  int n = 0;
  int n_planes = 0;
  int next_slot = 0, chunk_end = 0;
  int band = -1;

  // ---- exchange ------------------------------------------------------------------
  // Every wave gives up to eight (uniform) words and reads every wave's: lane v
  // holds wave v's.  Two buffers in turn: a wave can be one exchange ahead of
  // another at most.
  int turn_buf = 0;
  struct Share {
    int4 a, b;
  };
  auto share = [&](int4 a, int4 b, bool both) -> Share {
    Share r;
    r.a = a;
    r.b = b;
    if (NW > 1) {
      int4* buf = (int4*)(shareb + turn_buf * NW * kTeamShareInts);
      turn_buf ^= 1;
      if (lane == 0) {
        buf[2 * w] = a;
        if (both) buf[2 * w + 1] = b;
      }
      sync();
      const int v = lane < NW ? lane : 0;
      r.a = buf[2 * v];
      if (both) r.b = buf[2 * v + 1];
    }
    return r;
  };
  const bool mate = lane < NW;  // lane v stands for wave v in an exchange
  auto share_any = [&](int bits) -> int {
    if (NW == 1) return bits;
    const Share r = share(make_int4(bits, 0, 0, 0), make_int4(0, 0, 0, 0), false);
    int any = 0;
#pragma unroll
    for (int k = 0; k < 4; k++)
      any |= __ballot(mate && ((r.a.x >> k) & 1) != 0) != 0 ? 1 << k : 0;
    return any;
  };
  // sum of the waves before this one / of all waves, from lane v's word (scans:
  // never under a lane's condition)
  auto before_sum = [&](int v) -> int {
    return w == 0 ? 0 : __builtin_amdgcn_readlane(ScanSum(mate ? v : 0), w == 0 ? 0 : w - 1);
  };
  auto all_sum = [&](int v) -> int {
    return __builtin_amdgcn_readlane(ScanSum(mate ? v : 0), kWave - 1);
  };

  // ---- what a list change updates ------------------------------------------------
  // The edges that open and close intervals (drawing teams, of one wave) and
  // the neighbouring waves' end elements.
  int nr_all = 0;
  bool open_end = false;
  uint64_t bl = 0, br = 0;
  Fixed pX = kMinS32, pDX = 0;  // lane 63 of the wave before
  auto ends_words = [&]() -> int4 {
    return make_int4(__builtin_amdgcn_readlane(X, kWave - 1),
                     __builtin_amdgcn_readlane(DX, kWave - 1), 0, 0);
  };
  auto take_ends = [&](int4 e) {
    const int pv = w > 0 ? w - 1 : 0;
    pX = w > 0 ? __builtin_amdgcn_readlane(e.x, pv) : kMinS32;
    pDX = w > 0 ? __builtin_amdgcn_readlane(e.y, pv) : 0;
  };
  auto relink = [&]() {
    if (NW > 1) {
      const Share r = share(ends_words(), make_int4(0, 0, 0, 0), false);
      take_ends(r.a);
    }
    if (kBlit) {
      const uint64_t bval = n >= kWave ? ~0ull : (1ull << n) - 1;
      const bool neg = (M & 1) != 0;
      const uint64_t bneg = __ballot(neg) & bval, bpos = bval & ~bneg;
      const int incl = CountBelow(bpos) - CountBelow(bneg) + (neg ? -1 : 1);
      const uint64_t bin = __ballot((incl & winding_mask) != 0) & bval;
      const uint64_t prev = bin << 1;
      bl = bin & ~prev;
      br = bval & ~bin & prev;
      nr_all = __popcll(br);
      open_end = __popcll(bl) != nr_all;
    }
  };

  // ---- tile planes ---------------------------------------------------------------
  // (as in hipr_walk.hpp)
  auto take_planes = [&](bool need0, bool need1, int c) {
    int a0 = 0, a1 = 0;
    if (kWrite) {
      const int req = triple ? (need0 ? 3 : 0) : (need0 ? 1 : 0) + (need1 ? 1 : 0);
      const int rincl = ScanSum(req);
      const int rtot = __builtin_amdgcn_readlane(rincl, kWave - 1);
      a0 = next_slot + rincl - req;
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
    if (need0) slot0[c] = a0;
    if (need1) slot1[c] = a1;
    WaveSync();
  };

  // Finish a band: publish the tile slots and complete the planes (as in
  // hipr_walk.hpp).
  auto finish_band = [&]() {
    if (band < 0) return;
    const int trow = band - tr.tr0;
    const int brows = cv.height - band * kTile;
    const int all_rows = brows >= kTile ? 0xFFFF : (1 << brows) - 1;
    for (int c0 = 0; c0 < tr.ntc; c0 += kWave) {
      const int c = c0 + lane;
      const bool ok = c < tr.ntc;
      uint32_t written = 0;
      int fm = 0;
      if (ok) {
        written = (uint32_t)rowsw[c];
        fm = (fullw[c >> 1] >> (16 * (c & 1))) & 0xFFFF;
      }
      const bool has0 = (written & 0xFFFF) != 0 || fm != 0, has1 = (written >> 16) != 0;
      n_tiles += has0 ? 1 : 0;
      n_planes += triple ? (has0 ? 3 : 0) : (has0 ? 1 : 0) + (has1 ? 1 : 0);
      if (kWrite) {
        const bool solid = fm == all_rows && (written & 0xFFFF) == 0;
        const bool need = fm != 0 && !solid && slot0[ok ? c : 0] < 0;
        if (__ballot(need) != 0) take_planes(need, false, c);
        const int s0 = ok ? slot0[c] : -1, s1 = ok ? slot1[c] : -1;
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
        slot0[c] = -1;
        slot1[c] = -1;
        rowsw[c] = 0;
        if ((c & 1) == 0) fullw[c >> 1] = 0;  // (c + 1 was read with c)
      }
    }
    sync();
  };

  // covers of a pixel whose deltas sum to S (as in hipr_walk.hpp)
  auto covers = [&](int S, uint32_t* first, uint32_t* second, uint32_t* third) {
    const int a = S & 0xFFFF, dd = S >> 16;
    const int av = a > 255 ? 255 : a;
    const int cnt = dd >> 12;  // direct spans
    const bool dir = cnt != 0;
    const int dv = dd & (kDirectCount - 1);
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
  // a tile column's plane row: asks for planes when the column has none
  auto ensure_planes = [&](bool plane0, bool plane1, int c, bool several) {
    bool need0 = plane0 && slot0[c] < 0, need1 = plane1 && slot1[c] < 0;
    if (__ballot(need0 || need1) != 0) {
      // several rows may meet the same column here: one of them asks
      if (several) {
        if (need0) need0 = atomicCAS(&slot0[c], -1, -2) == -1;
        if (need1) need1 = atomicCAS(&slot1[c], -1, -2) == -1;
      }
      take_planes(need0, need1, c);
    }
  };

  // Resolve the `rows` pixel rows from r on (delta rows 0 .. rows - 1, all in
  // one band) and emit their tile rows: the touched columns are summed, 16 at
  // a time, then the columns between take the value at the end of the touched
  // column before them.  The rows lie end to end: a row's deltas add up to
  // zero.
  auto flush_rows = [&](int r, int rows) {
    const int rb = r >> 4;
    if (rb != band) {
      finish_band();
      band = rb;
    }
    const int rowk0 = r & 15;
    const int cols = rows * ncol;
    const int ng = (cols + kWave - 1) / kWave;  // groups of 64 columns (up to 17)
    const float inv = rows > 1 ? __builtin_amdgcn_rcpf((float)ncol) : 0.f;
    auto place = [&](int col, int* row, int* tcol) {
      *row = 0;
      *tcol = col;
      if (rows > 1) {
        // (col < 2^11: a quotient is at least 1 / (2 ncol) from an integer)
        const int q = (int)(((float)col + 0.5f) * inv);
        *row = q;
        *tcol = col - __mul24(q, ncol);
      }
    };
    // lane g: group g's touched columns, how many come before them, and the
    // last touched column before the group
    uint32_t t0 = 0, t1 = 0;
    if (lane < ng) {
      t0 = touch[2 * lane];
      t1 = touch[2 * lane + 1];
    }
    const int cnt = __popc(t0) + __popc(t1);
    const int cincl = ScanSum(cnt);
    const int nt = __builtin_amdgcn_readlane(cincl, kWave - 1);
    const int last = t1 != 0 ? lane * kWave + 63 - __clz((int)t1)
                     : t0 != 0 ? lane * kWave + 31 - __clz((int)t0) : -1;
    const int lastb = ShiftUp(ScanMax(last), -1);
    if (nt == 0) return;
    auto group_mask = [&](int g) -> uint64_t {
      return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)t0, g) |
             (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)t1, g) << 32;
    };
    for (int g = 0; g < ng; g++) {
      const uint64_t T = group_mask(g);
      const int from = __builtin_amdgcn_readlane(cincl - cnt, g);
      if (__builtin_amdgcn_inverse_ballot_w64(T)) list[CountBelow(T, from)] = g * kWave + lane;
    }
    sync();
    int carry = 0;
    for (int b = 0; b < nt; b += kWave / 4) {
      const int ti = b + (lane >> 2), sub = lane & 3;
      const bool held = ti < nt;
      const int col = held ? list[ti] : 0;
      int jrow, tcol;
      place(col, &jrow, &tcol);
      const bool ok = held && tcol < tr.ntc;  // not the end-of-row column
      const int rowk = rowk0 + jrow;
      int4 dv = make_int4(0, 0, 0, 0);
      if (held) {
        int4* dp = (int4*)(d + col * kTile + 4 * sub);
        dv = *dp;
        *dp = make_int4(0, 0, 0, 0);
      }
      const int s1 = dv.x + dv.y, s2 = s1 + dv.z, s3 = s2 + dv.w;
      const int incl = ScanSum(s3);
      const int e = incl - s3 + carry;
      carry += __builtin_amdgcn_readlane(incl, kWave - 1);
      if (held && sub == 3) vend[col] = e + s3;
      // Most rows have only one kind of span in 16 columns: steps of less
      // than a row accumulate, and a step of a whole row sends its spans
      // directly unless edges are close.
      const int v0 = e + dv.x, v1 = e + s1, v2 = e + s2, v3 = e + s3;
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
        uint32_t f, g2, t;
        covers(v0, &f, &g2, &t);
        c0 = f, c1 = g2, c2 = t;
        covers(v1, &f, &g2, &t);
        c0 |= f << 8, c1 |= g2 << 8, c2 |= t << 8;
        covers(v2, &f, &g2, &t);
        c0 |= f << 16, c1 |= g2 << 16, c2 |= t << 16;
        covers(v3, &f, &g2, &t);
        c0 |= f << 24, c1 |= g2 << 24, c2 |= t << 24;
      }
      // the tile row's state over its four lanes: bit 0 a cover in plane 0,
      // bit 1 one in plane 1, bit 2 not full
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
        if ((st & 5) == 1) atomicOr(&fullw[cc >> 1], 1 << (16 * (cc & 1) + rowk));
        const int wr = (plane0 ? 1 << rowk : 0) | (plane1 ? 1 << (16 + rowk) : 0);
        if (wr) atomicOr(&rowsw[cc], wr);
      }
      ensure_planes(sub == 0 && plane0, sub == 0 && plane1, cc, rows > 1);
      if (kWrite) {
        if (plane0) {
          const int cur = slot0[cc];
          if (cur != kNoPlane) {
            uint32_t* pl = (uint32_t*)(planes + (int64_t)cur * kTilePlaneBytes);
            pl[rowk * 4 + sub] = c0;
            if (triple) {
              pl[kTilePlaneBytes / 4 + rowk * 4 + sub] = c1;
              pl[2 * kTilePlaneBytes / 4 + rowk * 4 + sub] = c2;
            }
          }
        }
        if (plane1) {
          const int cur = slot1[cc];
          if (cur != kNoPlane) {
            uint32_t* pl = (uint32_t*)(planes + (int64_t)cur * kTilePlaneBytes);
            pl[rowk * 4 + sub] = c1;
          }
        }
      }
    }
    sync();
    // the other columns
    for (int g = 0; g < ng; g++) {
      const uint64_t T = group_mask(g);
      const int pc = __builtin_amdgcn_readlane(lastb, g);
      if (T != 0 && lane < 2) touch[2 * g + lane] = 0;
      const uint64_t below = T & ((1ull << lane) - 1);
      const int src = below ? g * kWave + kWave - 1 - __builtin_clzll(below) : pc;
      const int v = src >= 0 ? vend[src] : 0;
      int jrow, c;
      place(g * kWave + lane, &jrow, &c);
      const int rowk = rowk0 + jrow;
      const bool rest = g * kWave + lane < cols && c < tr.ntc && ((T >> lane) & 1) == 0 && v != 0;
      if (__ballot(rest) == 0) continue;
      uint32_t f = 0, g2 = 0, t = 0;
      if (rest) covers(v, &f, &g2, &t);
      const bool is_full = !triple && f == 255 && g2 == 0;
      const bool plane0 = rest && !is_full && (triple ? (f | g2 | t) != 0 : f != 0);
      const bool plane1 = rest && !triple && g2 != 0;
      if (rest && is_full) atomicOr(&fullw[c >> 1], 1 << (16 * (c & 1) + rowk));
      if (__ballot(plane0 || plane1) == 0) continue;
      const int cc = rest ? c : 0;
      const int wr = (plane0 ? 1 << rowk : 0) | (plane1 ? 1 << (16 + rowk) : 0);
      if (wr) atomicOr(&rowsw[cc], wr);
      ensure_planes(plane0, plane1, cc, rows > 1);
      if (kWrite) {
        auto put = [&](int slot, uint32_t b) {
          const int x = (int)(b * 0x01010101u);
          ((int4*)(planes + (int64_t)slot * kTilePlaneBytes))[rowk] = make_int4(x, x, x, x);
        };
        if (plane0) {
          const int cur = slot0[cc];
          if (cur != kNoPlane) {
            put(cur, f);
            if (triple) {
              put(cur + 1, g2);
              put(cur + 2, t);
            }
          }
        }
        if (plane1) {
          const int cur = slot1[cc];
          if (cur != kNoPlane) put(cur, g2);
        }
      }
    }
    sync();
  };

  // ---- pending edges ---------------------------------------------------------
  // the next 64, as in hipr_walk.hpp, in every wave alike
  int pp = 0;
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
  auto pending_upper = [&]() -> Fixed {
    if (pp - w_base >= kWave) load_window(pp);
    return __builtin_amdgcn_readlane(w_uy, pp - w_base);
  };
  Fixed nny = kMaxS32;
  Fixed min_ly = kMaxS32;  // smallest lower_y of the active list
  auto store_fields = [&](int c) {
    sX[c] = X;
    sDX[c] = DX;
    sDY[c] = DY;
    sLY[c] = LY;
    sM[c] = M;
  };
  auto load_fields = [&](int c) {
    X = sX[c];
    DX = sDX[c];
    DY = sDY[c];
    LY = sLY[c];
    M = sM[c];
  };

  // Takes the pending edges with upper_y <= y into the active list
  // (insert_new_edges; with an empty list, the initial activation): sorted by
  // (x, dx, index), new edge i goes to P_i + i and list element q to
  // q + #{i : P_i <= q}, with P0 = #{a : x_a <= x_N0} and
  // Pi = max(P(i-1), #{a : x_a < x_Ni}).  The scratch is free on entry.
  // Returns false when the list outgrows the walk.
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
    int mn, least, shift = 0;  // smallest lower_y after y, and of all
    bool crosses = false;
    if (k <= kTile) {
      // a few: lane i of every wave takes new edge i
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
      least = DppWaveMin(mine ? nLY : kMaxS32);
      mn = initial ? DppWaveMin(mine && nLY > y ? nLY : kMaxS32) : least;
      int cnt = 0;
      if (n > 0) {
        for (int i = 0; i < k; i++) {
          const Fixed xi = __builtin_amdgcn_readlane(nX, i);
          const int c = __popcll(__ballot(me < n && (i == 0 ? X <= xi : X < xi)));
          cnt = lane == i ? c : cnt;
        }
        if (me < n) wide[me] = X + DX;
        if (NW > 1 && mine) cntb[w * kTile + lane] = cnt;
        sync();
        if (NW > 1 && mine) {
          cnt = 0;
#pragma unroll
          for (int v = 0; v < NW; v++) cnt += cntb[v * kTile + lane];
        }
      }
      const int pos = ScanMax(mine ? cnt : 0);
      for (int i = 0; i < k; i++) shift += me >= __builtin_amdgcn_readlane(pos, i) ? 1 : 0;
      if (!initial) {
        // check_intersection with the predecessor at insertion: the new edge
        // before it if that sits right there, else the list element before
        const Fixed v = nX + nDX, pv = ShiftUp(v, 0);
        const int ppos = ShiftUp(pos, -1);
        bool f = false;
        if (mine) {
          if (lane > 0 && ppos == pos) {
            f = pv > v;
          } else if (pos > 0) {
            f = wide[pos - 1] > v;
          }
        }
        crosses = __ballot(f) != 0;
      }
      if (me < n) store_fields(me + shift);
      if (w == 0 && mine) {
        const int c = pos + lane;
        sX[c] = nX;
        sDX[c] = nDX;
        sDY[c] = nDY;
        sLY[c] = nLY;
        sM[c] = nM;
      }
    } else {
      // many: one new edge per thread
      const bool mine = me < k;
      Fixed nX = 0, nDX = 0, nDY = 0, nLY = kMaxS32;
      int nM = 0;
      if (mine) {
        const int4* e = (const int4*)&E[pp + me];
        const int4 a = e[0], b = e[1];
        nX = a.x;
        nDX = a.z;
        nDY = a.w;
        nLY = b.z;
        nM = MakeMeta(EdgeWinding(b.w), EdgeIsQuad(b.w), false, pp + me);
        sX[me] = nX;
        sDX[me] = nDX;
      }
      if (me < n) {
        wide[me] = X;
        wide[CAP + me] = X + DX;
      }
      least = DppWaveMin(mine ? nLY : kMaxS32);
      mn = initial ? DppWaveMin(mine && nLY > y ? nLY : kMaxS32) : least;
      sync();
      int r = 0;
      for (int q = 0; q < k; q++) {
        const Fixed xq = sX[q], dxq = sDX[q];
        r += (xq < nX || (xq == nX && (dxq < nDX || (dxq == nDX && q < me)))) ? 1 : 0;
      }
      int top = 1;
      while (2 * top <= n) top *= 2;
      int lo = 0;  // list elements before it
      for (int st = top; st > 0; st >>= 1) {
        const int t = lo + st;
        if (t <= n && (r == 0 ? wide[t - 1] <= nX : wide[t - 1] < nX)) lo = t;
      }
      sync();
      if (mine) {
        sX[r] = nX;
        sDX[r] = nDX;
        sLY[r] = lo;
      }
      sync();
      const int p0 = sLY[0];
      const int pos = Max32(p0, lo);
      bool f = false;
      if (mine && !initial) {
        if (r > 0 && Max32(p0, sLY[r - 1]) == pos) {
          f = sX[r - 1] + sDX[r - 1] > nX + nDX;
        } else if (pos > 0) {
          f = wide[CAP + pos - 1] > nX + nDX;
        }
      }
      if (me < n && me >= p0) {
        // 1 + #{i >= 1 : P_i <= me} (the counts do not decrease from i = 1 on)
        int tk = 1;
        while (2 * tk <= k - 1) tk *= 2;
        int c = 0;
        for (int st = tk; st > 0; st >>= 1) {
          const int t = c + st;
          if (t <= k - 1 && sLY[t] <= me) c = t;
        }
        shift = 1 + c;
      }
      const Share s = share(make_int4(__ballot(f) != 0 ? 1 : 0, mn, least, 0),
                            make_int4(0, 0, 0, 0), false);
      if (NW == 1) sync();
      crosses = __ballot(mate && s.a.x != 0) != 0;
      mn = DppWaveMin(mate ? s.a.y : kMaxS32);
      least = DppWaveMin(mate ? s.a.z : kMaxS32);
      if (me < n) store_fields(me + shift);
      if (mine) {
        const int c = pos + r;
        sX[c] = nX;
        sDX[c] = nDX;
        sDY[c] = nDY;
        sLY[c] = nLY;
        sM[c] = nM;
      }
    }
    sync();
    n += k;
    pp += k;
    if (me < n) load_fields(me);
    if (!initial && crosses) nny = y + (kFixed1 >> kAcc);
    min_ly = Min32(min_ly, least);
    if (mn > y && mn < nny) nny = mn;
    sync();
    relink();
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
    if (me < n) {
      X = a[me];
      DX = a[CAP + me];
      DY = a[2 * CAP + me];
      LY = a[3 * CAP + me];
      M = a[4 * CAP + me];
      if (MetaMoved(M)) Q[MetaIndex(M)] = qs[me];
    }
    const int mn = DppWaveMin(me < n ? LY : kMaxS32);
    const Share s = share(make_int4(mn, 0, 0, 0), make_int4(0, 0, 0, 0), false);
    min_ly = DppWaveMin(mate ? s.a.x : kMaxS32);
    load_window(pp);
    relink();
  } else {
    load_window(0);
    if (!insert_new(y, true)) flags |= 2;
    const Fixed nu = pending_upper();
    if (nu > y && nu < nny) nny = nu;
  }

  const Fixed stop_fixed = IntToFixed(pb.b);
  int guard = 0;  // steps taken
  uint32_t turn = 0;
  // Phase times (10 ns units) of every 16th turn (see hipr_walk.hpp).
  uint64_t ph[5] = {0, 0, 0, 0, 0};
  const uint64_t tp_loop = wall_clock64();
  int next_b = 1;  // next band snapshot to record (count / schedule passes)
  for (;;) {
    if (y >= stop_y) break;  // the next band starts here
    if (!kWrite && next_b < nb && (y & 0xFFFF) == 0 && ((y >> 16) & (kTile - 1)) == 0) {
      const int yrow = y >> 16;
      while (next_b < nb && yrow >= BandStartRow(pb, nb, next_b)) {
        SnapHeader* h = snap_at(next_b);
        if (me == 0) {
          h->y = y;
          h->nny = nny;
          h->pp = pp;
          h->n = n;
        }
        int32_t* a = (int32_t*)(h + 1);
        EdgeRec* qs = (EdgeRec*)(a + 5 * CAP);
        if (me < n) {
          a[me] = X;
          a[CAP + me] = DX;
          a[2 * CAP + me] = DY;
          a[3 * CAP + me] = LY;
          a[4 * CAP + me] = M;
          if (MetaMoved(M)) qs[me] = Q[MetaIndex(M)];
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
    const bool valid = me < n;
    // rows off the canvas are stepped but not drawn
    const bool draw = kBlit && row >= cy0 && row < cy1;
    // ---- several rows at once ----------------------------------------------------
    // From a whole row on, until the first event (an edge ends or begins),
    // every step is one whole row as long as no two edges cross, and the list
    // stays as it is: row i is x + i dx.  Each neighbouring pair moves apart
    // or together linearly, so a list in order now and after `rows` rows is in
    // order on all rows between, and the steps up to there are taken as one.
    // A list of few edges takes 16 rows (a band, as many delta rows as fit)
    // in little more than the time of one.  (Not where edges have ended before
    // the first row, see hipr_walk.hpp.)
    int rows = 1;
    if ((y & 0xFFFF) == 0 && min_ly > y) {
      int most = Min32((nny - 1) >> 16, stop_fixed >> 16) - row;
      if (kWrite && stop_y != kMaxS32) most = Min32(most, (stop_y >> 16) - row);
      if (!kWrite && next_b < nb) {
        // not past the row of the next snapshot
        const int snap_row =
            Max32(BandStartRow(pb, nb, next_b), (row + kTile) & ~(kTile - 1));
        most = Min32(most, snap_row - row);
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
        const Fixed xj = X + __mul24(DX, most);
        const Fixed p0 = ShiftUp(X, pX), pj = ShiftUp(xj, pX + __mul24(pDX, most));
        const bool off = valid && (p0 > X || pj > xj || (uint32_t)(DX + (1 << 23)) >= (1u << 24) ||
                                   (uint32_t)(X + (1 << 30)) >= (1u << 31));
        if (share_any(__ballot(off) != 0 ? 1 : 0) == 0) {
          rows = most;
          next_y = y + rows * kFixed1;
          guard += rows - 1;
        }
      }
    }

    uint64_t tp0 = 0, tp1 = 0, tp2 = 0, tp3 = 0, tp4 = 0;
    if (sample) tp0 = wall_clock64();
    // ---- interval edges, step, order checks ------------------------------------
    const Fixed xo = X, step = DX >> y_shift;
    X = rows > 1 ? xo + __mul24(DX, rows) : xo + step;
    if (draw) {
      const Fixed nxo = ShiftDown(xo, xo), ndx = ShiftDown(DX, DX);
      if (__builtin_amdgcn_inverse_ballot_w64(bl))
        iL[CountBelow(bl)] = make_int4(xo, step, DY, 0);
      if (__builtin_amdgcn_inverse_ballot_w64(br)) {
        const int c = CountBelow(br);
        iR[c] = make_int4(xo, step, DY, me + 1 < n ? kNextCheck : kNextNone);
        iN[c] = make_int2(nxo, ndx);
      }
      if (open_end && me == 0) {
        // open interval at the end of the list (right edge culled away): it
        // runs to the right clip and is emitted as accumulated coverage (see
        // hipr_walk.hpp)
        iR[nr_all] = make_int4(right_clip, 0, 0, kNextClose);
        iN[nr_all] = make_int2(0, 0);
      }
    }
    if (NW > 1 && w > 0) pX = rows > 1 ? pX + __mul24(pDX, rows) : pX + (pDX >> y_shift);
    auto order = [&](bool* bad, bool* cross) {
      const Fixed v = X + DX;
      const Fixed px = ShiftUp(X, pX), pv = ShiftUp(v, w > 0 ? pX + pDX : kMinS32);
      *bad = __ballot(valid && px > X) != 0;
      *cross = __ballot(valid && pv > v) != 0;
    };
    bool ends, bad, cross;
    {
      const bool e0 = __ballot(valid && LY <= next_y) != 0;
      bool b0, c0;
      order(&b0, &c0);
      const int any = share_any((e0 ? 1 : 0) | (b0 ? 2 : 0) | (c0 ? 4 : 0));
      ends = (any & 1) != 0;
      bad = (any & 2) != 0;
      cross = (any & 4) != 0;
    }
    // ---- the step's trapezoids -------------------------------------------------
    if (draw) {
      WaveSync();
      const int nr = nr_all + (open_end ? 1 : 0);
      if (open_end) flags |= 8;
      // two lanes (left and right edge) per interval and row (rows > 1: t / nr
      // by a product; t < 2^13, and a quotient is at least 1 / (2 nr) from an
      // integer)
      const int total = nr * rows;
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
          l = iL[k];
          r = iR[k];
          nx = iN[k];
          if (k > 0) q = iR[k - 1];
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
        const bool close_next = r.w == kNextClose ||
                                (r.w == kNextCheck && (rxn + kFixed1 >= nx.x - Abs32(nx.y)));
        const bool no_real = full == 0xFF && (close_prev || close_next);
        BlitEdges(sink, blit, act, lane & 1, jr, left, right, next_left, next_right, l.z, r.z,
                  full, no_real);
      }
      sync();
    }

    if (sample) {
      tp1 = wall_clock64();
      ph[0] += tp1 - tp0;
    }
    // ---- quad updates ------------------------------------------------------------
    bool dead = false;
    if (ends) {
      bool flip = false;
      if (valid && LY <= next_y && MetaQuad(M)) {
        // while (lower_y <= next_y) { KeepContinuous; UpdateQuad } with
        // KeepContinuous taking the edge's current x and y
        // (sw_raster.cc:628-638, sw_edge.cc:294-297).
        const int idx = MetaIndex(M);
        EdgeRec e;
        {
          const int4* src = (const int4*)(MetaMoved(M) ? (const EdgeRec*)&Q[idx] : &E[idx]);
          int4* dst = (int4*)&e;
          const int4 q0 = src[0], q1 = src[1], q2 = src[2], q3 = src[3];
          dst[0] = q0;
          dst[1] = q1;
          dst[2] = q2;
          dst[3] = q3;
        }
        Fixed sy = next_y;
        Fixed cx = X;
        while (LY <= next_y && EdgeCurveCount(e.packed) > 0) {
          e.snapped_x = cx;
          if (!UpdateQuad(&e, sy)) break;
          cx = e.x;
          sy = e.upper_y;
          DX = e.dx;
          DY = e.dy;
          LY = e.lower_y;
        }
        X = cx;
        const int m1 = MakeMeta(EdgeWinding(e.packed), true, true, idx);
        flip = ((m1 ^ M) & 1) != 0;
        M = m1;
        Q[idx] = e;
      }
      const int st = (__ballot(valid && LY <= next_y) != 0 ? 1 : 0) |
                     (__ballot(flip) != 0 ? 2 : 0);
      const Share s = share(ends_words(), make_int4(st, 0, 0, 0), true);
      dead = __ballot(mate && (s.b.x & 1) != 0) != 0;
      flip = __ballot(mate && (s.b.x & 2) != 0) != 0;
      if (!dead) {
        // every edge lives on: check the order in place
        take_ends(s.a);
        bool b0, c0;
        order(&b0, &c0);
        const int mn = DppWaveMin(valid ? LY : kMaxS32);
        const Share s2 = share(make_int4((b0 ? 1 : 0) | (c0 ? 2 : 0), mn, 0, 0),
                               make_int4(0, 0, 0, 0), false);
        bad = __ballot(mate && (s2.a.x & 1) != 0) != 0;
        cross = __ballot(mate && (s2.a.x & 2) != 0) != 0;
        min_ly = DppWaveMin(mate ? s2.a.y : kMaxS32);
        if (flip && !bad) relink();
      }
    }

    if (sample) {
      tp2 = wall_clock64();
      ph[1] += tp2 - tp1;
    }
    // ---- survivors, stable x order, intersection checks ------------------------
    if (dead || bad) {
      const bool sv = valid && LY > next_y;
      const uint64_t b = __ballot(sv);
      const Share s = share(make_int4(__popcll(b), 0, 0, 0), make_int4(0, 0, 0, 0), false);
      const int m = all_sum(s.a.x);
      const int place = CountBelow(b, before_sum(s.a.x));
      if (sv) store_fields(place);
      sync();
      const bool in = me < m;
      bool f = false, g = false;
      if (in) {
        load_fields(me);
        if (me > 0) {
          const Fixed px = sX[me - 1], pdx = sDX[me - 1];
          f = px > X;
          g = px + pdx > X + DX;
        }
      }
      const int mn = DppWaveMin(in ? LY : kMaxS32);
      // (the largest x up to here, for the re-sort)
      const int hi = ScanMax(in ? X : kMinS32);
      const Share s2 = share(make_int4((__ballot(f) != 0 ? 1 : 0) | (__ballot(g) != 0 ? 2 : 0), mn,
                                       __builtin_amdgcn_readlane(hi, kWave - 1), 0),
                             make_int4(0, 0, 0, 0), false);
      min_ly = DppWaveMin(mate ? s2.a.y : kMaxS32);
      bad = __ballot(mate && (s2.a.x & 1) != 0) != 0;
      cross = __ballot(mate && (s2.a.x & 2) != 0) != 0;
      if (bad) {
        // Stable re-sort by x.  The elements that stand behind a larger one
        // (the movers, few of the list) are taken out, which leaves the
        // others in order; each of those then counts the movers before it,
        // and each mover the elements after it.
        const int before =
            w == 0 ? kMinS32
                   : __builtin_amdgcn_readlane(ScanMax(mate ? s2.a.z : kMinS32), w == 0 ? 0 : w - 1);
        const int top = Max32(ShiftUp(hi, kMinS32), before);
        const bool mv = in && X < top;
        const uint64_t mb = __ballot(mv);
        const Share s3 = share(make_int4(__popcll(mb), 0, 0, 0), make_int4(0, 0, 0, 0), false);
        const int nm = all_sum(s3.a.x);
        const int idx = CountBelow(mb, before_sum(s3.a.x));  // movers before this element
        int rank = me - idx;
        int32_t* mvx = wide;
        int32_t* mvp = wide + CAP;
        int32_t* after = wide + 2 * CAP;
        if (mv) {
          mvx[idx] = X;
          mvp[idx] = me;
        }
        if (me < nm) after[me] = 0;
        sync();
        for (int i0 = 0; i0 < nm; i0 += kWave) {
          const int kk = Min32(kWave, nm - i0);
          const int src = i0 + (lane < kk ? lane : 0);
          const Fixed mx = mvx[src];
          const int mp = mvp[src];
          int cnt = 0;
          for (int i = 0; i < kk; i++) {
            const Fixed xi = __builtin_amdgcn_readlane(mx, i);
            const int pi = __builtin_amdgcn_readlane(mp, i);
            const bool gt = in && (X > xi || (X == xi && me > pi));
            rank += gt ? 1 : 0;
            const int c = __popcll(__ballot(gt));
            cnt = lane == i ? c : cnt;
          }
          if (NW == 1) {
            if (lane < kk) after[i0 + lane] = cnt;
          } else {
            if (lane < kk) atomicAdd(&after[i0 + lane], cnt);
          }
        }
        sync();
        if (mv) rank = m - 1 - after[idx];
        // every field to its rank, with the list position and the next x
        if (in) {
          store_fields(rank);
          mvx[rank] = me;
          mvp[rank] = X + DX;
        }
        sync();
        // check_intersection with the predecessor at insertion time: the
        // nearest earlier element of the sorted list whose list position is
        // smaller (edges that moved in front of it were processed later).
        // That is the element right before for most; the others look further
        // only if none of those crosses.
        bool hit = false, far = false;
        int pos = 0;
        Fixed v = 0;
        if (in) {
          load_fields(me);
          pos = mvx[me];
          v = mvp[me];
          if (me > 0) {
            if (mvx[me - 1] > pos) {
              far = true;
            } else {
              hit = mvp[me - 1] > v;
            }
          }
        }
        int any = share_any((__ballot(hit) != 0 ? 1 : 0) | (__ballot(far) != 0 ? 2 : 0));
        if (any == 2) {
          if (far) {
            int q = me - 2;
            while (q >= 0 && mvx[q] > pos) q--;
            hit = q >= 0 && mvp[q] > v;
          }
          any = share_any(__ballot(hit) != 0 ? 1 : 0);
        }
        cross = (any & 1) != 0;
      }
      n = m;
      sync();
      relink();
    }
    nny = cross ? next_y + (kFixed1 >> kAcc) : min_ly;

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
      if (me == 0) snap_at(next_b)->y = kMaxS32;
  }
  n_tiles = WaveSum(n_tiles);
  n_planes = WaveSum(n_planes);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) flags |= __shfl_xor(flags, o, kWave);
  if (NW > 1) {
    const Share s = share(make_int4(n_tiles, n_planes, flags, 0), make_int4(0, 0, 0, 0), false);
    n_tiles = all_sum(s.a.x);
    n_planes = all_sum(s.a.y);
    flags = 0;
#pragma unroll
    for (int v = 0; v < NW; v++) flags |= __builtin_amdgcn_readlane(s.a.z, v);
  }
  if (me == 0) {
    uint64_t t_end = wall_clock64();
    uint64_t dt = t_end - t_start;
    // the sampled turns' split, scaled to the whole walk
    uint64_t sampled = 0;
    for (int k = 0; k < 5; k++) sampled += ph[k];
    if (sampled > 0) {
      const double scale = (double)(t_end - tp_loop) / (double)sampled;
      for (int k = 0; k < 5; k++) ph[k] = (uint64_t)((double)ph[k] * scale);
    } else {
      ph[4] = t_end - tp_loop;
    }
    int32_t dt32 = (int32_t)(dt < 0x7FFFFFFF ? dt : 0x7FFFFFFF);
    JobCov* c = &P.cov[j];
    c->left = pb.l;
    c->top = pb.t;
    c->right = pb.r;
    c->bottom = pb.b;
    if (kWrite) {
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

// Without a queue, workgroup i walks item i (the dispatcher hands out items in
// list order).  With a queue (persistent form), a grid sized to the resident
// teams takes items from an atomic counter until the list is exhausted; every
// team leaves when the counter passes n_walk.
// Held to 168 registers, three waves per SIMD: the drawing walk takes them
// without spilling, and its LDS allows about as many.
template <int NW, int kMode>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(3)))
TeamWalkKernel(WalkParams P) {
  extern __shared__ int32_t lds[];
  // one call site, so the item body is inlined once
  auto next = [&]() -> int {
    if (!P.queue) return (int)blockIdx.x;
    if (NW == 1) {
      int got = 0;
      if (Lane() == 0) got = atomicAdd(P.queue, 1);
      return __builtin_amdgcn_readlane(got, 0);
    }
    __syncthreads();
    if (threadIdx.x == 0) lds[0] = atomicAdd(P.queue, 1);
    __syncthreads();
    const int got = __builtin_amdgcn_readfirstlane(lds[0]);
    __syncthreads();
    return got;
  };
  for (int wi = next(); wi < P.n_walk; wi = next()) {
    TeamWalkItem<NW, kMode>(P, wi, lds);
    if (!P.queue) break;
    WaveSync();
  }
}

}  // namespace hipr

#endif  // SKITY_HIP_WALK_TEAM_HPP_
