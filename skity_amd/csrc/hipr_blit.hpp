// hipr_blit.hpp -- analytic trapezoid coverage of one scanline step.
//
// blit_trapezoid_row / blit_aaa_trapezoid_row and their alpha helpers
// (src/render/sw/sw_raster.cc:138-544), evaluated per pixel in closed form and
// spread over the lanes of a wave.
// Coverage goes into LDS delta rows, prefix-summed when the pixel rows are
// complete.  Each 32-bit entry carries two fields whose prefix sums are
// non-negative and below 2^16, so one integer prefix sum S decodes as
// A = S & 0xFFFF, D = S >> 16:
//   D: spans the reference sends straight to RealSpanBuilder (full-height
//      steps whose edges are not too close); each adds (1 << 12) + cover, so
//      D carries the number of such spans above bit 12;
//   A: spans the reference accumulates in SpanBuilder; saturating addition
//      of non-negative alphas equals min(255, sum), so plain sums suffice.
// Spans with cover 0 blend nothing and are skipped.
#ifndef SKITY_HIP_BLIT_HPP_
#define SKITY_HIP_BLIT_HPP_

#include "hipr_common.hpp"

namespace hipr {

typedef uint8_t Alpha;

constexpr int kDirectCount = 1 << 12;  // one direct span, in the D field

// A row covers the visible pixels [left, left + width) of the path's
// canvas.  A span's two delta entries are clamped into [0, width]: deltas left
// of the canvas fold into entry 0 and deltas right of it into entry `width`,
// which no visible pixel's prefix sum reads, so every visible pixel sums the
// same deltas as over the path's full width.
struct RowSink {
  int32_t* d;       // the delta entry of the first visible column
  uint32_t* touch;  // a bit per tile column, from the first visible column's
  int32_t pitch;    // delta entries of a row (16 per tile column and 16 more)
  int32_t left;     // pixel x of delta index 0 (the first visible column)
  int32_t width;    // visible columns; entry `width` is the end-of-row entry
  // Direct spans of cover 0 blend nothing in src-over, and are dropped; a
  // job whose blend mode does change pixels under a transparent source keeps
  // them (they still count as a direct span of the pixel).
  bool keep_zero;
  // Adds v to row r's delta at pixel x (clamped into the row).
  __device__ __forceinline__ void Add(int r, int x, int v) {
    if (v == 0) return;
    const int i = x - left;
    atomicAdd(&d[r * pitch + (i < 0 ? 0 : (i > width ? width : i))], v);
  }
  // Marks the tile columns of row r's deltas at pixels a .. b (clamped into
  // the row) as touched.
  __device__ __forceinline__ void Touch(int r, int a, int b) {
    const int c0 = (left >> 4) - r * (pitch >> 4);
    const int lo = (Min32(Max32(a, left), left + width) >> 4) - c0;
    const int hi = (Min32(Max32(b, left), left + width) >> 4) - c0;
    for (int w = lo >> 5; w <= hi >> 5; w++) {
      const uint32_t from = w == lo >> 5 ? ~0u << (lo & 31) : ~0u;
      const uint32_t to = w == hi >> 5 ? (2u << (hi & 31)) - 1 : ~0u;
      atomicOr(&touch[w], from & to);
    }
  }
  // A one-pixel span of cover v at a visible pixel of row r.
  __device__ __forceinline__ void Pixel(int r, bool direct, int x, int v) {
    if (v == 0 && !(direct && keep_zero)) return;
    const int inc = direct ? (kDirectCount + v) << 16 : v;
    int32_t* e = &d[r * pitch + x - left];
    atomicAdd(e, inc);
    atomicAdd(e + 1, -inc);
  }
};

__device__ __forceinline__ Alpha PartialAlphaA(Alpha a, Alpha full) {
  return (Alpha)((a * full) >> 8);
}
__device__ __forceinline__ Alpha TrapezoidToAlpha(Fixed l1, Fixed l2) {
  Fixed area = (l1 + l2) / 2;
  return (Alpha)(area >> 8);
}
__device__ __forceinline__ Alpha PartialTriangleToAlpha(Fixed a, Fixed b) {
  Fixed area = (a >> 11) * (a >> 11) * (b >> 11);
  return (Alpha)((area >> 8) & 0xFF);
}
__device__ __forceinline__ Fixed ApproxIntersection(Fixed l1, Fixed r1, Fixed l2,
                                                    Fixed r2) {
  if (l1 > r1) {
    Fixed t = l1;
    l1 = r1;
    r1 = t;
  }
  if (l2 > r2) {
    Fixed t = l2;
    l2 = r2;
    r2 = t;
  }
  return (Max32(l1, l2) + Min32(r1, r2)) / 2;
}

// Entry i of compute_alpha_below_line(l, r, dY, full) (sw_raster.cc:343-368),
// R = ceil(r) > 0.
__device__ __forceinline__ Alpha AlphaBelow(int i, int R, Fixed l, Fixed r, Fixed dY,
                                            Alpha full) {
  if (R == 1) return PartialAlphaA(TrapezoidToAlpha(l, r), full);
  Fixed last = r - ((R - 1) << 16);
  Fixed last_h = FixedMul(last, dY);
  if (i == R - 1) return (Alpha)(FixedMul(last, last_h) >> 9);
  if (i == 0) return (Alpha)(full - PartialTriangleToAlpha(kFixed1 - l, dY));
  // alpha16 starts at last_h + dY/2 for i = R-2 and grows by dY per step left.
  Fixed a16 = (Fixed)((uint32_t)(last_h + (dY >> 1)) + (uint32_t)(R - 2 - i) * (uint32_t)dY);
  return (Alpha)((a16 >> 8) & 0xFF);
}
// Entry i of compute_alpha_above_line (sw_raster.cc:312-339).
__device__ __forceinline__ Alpha AlphaAbove(int i, int R, Fixed l, Fixed r, Fixed dY,
                                            Alpha full) {
  if (R == 1) return PartialAlphaA((Alpha)(((R << 17) - l - r) >> 9), full);
  Fixed first = kFixed1 - l;
  Fixed first_h = FixedMul(first, dY);
  if (i == 0) return (Alpha)(FixedMul(first, first_h) >> 9);
  if (i == R - 1) {
    Fixed last = r - ((R - 1) << 16);
    return (Alpha)(full - PartialTriangleToAlpha(last, dY));
  }
  Fixed a16 = (Fixed)((uint32_t)(first_h + (dY >> 1)) + (uint32_t)(i - 1) * (uint32_t)dY);
  return (Alpha)(a16 >> 8);
}

// Cover of pixel x of blit_aaa_trapezoid_row (sw_raster.cc:370-455): `full`
// less what lies left of the left edge (ul at the step's top, ll at its
// bottom) and right of the right edge.  The left edge covers the pixels
// [floor(ul), ceil(ll)) in part, the right edge [floor(ur), ceil(lr)).
__device__ __forceinline__ Alpha TrapezoidPixel(int x, Fixed ul, Fixed ur, Fixed ll, Fixed lr,
                                                Fixed lDY, Fixed rDY, Alpha full) {
  const int uL = FixedFloorToInt(ul), lL = FixedCeilToInt(ll);
  const int uR = FixedFloorToInt(ur), lR = FixedCeilToInt(lr);
  Alpha a = full;
  if (x >= uL && x < lL) {
    Alpha t;
    if (uL + 2 == lL) {
      const Fixed first = IntToFixed(uL) + kFixed1 - ul;
      t = x == uL ? (Alpha)(full - PartialTriangleToAlpha(first, lDY))
                  : PartialTriangleToAlpha(ll - ul - first, lDY);
    } else {
      const Fixed l = ul - IntToFixed(uL), r = ll - IntToFixed(uL);
      t = AlphaBelow(x - uL, FixedCeilToInt(r), l, r, lDY, full);
    }
    a = a > t ? (Alpha)(a - t) : 0;
  }
  if (x >= uR && x < lR) {
    Alpha t;
    if (uR + 2 == lR) {
      const Fixed first = IntToFixed(uR) + kFixed1 - ur;
      t = x == uR ? PartialTriangleToAlpha(first, rDY)
                  : (Alpha)(full - PartialTriangleToAlpha(lr - ur - first, rDY));
    } else {
      const Fixed l = ur - IntToFixed(uR), r = lr - IntToFixed(uR);
      t = AlphaAbove(x - uR, FixedCeilToInt(r), l, r, rDY, full);
    }
    a = a > t ? (Alpha)(a - t) : 0;
  }
  return a;
}

// Number of lanes below this one whose bit is set.
__device__ __forceinline__ int CountBelow(uint64_t m, int base = 0) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)base));
}

// LDS of BlitEdges: two int4 per lane with per-pixel work, and one mark per
// work item of a pass.
struct BlitScratch {
  int4* items;   // 2 x 64
  int32_t* mark; // 64
};
constexpr int kBlitScratchInts = 2 * kWave * 4 + kWave;

// blit_trapezoid_row (sw_raster.cc:457-544) for up to 32 trapezoids, two lanes
// each (`act`; `side` 0 its left edge, 1 its right edge), on delta row `r` of
// their lanes.
//
// A trapezoid is a run of `full` pixels between a left and a right edge, each
// of which covers R pixels in part.  The right edge is the left edge's mirror
// image, in every formula and to the bit (distances are taken from the outer
// pixel boundary), so one lane per edge runs one code path where one lane per
// trapezoid ran two.  An edge that stays within one or two pixels is done by
// its lane as deltas.  A flatter one gives every pixel its own cover
// (TrapezoidPixel), as do all pixels of a trapezoid whose edges share pixels
// (drawn from side 0).  Those pixels, a few for most trapezoids and hundreds
// for a nearly horizontal edge, are laid end to end and handed out one per
// lane, so a wave takes ceil(total / 64) passes over them however unevenly
// they are spread; looping over them per lane takes as many passes as the
// longest one has pixels.
__device__ __forceinline__ void BlitEdges(RowSink& s, const BlitScratch& L, bool act, int side,
                                          int r, Fixed ul, Fixed ur, Fixed ll, Fixed lr, Fixed lDY,
                                          Fixed rDY, Alpha full, bool no_real) {
  const int lane = Lane();
  bool go = act && ul <= ur;
  if (ll > lr) ll = lr = ApproxIntersection(ul, ll, ur, lr);
  go = go && !(ul == ur && ll == lr);
  if (ul > ll) {
    Fixed t = ul;
    ul = ll;
    ll = t;
  }
  if (ur > lr) {
    Fixed t = ur;
    ur = lr;
    lr = t;
  }
  const bool direct = full == 0xFF && !no_real;
  // a span's increment at its first pixel; its end takes it back
  auto inc = [&](int v) -> int {
    if (!direct) return v;
    return v != 0 || s.keep_zero ? (kDirectCount + v) << 16 : 0;
  };
  auto part = [&](Alpha a) -> int { return inc(direct ? a : PartialAlphaA(a, full)); };
  int cnt = 0;
  const Fixed join_left = FixedCeilToFixed(ll), join_rite = FixedFloorToFixed(ur);
  const int x0 = ul >> 16;
  if (go && join_left <= join_rite) {
    const int JL = join_left >> 16, JR = join_rite >> 16;
    // the edge's pixels [from, from + R) and, from its outer end, where it
    // enters (l) and leaves (rr) them
    const int from = side ? JR : x0;
    const int R = side ? FixedCeilToInt(lr) - JR : JL - x0;
    Fixed l = (side ? ur : ul) - IntToFixed(from), rr = (side ? lr : ll) - IntToFixed(from);
    if (side) {
      const Fixed t = IntToFixed(R) - rr;
      rr = IntToFixed(R) - l;
      l = t;
    }
    const Fixed dY = side ? rDY : lDY;
    int inner = 0, outer = 0;  // increments of the pixels next to the run
    if (R == 1) {
      inner = part(TrapezoidToAlpha(kFixed1 - l, kFixed1 - rr));
    } else if (R == 2) {
      outer = inc(PartialTriangleToAlpha(kFixed1 - l, dY));
      inner = inc((Alpha)(full - PartialTriangleToAlpha(rr - kFixed1, dY)));
    } else {
      cnt = Max32(0, Min32(from + R, s.left + s.width) - Max32(from, s.left));
    }
    const int run = JL < JR ? inc(full) : 0;
    const int at = side ? JR : JL, d = side ? 1 : -1;
    const int sg = side ? -1 : 0;  // negates the right edge's increments
    s.Add(r, at, ((run - inner) ^ sg) - sg);
    s.Add(r, at + d, ((inner - outer) ^ sg) - sg);
    s.Add(r, at + 2 * d, (outer ^ sg) - sg);
    s.Touch(r, from, from + R);
  } else if (go && side == 0) {
    const int R = FixedCeilToInt(lr);
    s.Touch(r, x0, R);
    if (R - x0 == 1) {
      const int v = part(TrapezoidToAlpha(ur - ul, lr - ll));
      s.Add(r, x0, v);
      s.Add(r, R, -v);
    } else {
      cnt = Max32(0, Min32(R, s.left + s.width) - Max32(x0, s.left));
    }
  }
  const uint64_t have = __ballot(cnt > 0);
  if (have == 0) return;
  const int incl = ScanSum(cnt);
  const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
  const int start = incl - cnt;
  if (cnt > 0) {
    int4* it = L.items + 2 * CountBelow(have);
    it[0] = make_int4(ul, ur, ll, lr);
    it[1] = make_int4(lDY, rDY, (r << 2) | (side << 1) | (direct ? 1 : 0), start);
  }
  int before = 0;  // lanes whose pixels start before this pass
  for (int base = 0; base < total; base += kWave) {
    // mark where each lane's pixels start; the marks up to a pixel count the
    // lanes up to its own
    L.mark[lane] = 0;
    WaveSync();
    if (cnt > 0 && start >= base && start < base + kWave) L.mark[start - base] = 1;
    WaveSync();
    const uint64_t marks = __ballot(L.mark[lane] != 0);
    const int t = base + lane;
    if (t < total) {
      const int own = CountBelow(marks, before) + (int)((marks >> lane) & 1) - 1;
      const int4 a = L.items[2 * own], b = L.items[2 * own + 1];
      const int x = Max32(FixedFloorToInt((b.z & 2) != 0 ? a.y : a.x), s.left) + (t - b.w);
      const Alpha v = TrapezoidPixel(x, a.x, a.y, a.z, a.w, b.x, b.y, full);
      s.Pixel(b.z >> 2, (b.z & 1) != 0, x, v);
    }
    before += __popcll(marks);
    WaveSync();
  }
}

}  // namespace hipr

#endif  // SKITY_HIP_BLIT_HPP_
