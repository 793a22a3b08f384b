// Integer arithmetic of the texture backward's LDS windows (k_tex_bwd_win,
// k_tex_bwd_many in texture.hip), shared with a host-side check over every
// box size the window coordinates allow (tests/texture_windows.cpp).
#pragma once

#ifdef __HIPCC__
#define DR_WB_FN __host__ __device__ __attribute__((always_inline)) inline
#else
#define DR_WB_FN inline
#endif

namespace dr {

// The wrap mode's window coordinates are the texel coordinates before the
// wrap (reduced to texels when the window is written out), so a footprint
// across the texture's border, and a tiled texture's pixels on both sides of
// a repeat, stay neighbours: with wrapped coordinates their box spans the
// texture and no window holds it.  Coordinates too far out for the packed
// 16-bit boxes are taken wrapped, which is the same texel.
constexpr int kWinCoordMax = 32000;
DR_WB_FN int win_coord(int t, int wrapped) {
  return (unsigned)t + kWinCoordMax <= 2u * kWinCoordMax ? t : wrapped;
}

// One bilinear footprint on one level, in window coordinates.
struct TapSlot {
  int k;         // level
  float scale;   // (1 - frac) or frac; 0 = unused
  int ix0, ix1, iy0, iy1;
  float w00, w10, w01, w11;
};

// The box of a footprint's taps with a nonzero weight (x1 < x0: none).
// Coordinates may be negative: maxima that began at -1 stretched every box
// left of or above the origin to it, and no window held such a box (bilinear
// wrap, 4 x 1000^2 x 3, uv shifted by -2 repeats: 349 us a pass, now 230 as
// without the shift; trilinear, 2 x 768^2 x 16: 541 -> 308).
DR_WB_FN void slot_box(const TapSlot& q, int& x0, int& x1, int& y0, int& y1) {
  const bool c0 = q.w00 != 0.0f || q.w01 != 0.0f, c1 = q.w10 != 0.0f || q.w11 != 0.0f;
  const bool r0 = q.w00 != 0.0f || q.w10 != 0.0f, r1 = q.w01 != 0.0f || q.w11 != 0.0f;
  const int lo = -0x7fffffff, hi = 0x7fffffff;
  const int xa = c0 ? q.ix0 : hi, xb = c1 ? q.ix1 : hi, ya = r0 ? q.iy0 : hi, yb = r1 ? q.iy1 : hi;
  x0 = xa < xb ? xa : xb;
  y0 = ya < yb ? ya : yb;
  const int xc = c0 ? q.ix0 : lo, xd = c1 ? q.ix1 : lo, yc = r0 ? q.iy0 : lo, yd = r1 ? q.iy1 : lo;
  x1 = xc > xd ? xc : xd;
  y1 = yc > yd ? yc : yd;
}

// Texels of a w x h box (0 x 0: no box) when a pool of `cap` texels holds it,
// else 0.  A side of wrap coordinates is at most 32767 + kWinCoordMax + 1 =
// 64768, so the product of two does not fit 32 bits: the sides are held to
// the pool first.
DR_WB_FN int win_fit(int w, int h, int cap) {
  if (w > cap || h > cap) return 0;
  return w * h <= cap ? w * h : 0;
}

// A window's width, height and place in the pool (all below 1024, at >= 0)
// in one word; 0 is no window.
DR_WB_FN int win_pack(int w, int h, int at) { return w | (h << 10) | ((at + 1) << 20); }
DR_WB_FN int win_w(int p) { return p & 0x3ff; }
DR_WB_FN int win_h(int p) { return (p >> 10) & 0x3ff; }
DR_WB_FN int win_at(int p) { return (p >> 20) - 1; }

// Whole rows of a box w texels wide that the pool holds (0: too wide).
DR_WB_FN int win_rows(int w, int cap) { return w <= cap ? cap / w : 0; }

}  // namespace dr
