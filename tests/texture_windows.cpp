// Host-side check of the texture backward's window arithmetic
// (window_box.h) over every side a box of window coordinates can have: the
// area that is taken for a window against the exact product, the packed
// word against its fields, the bands' rows against the pool, and a
// footprint's box against its taps.  Prints the number of boxes; exits 1 on
// the first violation.
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "window_box.h"

using namespace dr;

constexpr int kMaxSide = 32767 + kWinCoordMax + 1;  // of coordinates in [-kWinCoordMax, 32767]

static int fail(const char* what, int w, int h, int cap) {
  std::printf("%s: %d x %d, pool %d\n", what, w, h, cap);
  return 1;
}

int main() {
  std::mt19937 rng(7);
  std::uniform_int_distribution<int> side(1, kMaxSide);
  long boxes = 0, fits = 0;
  for (const int cap : {928, 1008, 1024}) {
    for (int w = 1; w <= kMaxSide; ++w) {
      std::vector<int64_t> hs = {1, 2, 3, 16, cap - 1, cap, cap + 1, 32767, 46340, 46341, kMaxSide};
      for (int d = -1; d <= 1; ++d) {
        hs.push_back(cap / w + d);
        // around the products that leave 31 and 32 bits
        hs.push_back((1ll << 31) / w + d);
        hs.push_back((1ll << 32) / w + d);
      }
      for (int i = 0; i < 8; ++i) hs.push_back(side(rng));
      for (const int64_t h64 : hs) {
        if (h64 < 1 || h64 > kMaxSide) continue;
        const int h = (int)h64;
        ++boxes;
        const int64_t area = (int64_t)w * h;
        const int fit = win_fit(w, h, cap);
        if (fit != (area <= cap ? (int)area : 0)) return fail("area", w, h, cap);
        if (fit == 0 || cap >= 1024) continue;
        ++fits;
        for (const int at : {0, 1, cap - fit}) {  // (a window ends inside the pool)
          const int p = win_pack(w, h, at);
          if (p == 0 || win_w(p) != w || win_h(p) != h || win_at(p) != at)
            return fail("packed", w, h, cap);
        }
      }
      const int rows = win_rows(w, cap);
      if (rows != (w <= cap ? cap / w : 0) || (int64_t)rows * w > cap) return fail("rows", w, 0, cap);
    }
  }
  // every coordinate a window can have fits the packed 16-bit boxes, and
  // names the texel it stands for
  for (const int size : {1, 3, 1000, 32767})
    for (int64_t t = -200000; t <= 200000; ++t) {
      const int wrapped = (int)(((t % size) + size) % size);
      const int c = win_coord((int)t, wrapped);
      if (c < -kWinCoordMax || c + 1 > 32767 || ((c % size) + size) % size != wrapped)
        return fail("coordinate", (int)t, size, 0);
    }
  // a footprint's box is that of its taps with a nonzero weight, on either
  // side of the origin
  std::uniform_int_distribution<int> coord(-kWinCoordMax, 32766), bits(0, 15), far(0, 3);
  for (int i = 0; i < 1000000; ++i) {
    const int span = far(rng) ? 20 : kWinCoordMax;  // mostly around the origin
    TapSlot q{};
    q.ix0 = coord(rng) % span; q.ix1 = bits(rng) ? q.ix0 + 1 : coord(rng) % span;
    q.iy0 = coord(rng) % span; q.iy1 = bits(rng) ? q.iy0 + 1 : coord(rng) % span;
    const int m = bits(rng);
    q.w00 = m & 1 ? 0.25f : 0.0f; q.w10 = m & 2 ? 0.25f : 0.0f;
    q.w01 = m & 4 ? 0.25f : 0.0f; q.w11 = m & 8 ? -0.25f : 0.0f;
    int x0, x1, y0, y1;
    slot_box(q, x0, x1, y0, y1);
    if (m == 0) {
      if (x1 >= x0 || y1 >= y0) return fail("box of nothing", q.ix0, q.iy0, 0);
      continue;
    }
    int a0 = 1 << 30, a1 = -(1 << 30), b0 = 1 << 30, b1 = -(1 << 30);
    for (int t = 0; t < 4; ++t) {
      if (!((m >> t) & 1)) continue;
      const int x = t & 1 ? q.ix1 : q.ix0, y = t & 2 ? q.iy1 : q.iy0;
      a0 = x < a0 ? x : a0; a1 = x > a1 ? x : a1;
      b0 = y < b0 ? y : b0; b1 = y > b1 ? y : b1;
    }
    if (x0 != a0 || x1 != a1 || y0 != b0 || y1 != b1) return fail("box", q.ix0, q.iy0, m);
  }
  std::printf("%ld boxes, %ld windows\n", boxes, fits);
  return 0;
}
