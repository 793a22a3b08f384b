// texture: mip pyramid, nearest / bilinear / mip-nearest / trilinear / cube
// sampling, and one fused backward per filter (d_tex or d_pyramid scatter,
// d_uv, d_uvDA and the mip-bias gradient in a single pass).
//
// Semantics follow Sources/MLXDiffRast/Texture.swift of the reference:
//   boundary modes     :336-354       bilinear   :359-403, :407-521
//   nearest            :545-605       cube       :616-738
//   LOD + levels       :764-790       mip fwd    :795-863
//   mip backward       :870-1102      pyramid    :144-161 (2x2 mean)
//   mip bias fold      :104-126 (uvDA * 2^map * 2^bias, folded in-kernel)
// The pyramid is built once per distinct texture (Nt = 1 serves every
// image), not once per broadcast copy; d_tex of a shared texture is the sum
// over images, as MLX's broadcast backward gives.
#include <mutex>
#include <string>
#include <type_traits>

#include "common.h"
#include "window_box.h"

namespace dr {

constexpr int kMaxLevels = 16;

// Pyramid geometry.  Level 0 is the texture itself; levels 1..L-1 live in
// one buffer, level-major, each [Nt, Hk, Wk, C].
struct MipDesc {
  int L;
  int h[kMaxLevels];
  int w[kMaxLevels];
  int64_t off[kMaxLevels];  // float offset of level k (k >= 1) in the pyramid buffer
  int64_t nc;               // Nt * C
};

// Level k's size and pyramid offset computed from level 0 (every level
// halves both sizes exactly), so a per-lane level never indexes the
// descriptor arrays in kernel-argument memory.  Valid for 0 <= k < L.
__device__ __forceinline__ int mip_h(const MipDesc& m, int k) { return m.h[0] >> k; }
__device__ __forceinline__ int mip_w(const MipDesc& m, int k) { return m.w[0] >> k; }
__device__ __forceinline__ int64_t mip_off(const MipDesc& m, int k) {
  // sum_{j=1}^{k-1} Nt*C*(H*W / 4^j) = Nt*C*(H*W - H_{k-1}*W_{k-1}) / 3
  const int j = k > 0 ? k - 1 : 0;
  const uint64_t a = (uint64_t)(uint32_t)m.h[0] * (uint32_t)m.w[0];
  if (a < (1ull << 32)) {  // 32-bit arithmetic (uniform branch)
    const uint32_t b = ((uint32_t)m.h[0] >> j) * ((uint32_t)m.w[0] >> j);
    return m.nc * (int64_t)(((uint32_t)a - b) / 3u);
  }
  const uint64_t b = (uint64_t)(m.h[0] >> j) * (uint64_t)(m.w[0] >> j);
  return m.nc * (int64_t)((a - b) / 3);
}

// Texture.swift:336-354.
__device__ __forceinline__ int apply_boundary(int t, int size, int mode, float& oob) {
  if (mode == DR_BOUNDARY_ZERO) {
    if (t < 0 || t >= size) {
      oob = 1.0f;
      return 0;
    }
    oob = 0.0f;
    return t;
  }
  if (mode == DR_BOUNDARY_CLAMP) {
    oob = 0.0f;
    return t < 0 ? 0 : (t >= size ? size - 1 : t);
  }
  oob = 0.0f;
  int r = t % size;
  if (r < 0) r += size;
  return r;
}

// t mod size and (t + 1) mod size, both in [0, size).  While |t| < 2^22 the
// quotient comes from a float product whose error is below one (t is exact
// in fp32, the reciprocal good to an ulp), corrected by one step; the
// integer remainder it replaces is a 25-instruction sequence per tap
// (bilinear wrap, 4 x 1000^2 x 3: forward 40 -> 38 us).
__device__ __forceinline__ void wrap_pair(int t, int size, int& i0, int& i1) {
  if ((unsigned)t + (1u << 22) < (1u << 23)) {
    const int q = f2i(floorf((float)t * __builtin_amdgcn_rcpf((float)size)));
    int r = t - q * size;
    r += r < 0 ? size : 0;
    r -= r >= size ? size : 0;
    i0 = r;
    i1 = r + 1 == size ? 0 : r + 1;
  } else {
    float unused;
    i0 = apply_boundary(t, size, DR_BOUNDARY_WRAP, unused);
    i1 = apply_boundary(inc(t), size, DR_BOUNDARY_WRAP, unused);
  }
}

struct Bilin {
  int ix0, ix1, iy0, iy1;
  int tx0, ty0;  // ix0, iy0 before the boundary mode
  float fx, fy, m00, m10, m01, m11, w00, w10, w01, w11;
};

// The bilinear footprint of Texture.swift:372-391 (and its copies).
__device__ __forceinline__ Bilin bilin(float u, float v, int Wk, int Hk, int mode) {
  Bilin b;
  const float tx = u * (float)Wk - 0.5f;
  const float ty = v * (float)Hk - 0.5f;
  const int tx0 = f2i(floorf(tx)), ty0 = f2i(floorf(ty));
  const int tx1 = inc(tx0), ty1 = inc(ty0);
  b.fx = tx - (float)tx0;
  b.fy = ty - (float)ty0;
  b.tx0 = tx0;
  b.ty0 = ty0;
  float ox0 = 0.0f, ox1 = 0.0f, oy0 = 0.0f, oy1 = 0.0f;
  if (mode == DR_BOUNDARY_WRAP) {
    wrap_pair(tx0, Wk, b.ix0, b.ix1);
    wrap_pair(ty0, Hk, b.iy0, b.iy1);
  } else {
    b.ix0 = apply_boundary(tx0, Wk, mode, ox0);
    b.ix1 = apply_boundary(tx1, Wk, mode, ox1);
    b.iy0 = apply_boundary(ty0, Hk, mode, oy0);
    b.iy1 = apply_boundary(ty1, Hk, mode, oy1);
  }
  b.m00 = (1.0f - ox0) * (1.0f - oy0);
  b.m10 = (1.0f - ox1) * (1.0f - oy0);
  b.m01 = (1.0f - ox0) * (1.0f - oy1);
  b.m11 = (1.0f - ox1) * (1.0f - oy1);
  const float fx = b.fx, fy = b.fy;
  b.w00 = (1.0f - fx) * (1.0f - fy) * (1.0f - ox0) * (1.0f - oy0);
  b.w10 = (fx) * (1.0f - fy) * (1.0f - ox1) * (1.0f - oy0);
  b.w01 = (1.0f - fx) * (fy) * (1.0f - ox0) * (1.0f - oy1);
  b.w11 = (fx) * (fy) * (1.0f - ox1) * (1.0f - oy1);
  return b;
}

// The nearest texel as a one-tap footprint (Texture.swift:555-571).
__device__ __forceinline__ Bilin nearest_tap(float u, float v, int Wk, int Hk, int mode) {
  Bilin b;
  float ox, oy;
  b.tx0 = f2i(floorf(u * (float)Wk));
  b.ty0 = f2i(floorf(v * (float)Hk));
  b.ix0 = b.ix1 = apply_boundary(b.tx0, Wk, mode, ox);
  b.iy0 = b.iy1 = apply_boundary(b.ty0, Hk, mode, oy);
  b.fx = b.fy = 0.0f;
  b.w00 = b.m00 = b.m10 = b.m01 = b.m11 = (1.0f - ox) * (1.0f - oy);
  b.w10 = b.w01 = b.w11 = 0.0f;
  return b;
}

// Texture.swift:616-672: cube face + clamped bilinear footprint.
__device__ __forceinline__ int cube_bilin(float x, float y, float z, int Wt, int Ht, Bilin& b) {
  const float ax = fabsf(x), ay = fabsf(y), az = fabsf(z);
  int face;
  float sc, tc, ma;
  if (ax >= ay && ax >= az) {
    ma = ax;
    if (x > 0.0f) { face = 0; sc = -z; tc = -y; }
    else          { face = 1; sc = z;  tc = -y; }
  } else if (ay >= az) {
    ma = ay;
    if (y > 0.0f) { face = 2; sc = x; tc = z; }
    else          { face = 3; sc = x; tc = -z; }
  } else {
    ma = az;
    if (z > 0.0f) { face = 4; sc = x;  tc = -y; }
    else          { face = 5; sc = -x; tc = -y; }
  }
  const float inv_ma = 1.0f / ma;
  const float u = (sc * inv_ma + 1.0f) * 0.5f;
  const float v = (tc * inv_ma + 1.0f) * 0.5f;
  const float txr = u * (float)Wt - 0.5f;
  const float tyr = v * (float)Ht - 0.5f;
  const int tx0 = f2i(floorf(txr)), ty0 = f2i(floorf(tyr));
  const int tx1 = inc(tx0), ty1 = inc(ty0);
  const float fx = txr - (float)tx0, fy = tyr - (float)ty0;
  b.fx = fx;
  b.fy = fy;
  b.ix0 = max(0, min(Wt - 1, tx0));
  b.ix1 = max(0, min(Wt - 1, tx1));
  b.iy0 = max(0, min(Ht - 1, ty0));
  b.iy1 = max(0, min(Ht - 1, ty1));
  b.m00 = b.m10 = b.m01 = b.m11 = 1.0f;
  b.w00 = (1.0f - fx) * (1.0f - fy);
  b.w10 = fx * (1.0f - fy);
  b.w01 = (1.0f - fx) * fy;
  b.w11 = fx * fy;
  return face;
}

// Texture.swift:764-790 on the bias-folded derivatives.
struct Lod {
  int k0, k1;
  float frac;
};

__device__ __forceinline__ Lod mip_lod(float4 da, int Ht, int Wt, int L, bool linear) {
  const float sx = da.x * (float)Wt, sy = da.y * (float)Wt;
  const float tx = da.z * (float)Ht, ty = da.w * (float)Ht;
  const float rho_sq = fmaxf(sx * sx + tx * tx, sy * sy + ty * ty);
  float lod = 0.5f * log2f(fmaxf(rho_sq, 1e-20f));
  lod = fmaxf(0.0f, fminf((float)(L - 1), lod));
  Lod r;
  if (linear) {
    r.k0 = f2i(floorf(lod));
    r.k1 = min(r.k0 + 1, L - 1);
    r.frac = lod - (float)r.k0;
  } else {
    r.k0 = min(f2i(floorf(lod + 0.5f)), L - 1);
    r.k1 = r.k0;
    r.frac = 0.0f;
  }
  return r;
}

// uvDA * (2^map * 2^bias) (Texture.swift:109-126).  scale_bias = 2^bias.
__device__ __forceinline__ float bias_scale(const float* __restrict__ bias_map, int64_t pix,
                                            float scale_bias, bool has_bias) {
  if (bias_map) {
    const float s = exp2f(bias_map[pix]);
    return has_bias ? s * scale_bias : s;
  }
  return scale_bias;
}

template <int CT>
__device__ __forceinline__ int dimC(int C) { return CT > 0 ? CT : C; }

// Loads channels [0,C) of one texel.
template <int CT>
__device__ __forceinline__ void load_texel(const float* __restrict__ p, int C, float* out) {
  if (CT == 4) {
    const float4 q = *reinterpret_cast<const float4*>(p);
    out[0] = q.x; out[1] = q.y; out[2] = q.z; out[3] = q.w;
  } else {
#pragma unroll
    for (int c = 0; c < dimC<CT>(C); ++c) out[c] = p[c];
  }
}

constexpr int kMaxC = 4;  // register arrays for compile-time C; larger C uses CT = 0

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------

template <int FILTER, bool CUBE, int CT>
__device__ __forceinline__ void tex_fwd_px(
    const float* __restrict__ tex, const float* __restrict__ pyr, const MipDesc& md,
    int64_t tex_stride, int Ht, int Wt, int C_, const float* __restrict__ uv,
    const float* __restrict__ uv_da, const float* __restrict__ bias_map, float scale_bias,
    int has_bias, int boundary, int64_t P, int n, float* __restrict__ out, int64_t pix) {
  static_assert(CT >= 1 && CT <= kMaxC, "more channels: k_tex_fwd_many");
  if (pix >= P) return;
  const int C = dimC<CT>(C_);
  float* o = out + pix * C;
  if (CUBE) {  // Texture.swift:638-684
    const float x = uv[pix * 3 + 0], y = uv[pix * 3 + 1], z = uv[pix * 3 + 2];
    Bilin b;
    const int face = cube_bilin(x, y, z, Wt, Ht, b);
    const float* fb = tex + n * tex_stride + (int64_t)face * Ht * Wt * C;
    for (int c = 0; c < C; ++c) {
      const float t00 = fb[((int64_t)b.iy0 * Wt + b.ix0) * C + c];
      const float t10 = fb[((int64_t)b.iy0 * Wt + b.ix1) * C + c];
      const float t01 = fb[((int64_t)b.iy1 * Wt + b.ix0) * C + c];
      const float t11 = fb[((int64_t)b.iy1 * Wt + b.ix1) * C + c];
      o[c] = b.w00 * t00 + b.w10 * t10 + b.w01 * t01 + b.w11 * t11;
    }
    return;
  }
  const float2 uvp = ld_nt2(uv + pix * 2);
  if (FILTER == DR_FILTER_NEAREST) {  // Texture.swift:545-572
    const int tx = f2i(floorf(uvp.x * (float)Wt));
    const int ty = f2i(floorf(uvp.y * (float)Ht));
    float ox, oy;
    const int ix = apply_boundary(tx, Wt, boundary, ox);
    const int iy = apply_boundary(ty, Ht, boundary, oy);
    const float mask = (1.0f - ox) * (1.0f - oy);
    const float* tp = tex + n * tex_stride + ((int64_t)iy * Wt + ix) * C;
    for (int c = 0; c < C; ++c) o[c] = tp[c] * mask;
    return;
  }
  if (FILTER == DR_FILTER_LINEAR) {  // Texture.swift:359-403
    const Bilin b = bilin(uvp.x, uvp.y, Wt, Ht, boundary);
    const float* tb = tex + n * tex_stride;
    float t00[kMaxC], t10[kMaxC], t01[kMaxC], t11[kMaxC];
    load_texel<CT>(tb + ((int64_t)b.iy0 * Wt + b.ix0) * C, C, t00);
    load_texel<CT>(tb + ((int64_t)b.iy0 * Wt + b.ix1) * C, C, t10);
    load_texel<CT>(tb + ((int64_t)b.iy1 * Wt + b.ix0) * C, C, t01);
    load_texel<CT>(tb + ((int64_t)b.iy1 * Wt + b.ix1) * C, C, t11);
#pragma unroll
    for (int c = 0; c < CT; ++c)
      o[c] = b.w00 * t00[c] + b.w10 * t10[c] + b.w01 * t01[c] + b.w11 * t11[c];
    return;
  }
  // Mip filters (Texture.swift:795-863).
  float4 da = ld_nt4(uv_da + pix * 4);
  const float s = bias_scale(bias_map, pix, scale_bias, has_bias != 0);
  if (bias_map || has_bias) da = make_float4(da.x * s, da.y * s, da.z * s, da.w * s);
  const Lod ld = mip_lod(da, Ht, Wt, md.L, FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR);
  const bool shared = tex_stride == 0;
  // texels as vectors, the sum in registers
  float acc[CT];
#pragma unroll
  for (int li = 0; li < 2; ++li) {
    // a zero weight adds +0 to every channel: the second level is not read
    // (the result differs only for non-finite texels, where 0 * inf is NaN)
    if (li == 1 && ld.frac == 0.0f) break;
    const int k = li == 0 ? ld.k0 : ld.k1;
    const int Hk = mip_h(md, k), Wk = mip_w(md, k);
    const float* lv = k == 0 ? tex + n * tex_stride
                             : pyr + mip_off(md, k) + (shared ? 0 : (int64_t)n * Hk * Wk * C);
    const Bilin b = bilin(uvp.x, uvp.y, Wk, Hk, boundary);
    const float wgt = li == 0 ? (1.0f - ld.frac) : ld.frac;
    float t00[kMaxC], t10[kMaxC], t01[kMaxC], t11[kMaxC];
    load_texel<CT>(lv + ((int64_t)b.iy0 * Wk + b.ix0) * C, C, t00);
    load_texel<CT>(lv + ((int64_t)b.iy0 * Wk + b.ix1) * C, C, t10);
    load_texel<CT>(lv + ((int64_t)b.iy1 * Wk + b.ix0) * C, C, t01);
    load_texel<CT>(lv + ((int64_t)b.iy1 * Wk + b.ix1) * C, C, t11);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const float sample = b.w00 * t00[c] + b.w10 * t10[c] + b.w01 * t01[c] + b.w11 * t11[c];
      acc[c] = li == 0 ? wgt * sample : acc[c] + wgt * sample;  // two roundings, as :855 / :858
    }
  }
  if constexpr (CT == 4) {
    *reinterpret_cast<float4*>(o) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  } else {
#pragma unroll
    for (int c = 0; c < CT; ++c) o[c] = acc[c];
  }
}

// BND: the boundary mode as a compile-time constant (DR_BOUNDARY_CUBE for
// cube maps), so the clamp and wrap footprints carry no out-of-range masks.
// One workgroup per 16x16 pixel tile, a 16x4 strip per wave: neighbouring
// pixels sample neighbouring texels, so a wave's gathers share cache lines
// (measured 0.105 -> 0.089 ms at 8 x 1024^2 against whole pixel rows).
template <int FILTER, int BND, int CT>
__global__ void __launch_bounds__(256) k_tex_fwd(
    const float* __restrict__ tex, const float* __restrict__ pyr, MipDesc md, int64_t tex_stride,
    int Ht, int Wt, int C_, const float* __restrict__ uv, const float* __restrict__ uv_da,
    const float* __restrict__ bias_map, float scale_bias, int has_bias, int64_t P, int Hi,
    int Wi, float* __restrict__ out) {
  const int ntx = (Wi + 15) >> 4, tiles = ntx * ((Hi + 15) >> 4);
  const int b = (int)blockIdx.x, n = b / tiles, tile = b - n * tiles;
  const int ty = tile / ntx, tx = tile - ty * ntx;
  const int ph = ty * 16 + ((int)threadIdx.x >> 4), pw = tx * 16 + ((int)threadIdx.x & 15);
  // pixels past the image's right or bottom edge get index P: no work
  const int64_t pix = ph < Hi && pw < Wi ? ((int64_t)n * Hi + ph) * Wi + pw : P;
  tex_fwd_px<FILTER, BND == DR_BOUNDARY_CUBE, CT>(tex, pyr, md, tex_stride, Ht, Wt, C_, uv, uv_da,
                                                  bias_map, scale_bias, has_bias, BND, P, n, out,
                                                  pix);
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------

// Per-wave accumulator of one bilinear footprint's gradient.  A large group
// of lanes on one footprint (in practice: every background pixel samples the
// same clamped texel) adds its wave-summed values here instead of issuing
// atomics; the accumulator is written out when a different footprint takes
// its place and when the wave has finished all its tiles.  Wave-uniform.
// (V: double where the sums are fp64 all the way, k_tex_bwd_win.)
template <int CT, typename V = float>
struct FootAcc {
  float* p[4];  // the footprint's four texels (wave-uniform)
  V v;          // lane j < 4*CT: running sum of value j = 4 * channel + tap
  bool on;
};

template <int CT, typename V>
__device__ __forceinline__ void acc_init(FootAcc<CT, V>& a) {
  a.on = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) a.p[i] = nullptr;
  a.v = 0;
}

template <int CT, typename V>
__device__ __forceinline__ void acc_flush(FootAcc<CT, V>& a) {
  if (!a.on) return;
  const int l = lane_id();
  if (l < 4 * CT && a.v != 0) {
    const int tap = l & 3;
    float* q = tap == 0 ? a.p[0] : tap == 1 ? a.p[1] : tap == 2 ? a.p[2] : a.p[3];
    unsafeAtomicAdd(q + (l >> 2), (float)a.v);
  }
  a.on = false;
}

// The accumulators of a workgroup's W waves at its end (every thread calls
// it): those of one footprint are added up in fp64 and written once.  The
// empty pixels' footprint collects one addition per value from every
// workgroup of the persistent grid, and the atomics on one address are
// serialised (about 80 M/s) just as the workgroups end: one per workgroup
// instead of one per wave (bilinear, 4 x 1000^2 x 3: 215 -> 193 us; 8 x 1024^2
// trilinear, whose waves end further apart: no change).
template <int CT, int W, typename V = float>
struct FootAccLds {
  uint64_t p[W][4];
  V v[W][4 * CT];
};

template <int CT, int W, typename V>
__device__ __forceinline__ void acc_flush_group(const FootAcc<CT, V>& a, FootAccLds<CT, W, V>& s) {
  const int wave = (int)threadIdx.x >> 6, l = lane_id();
  if (l < 4) {
    float* q = l == 0 ? a.p[0] : l == 1 ? a.p[1] : l == 2 ? a.p[2] : a.p[3];
    s.p[wave][l] = a.on ? (uint64_t)q : 0ull;
  }
  if (l < 4 * CT) s.v[wave][l] = a.on ? a.v : V(0);
  __syncthreads();
  if (!a.on) return;
  auto same = [&](int w) {
    return s.p[w][0] == s.p[wave][0] && s.p[w][1] == s.p[wave][1] &&
           s.p[w][2] == s.p[wave][2] && s.p[w][3] == s.p[wave][3];
  };
  for (int w = 0; w < wave; ++w)
    if (same(w)) return;  // an earlier wave writes this footprint
  if (l >= 4 * CT) return;
  double sum = 0.0;
  for (int w = wave; w < W; ++w)
    if (same(w)) sum += (double)s.v[w][l];
  if (sum != 0.0) unsafeAtomicAdd((float*)s.p[wave][l & 3] + (l >> 2), (float)sum);
}

// Adds the wave sums of val[0..M) (M <= 16) to the accumulator.
template <int CT, int M>
__device__ __forceinline__ void acc_add(FootAcc<CT>& a, const float (&val)[M], bool member) {
  static_assert(M <= 16, "at most 16 values");
  float x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = (i < M && member) ? val[i < M ? i : 0] : 0.0f;
  a.v += wave_sum16(x);
}

// Scatter of one bilinear footprint's gradient (w * g * scale) into one
// level.  Taps that land on the same texel (clamped borders) are merged
// first; lanes sharing the footprint are summed across the wave.
constexpr int kTexTable = 512;  // LDS aggregation entries per tile (texels)

template <int CT, int CAP = kTexTable>
using TexTable = LdsTable<(CT > 0 ? CT : 1), CAP>;

// The cube backward's table: a cube map's footprints spread over more
// texels per tile (a per-pixel LOD bias splits them over two or three
// levels), and a full table sends the rest of the tile's taps straight to
// device atomics.
//
// Slots keep texel order: eight consecutive texels hash to one block of eight
// slots, a texel taking its place in the block (or the same place of another
// block, when that is another texel's).  A bit per slot marks those taken, so
// the flush lists them in slot order and its atomics of neighbouring texels
// share cache-line requests, which is what the device's atomic units count
// (about 21 G/s; with entries in hash order the kernel issued 17.7 G/s of
// them).  4096 x 256^2, 6 x 512^2 x 3, a random bias map: 34.8 ms with 2,048
// entries in hash order, 30.8 in texel order, and then 25.6 with 1,536, which
// three workgroups per CU fit at three channels (27.2 with 1,152 and four).
constexpr int kCubeTable = 1536;
template <int CT>
struct CubeTable {
  static constexpr int NV = CT > 0 ? CT : 1, CAP = kCubeTable;
  static_assert(CAP % 32 == 0 && CAP / 8 <= 256, "a thread of the flush per block of slots");
  unsigned long long key[CAP];  // destination address
  double val[NV][CAP];          // component-major (LdsTable)
  uint32_t bits[CAP / 32];      // slots taken since the last flush
  uint16_t slot[CAP];           // the flush's list of them
  int wsum[4];
};

template <int CT>
__device__ __forceinline__ void cube_table_clear(CubeTable<CT>& t) {
  for (int i = threadIdx.x; i < CubeTable<CT>::CAP; i += 256) {
    t.key[i] = kEmptyKey;
#pragma unroll
    for (int j = 0; j < CubeTable<CT>::NV; ++j) t.val[j][i] = 0.0;
  }
  if (threadIdx.x < CubeTable<CT>::CAP / 32) t.bits[threadIdx.x] = 0;
}

// Adds v to the texel at dst, the texel's index within its level `texel`;
// `seed` differs from level to level.
template <int CT>
__device__ __forceinline__ void cube_table_add(CubeTable<CT>& t, float* dst, uint32_t seed,
                                               uint32_t texel, const float* v) {
  constexpr int NV = CubeTable<CT>::NV, CAP = CubeTable<CT>::CAP;
  bool any = false;
#pragma unroll
  for (int j = 0; j < NV; ++j) any = any || v[j] != 0.0f;
  if (!any) return;
  const unsigned long long key = (unsigned long long)dst;
  uint32_t h = __umulhi(((texel >> 3) + seed) * 0x9E3779B1u, CAP / 8) * 8 + (texel & 7);
#pragma unroll 1
  for (int probe = 0; probe < kLdsProbes; ++probe) {
    unsigned long long cur = t.key[h];
    if (cur == kEmptyKey) {
      cur = atomicCAS(&t.key[h], kEmptyKey, key);
      if (cur == kEmptyKey) atomicOr(&t.bits[h >> 5], 1u << (h & 31));  // taken here
    }
    if (cur == kEmptyKey || cur == key) {
#pragma unroll
      for (int j = 0; j < NV; ++j)
        if (v[j] != 0.0f) atomicAdd(&t.val[j][h], (double)v[j]);
      return;
    }
    h += 8 * 37;
    if (h >= CAP) h -= CAP;
  }
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (v[j] != 0.0f) unsafeAtomicAdd(dst + j, v[j]);
}

// Writes the taken slots out in slot order and leaves the table cleared (call
// after a barrier; ends with one).
template <int CT>
__device__ __forceinline__ void cube_table_flush(CubeTable<CT>& t) {
  constexpr int NV = CubeTable<CT>::NV;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // thread i: slots 8i .. 8i + 7
  uint32_t mine = tid < CubeTable<CT>::CAP / 8 ? (t.bits[tid >> 2] >> ((tid & 3) * 8)) & 0xff : 0;
  int inc = __popc(mine);
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int o = __shfl_up(inc, d, kWave);
    if (lane >= d) inc += o;
  }
  if (lane == 63) t.wsum[wave] = inc;
  __syncthreads();
  int at = inc - __popc(mine), m = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) at += t.wsum[w];
    m += t.wsum[w];
  }
  for (; mine; mine &= mine - 1) t.slot[at++] = (uint16_t)(tid * 8 + __builtin_ctz(mine));
  if (tid < CubeTable<CT>::CAP / 32) t.bits[tid] = 0;
  __syncthreads();
  for (int i = tid; i < m * NV; i += 256) {
    const int e = t.slot[i / NV], j = i - (i / NV) * NV;
    const double v = t.val[j][e];
    if (v != 0.0) unsafeAtomicAdd((float*)t.key[e] + j, (float)v);
    t.val[j][e] = 0.0;
  }
  __syncthreads();
  for (int i = tid; i < m; i += 256) t.key[t.slot[i]] = kEmptyKey;
  __syncthreads();
}

template <int CT, bool USE_ACC = true, typename Tab = TexTable<CT>>
__device__ __forceinline__ void scatter_footprint(bool valid, float* __restrict__ base, int Wk,
                                                  int C, const Bilin& b, const float* g,
                                                  float scale,
                                                  FootAcc<(CT > 0 ? CT : 1)>& acc,
                                                  Tab& tab) {
  float w00 = b.w00, w10 = b.w10, w01 = b.w01, w11 = b.w11;
  if (b.ix1 == b.ix0) {
    w00 += w10;
    w01 += w11;
    w10 = 0.0f;
    w11 = 0.0f;
  }
  if (b.iy1 == b.iy0) {
    w00 += w01;
    w10 += w11;
    w01 = 0.0f;
    w11 = 0.0f;
  }
  float* const p[4] = {base + ((int64_t)b.iy0 * Wk + b.ix0) * C, base + ((int64_t)b.iy0 * Wk + b.ix1) * C,
                       base + ((int64_t)b.iy1 * Wk + b.ix0) * C, base + ((int64_t)b.iy1 * Wk + b.ix1) * C};
  if (CT > 0) {
    constexpr int M = 4 * (CT > 0 ? CT : 1);
    float val[M];
#pragma unroll
    for (int c = 0; c < (CT > 0 ? CT : 1); ++c) {
      const float gc = valid ? g[c] * scale : 0.0f;
      val[4 * c + 0] = w00 * gc;
      val[4 * c + 1] = w10 * gc;
      val[4 * c + 2] = w01 * gc;
      val[4 * c + 3] = w11 * gc;
    }
    // The probes pay where many lanes share a footprint: a magnified
    // texture (a texel cell three or more pixels wide repeats its taps over
    // runs of three lanes or more along the pixel rows) or one texel under
    // a whole wave.  Unless at least two lanes share their first tap with
    // the lane two before them they are skipped: footprints shared in pairs
    // only, as under a per-pixel LOD bias, never form a group worth them
    // (cube backward at 4096 x 256^2: 39.0 -> 36.9 ms).  Every lane executes
    // the shifts (callers keep the wave convergent).
    const uint64_t a0 = (uint64_t)p[0];
    const uint32_t l_lo = (uint32_t)dpp_shift<0x112>((int)(uint32_t)a0);
    const uint32_t l_hi = (uint32_t)dpp_shift<0x112>((int)(uint32_t)(a0 >> 32));
    const bool run3 = valid && (lane_id() & 15) >= 2 && (((uint64_t)l_hi << 32) | l_lo) == a0;
    uint64_t pending = __popcll(__ballot(run3)) >= 2 ? __ballot(valid) : 0ull;
    bool mine = valid;
    const int lane = lane_id();
#pragma unroll 1
    for (int probe = 0; probe < kProbes && pending; ++probe) {
      const int leader = probe_leader(pending, probe);
      float* lp[4];
      bool same = mine;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        lp[t] = (float*)lane_value((uint64_t)p[t], leader);
        same = same && p[t] == lp[t];
      }
      const uint64_t members = __ballot(same);
      pending &= ~members;
      if (__popcll(members) >= kGroupMin && !USE_ACC) {
#pragma unroll
        for (int i = 0; i < M; ++i) {
          const float sm = wave_sum(same ? val[i] : 0.0f);
          if (lane == leader && sm != 0.0f) unsafeAtomicAdd(lp[i & 3] + (i >> 2), sm);
        }
        if (same) mine = false;
      } else if (__popcll(members) >= kGroupMin) {
        const bool hit = acc.on && acc.p[0] == lp[0] && acc.p[1] == lp[1] && acc.p[2] == lp[2] &&
                         acc.p[3] == lp[3];
        if (!hit) {
          acc_flush(acc);
#pragma unroll
          for (int t = 0; t < 4; ++t) acc.p[t] = (float*)uni((uint64_t)lp[t]);
          acc.v = 0.0f;
          acc.on = true;
        }
        acc_add(acc, val, same);
        if (same) mine = false;
      }
    }
    if (mine) {
      [[maybe_unused]] const uint32_t seed = (uint32_t)((uint64_t)base >> 5);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float v[CT > 0 ? CT : 1];
#pragma unroll
        for (int c = 0; c < (CT > 0 ? CT : 1); ++c) v[c] = val[4 * c + t];
        if constexpr (std::is_same_v<Tab, CubeTable<CT>>)
          cube_table_add<CT>(tab, p[t], seed,
                             (uint32_t)((t & 2) ? b.iy1 : b.iy0) * (uint32_t)Wk +
                                 (uint32_t)((t & 1) ? b.ix1 : b.ix0), v);
        else
          lds_table_add(tab, p[t], v);
      }
    }
  } else {
    const uint32_t key2 = ((uint32_t)b.ix1 << 16) ^ (uint32_t)b.iy1;
    for (int c = 0; c < C; ++c) {
      const float gc = valid ? g[c] * scale : 0.0f;
      float val[4] = {w00 * gc, w10 * gc, w01 * gc, w11 * gc};
      float* addr[4] = {p[0] + c, p[1] + c, p[2] + c, p[3] + c};
      group_atomic_add<4>(valid, (uint64_t)p[0], addr, val, key2);
    }
  }
}

// d_uv terms of one level (Texture.swift:500-520 / :979-995), summed over C.
// IDX: the element offsets' type, int64_t for any level, or uint32_t where
// the caller guarantees a level below 2^32 elements (sides at most 32767,
// C at most 4).
template <typename IDX = int64_t>
__device__ __forceinline__ void duv_level(const float* __restrict__ lv, int Wk, int C,
                                          const Bilin& b, const float* g, float scale,
                                          float& dfx, float& dfy, float& dlod_sample) {
  dfx = 0.0f;
  dfy = 0.0f;
  dlod_sample = 0.0f;
  const IDX r0 = (IDX)b.iy0 * (IDX)Wk, r1 = (IDX)b.iy1 * (IDX)Wk;
  const float* p00 = lv + (r0 + (IDX)b.ix0) * (IDX)C;
  const float* p10 = lv + (r0 + (IDX)b.ix1) * (IDX)C;
  const float* p01 = lv + (r1 + (IDX)b.ix0) * (IDX)C;
  const float* p11 = lv + (r1 + (IDX)b.ix1) * (IDX)C;
  for (int c = 0; c < C; ++c) {
    const float r00 = p00[c], r10 = p10[c], r01 = p01[c], r11 = p11[c];
    const float t00 = r00 * b.m00, t10 = r10 * b.m10, t01 = r01 * b.m01, t11 = r11 * b.m11;
    const float gc = g[c] * scale;
    dfx += gc * ((1.0f - b.fy) * (t10 - t00) + b.fy * (t11 - t01));
    dfy += gc * ((1.0f - b.fx) * (t01 - t00) + b.fx * (t11 - t10));
    const float sample = b.w00 * r00 + b.w10 * r10 + b.w01 * r01 + b.w11 * r11;
    dlod_sample += sample * g[c];
  }
}

struct TexBwdArgs {
  const float* tex;
  const float* pyr;
  MipDesc md;
  int64_t tex_stride;
  int Ht, Wt, C, boundary, has_bias;
  const float* uv;
  const float* uv_da;
  const float* bias_map;
  float scale_bias;
  int N, Hi, Wi, ntx, nty;
  const float* d_out;
  float* d_tex;
  float* d_pyr;
  float* d_uv;
  float* d_uv_da;
  float* d_bias;
};

// One 16x16 pixel tile of the fused backward (one 8x8 quadrant per wave).
template <int FILTER, bool CUBE, int CT>
__device__ __forceinline__ void tex_bwd_tile(const TexBwdArgs& A, int bidx,
                                             FootAcc<(CT > 0 ? CT : 1)>& acc0,
                                             TexTable<CT>& tab) {
  const float* __restrict__ tex = A.tex;
  const float* __restrict__ pyr = A.pyr;
  const MipDesc& md = A.md;
  const int64_t tex_stride = A.tex_stride;
  const int Ht = A.Ht, Wt = A.Wt, C_ = A.C, boundary = A.boundary, has_bias = A.has_bias;
  const float* __restrict__ uv = A.uv;
  const float* __restrict__ uv_da = A.uv_da;
  const float* __restrict__ bias_map = A.bias_map;
  const float scale_bias = A.scale_bias;
  const int Hi = A.Hi, Wi = A.Wi, ntx = A.ntx, nty = A.nty;
  const float* __restrict__ d_out = A.d_out;
  float* __restrict__ d_tex = A.d_tex;
  float* __restrict__ d_pyr = A.d_pyr;
  float* __restrict__ d_uv = A.d_uv;
  float* __restrict__ d_uv_da = A.d_uv_da;
  float* __restrict__ d_bias = A.d_bias;
  const int tiles = ntx * nty;
  const int n = bidx / tiles;
  const int tile = bidx - n * tiles;
  const int ty = tile / ntx, tx = tile - ty * ntx;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int qx0 = tx * 16 + (wave & 1) * 8, qy0 = ty * 16 + (wave >> 1) * 8;
  if (qx0 >= Wi || qy0 >= Hi) return;
  const int pw = qx0 + (lane & 7), ph = qy0 + (lane >> 3);
  const bool valid = pw < Wi && ph < Hi;
  const int64_t pix = ((int64_t)n * Hi + min(ph, Hi - 1)) * Wi + min(pw, Wi - 1);
  const int C = dimC<CT>(C_);
  float g[CT > 0 ? CT : kMaxC];
  const float* gp = d_out + pix * C;
  float* dt = d_tex + n * tex_stride;  // tex_stride 0: shared texture

  if (CUBE) {  // Texture.swift:686-738 (d_dir is zero: :196-198)
    const float x = uv[pix * 3 + 0], y = uv[pix * 3 + 1], z = uv[pix * 3 + 2];
    Bilin b;
    const int face = cube_bilin(x, y, z, Wt, Ht, b);
    float* fb = dt + (int64_t)face * Ht * Wt * C;
    if (CT > 0) {
#pragma unroll
      for (int c = 0; c < (CT > 0 ? CT : 1); ++c) g[c] = gp[c];
      scatter_footprint<CT>(valid, fb, Wt, C, b, g, 1.0f, acc0, tab);
    } else {
      for (int c = 0; c < C; ++c) {
        const float gc = valid ? gp[c] : 0.0f;
        float val[4] = {b.w00 * gc, b.w10 * gc, b.w01 * gc, b.w11 * gc};
        float* addr[4] = {fb + ((int64_t)b.iy0 * Wt + b.ix0) * C + c,
                          fb + ((int64_t)b.iy0 * Wt + b.ix1) * C + c,
                          fb + ((int64_t)b.iy1 * Wt + b.ix0) * C + c,
                          fb + ((int64_t)b.iy1 * Wt + b.ix1) * C + c};
        group_atomic_add<4>(valid, (uint64_t)addr[0], addr, val,
                            ((uint32_t)b.ix1 << 16) ^ (uint32_t)b.iy1);
      }
    }
    if (d_uv && valid) {
      d_uv[pix * 3 + 0] = 0.0f;
      d_uv[pix * 3 + 1] = 0.0f;
      d_uv[pix * 3 + 2] = 0.0f;
    }
    return;
  }

  const float2 uvp = ld_nt2(uv + pix * 2);
  if (FILTER == DR_FILTER_NEAREST) {  // Texture.swift:576-605; d_uv = 0 (:234)
    const int txi = f2i(floorf(uvp.x * (float)Wt));
    const int tyi = f2i(floorf(uvp.y * (float)Ht));
    float ox, oy;
    const int ix = apply_boundary(txi, Wt, boundary, ox);
    const int iy = apply_boundary(tyi, Ht, boundary, oy);
    const float mask = (1.0f - ox) * (1.0f - oy);
    float* tp = dt + ((int64_t)iy * Wt + ix) * C;
    if (CT > 0) {
      if (valid) {
        float v[CT > 0 ? CT : 1];
#pragma unroll
        for (int c = 0; c < (CT > 0 ? CT : 1); ++c) v[c] = gp[c] * mask;
        lds_table_add(tab, tp, v);
      }
    } else {
      for (int c = 0; c < C; ++c) {
        float val[1] = {valid ? gp[c] * mask : 0.0f};
        float* addr[1] = {tp + c};
        group_atomic_add<1>(valid, (uint64_t)tp, addr, val);
      }
    }
    if (d_uv && valid) *reinterpret_cast<float2*>(d_uv + pix * 2) = make_float2(0.0f, 0.0f);
    return;
  }

  for (int c = 0; c < C && c < (CT > 0 ? CT : kMaxC); ++c) g[c] = valid ? gp[c] : 0.0f;
  const float* gsrc = CT > 0 ? g : gp;  // run-time C reads d_out directly

  if (FILTER == DR_FILTER_LINEAR) {  // Texture.swift:407-521
    const Bilin b = bilin(uvp.x, uvp.y, Wt, Ht, boundary);
    const float* tb = tex + n * tex_stride;
    scatter_footprint<CT>(valid, dt, Wt, C, b, gsrc, 1.0f, acc0, tab);
    if (d_uv && valid) {
      float dfx, dfy, unused;
      duv_level(tb, Wt, C, b, gsrc, 1.0f, dfx, dfy, unused);
      *reinterpret_cast<float2*>(d_uv + pix * 2) = make_float2(dfx * (float)Wt, dfy * (float)Ht);
    }
    return;
  }

  // Mip filters: Texture.swift:870-1102 fused.
  const float4 da_in = *reinterpret_cast<const float4*>(uv_da + pix * 4);
  const float s = bias_scale(bias_map, pix, scale_bias, has_bias != 0);
  const bool scaled = bias_map || has_bias;
  const float4 da = scaled ? make_float4(da_in.x * s, da_in.y * s, da_in.z * s, da_in.w * s) : da_in;
  const bool linear = FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR;
  const Lod ld = mip_lod(da, Ht, Wt, md.L, linear);
  const bool shared = tex_stride == 0;
  auto level_ptr = [&](int k) -> const float* {
    return k == 0 ? tex + n * tex_stride
                  : pyr + mip_off(md, k) + (shared ? 0 : (int64_t)n * mip_h(md, k) * mip_w(md, k) * C);
  };
  auto dlevel_ptr = [&](int k) -> float* {
    return k == 0 ? dt : d_pyr + mip_off(md, k) + (shared ? 0 : (int64_t)n * mip_h(md, k) * mip_w(md, k) * C);
  };
  float dfx_total = 0.0f, dfy_total = 0.0f;
  float samp[2] = {0.0f, 0.0f};  // sum_c g_c * sample_c per level (for d_lod)
  for (int li = 0; li < 2; ++li) {
    const int k = li == 0 ? ld.k0 : ld.k1;
    const float scale = li == 0 ? (1.0f - ld.frac) : ld.frac;
    const int Hk = mip_h(md, k), Wk = mip_w(md, k);
    const Bilin b = bilin(uvp.x, uvp.y, Wk, Hk, boundary);
    // A zero weight adds nothing; skip the level's atomics (but keep the
    // wave convergent for the grouping).
    if (li == 0)
      scatter_footprint<CT, true>(valid && scale != 0.0f, dlevel_ptr(k), Wk, C, b, gsrc, scale, acc0,
                                  tab);
    else
      scatter_footprint<CT, false>(valid && scale != 0.0f, dlevel_ptr(k), Wk, C, b, gsrc, scale, acc0,
                                   tab);
    if (valid) {
      float dfx, dfy;
      duv_level(level_ptr(k), Wk, C, b, gsrc, scale, dfx, dfy, samp[li]);
      dfx_total += dfx * (float)Wk;
      dfy_total += dfy * (float)Hk;
    }
  }
  if (!valid) return;
  if (d_uv) *reinterpret_cast<float2*>(d_uv + pix * 2) = make_float2(dfx_total, dfy_total);
  if (!d_uv_da && !d_bias) return;
  // Texture.swift:1011-1102 (mip-nearest also takes this trilinear surrogate).
  const float sx = da.x * (float)Wt, sy = da.y * (float)Wt;
  const float tx_ = da.z * (float)Ht, ty_ = da.w * (float)Ht;
  const float Asq = sx * sx + tx_ * tx_;
  const float Bsq = sy * sy + ty_ * ty_;
  const float rho_sq = fmaxf(Asq, Bsq);
  const float lod_raw = 0.5f * log2f(fmaxf(rho_sq, 1e-20f));
  float4 d_eff = make_float4(0.f, 0.f, 0.f, 0.f);
  if (!(lod_raw <= 0.0f || lod_raw >= (float)(md.L - 1))) {
    float d_lod;
    const int k0 = f2i(floorf(lod_raw));
    if (linear) {
      d_lod = -samp[0] + samp[1];
    } else {
      const int k1 = min(k0 + 1, md.L - 1);
      float s0 = 0.0f, s1 = 0.0f, u0, u1;
      const Bilin b0 = bilin(uvp.x, uvp.y, mip_w(md, k0), mip_h(md, k0), boundary);
      duv_level(level_ptr(k0), mip_w(md, k0), C, b0, gsrc, 0.0f, u0, u1, s0);
      const Bilin b1 = bilin(uvp.x, uvp.y, mip_w(md, k1), mip_h(md, k1), boundary);
      duv_level(level_ptr(k1), mip_w(md, k1), C, b1, gsrc, 0.0f, u0, u1, s1);
      d_lod = -s0 + s1;
    }
    const float ln2 = 0.6931471805599453f;
    const float dlod_drho_sq = 1.0f / (2.0f * rho_sq * ln2);
    const float A_is_max = (Asq >= Bsq) ? 1.0f : 0.0f;
    const float B_is_max = 1.0f - A_is_max;
    d_eff = make_float4(d_lod * dlod_drho_sq * A_is_max * 2.0f * sx * (float)Wt,
                        d_lod * dlod_drho_sq * B_is_max * 2.0f * sy * (float)Wt,
                        d_lod * dlod_drho_sq * A_is_max * 2.0f * tx_ * (float)Ht,
                        d_lod * dlod_drho_sq * B_is_max * 2.0f * ty_ * (float)Ht);
  }
  // Backward of the bias fold: d_uvDA = d_eff * scale,
  // d_map = sum_c(d_eff_c * uvDA_c) * scale * ln 2.
  if (d_uv_da) {
    const float4 o = scaled ? make_float4(d_eff.x * s, d_eff.y * s, d_eff.z * s, d_eff.w * s) : d_eff;
    *reinterpret_cast<float4*>(d_uv_da + pix * 4) = o;
  }
  if (d_bias && bias_map) {
    const float gm = d_eff.x * da_in.x + d_eff.y * da_in.y + d_eff.z * da_in.z + d_eff.w * da_in.w;
    d_bias[pix] = gm * s * 0.6931471805599453f;
  }
}

template <int FILTER, bool CUBE, int CT>
__global__ void __launch_bounds__(256) k_tex_bwd(TexBwdArgs A, int total_tiles) {
  __shared__ TexTable<CT> tab;
  __shared__ FootAccLds<(CT > 0 ? CT : 1), 4> s_acc;
  FootAcc<(CT > 0 ? CT : 1)> acc0;
  acc_init(acc0);
  lds_table_clear(tab);
  __syncthreads();
  for (int t = (int)blockIdx.x; t < total_tiles; t += (int)gridDim.x) {
    tex_bwd_tile<FILTER, CUBE, CT>(A, t, acc0, tab);
    __syncthreads();
    lds_table_flush(tab);
    __syncthreads();
  }
  acc_flush_group(acc0, s_acc);
}

// ---------------------------------------------------------------------------
// Windowed backward, C in 1..4: every 2D filter, and bilinear cube maps (a
// face in the place of a level).  Per 16x16 pixel tile the texel bounding box
// of the footprints on each level in use is taken (window_box.h), and
// contributions are summed into dense fp64
// LDS windows over those boxes (direct indexing, no hashing; the windows
// share one pool).  The windows are written out row by row, so consecutive
// lanes issue atomics to consecutive addresses.  Groups of lanes on one
// footprint (empty pixels) go to the per-wave accumulator; a box the pool
// cannot hold goes through it in bands of rows (bilinear), or its taps go to
// memory a texel row at a time.  Before, such taps went through a small LDS
// hash table and mostly from there to one device atomic per value (bilinear,
// 4 x 1000^2 x 3 at 1-3 texels a pixel: 960 us, now 189; at 8 x 1024^2
// trilinear with 1.3% of them, no change: 238 us).  Cube maps and the nearest
// filter took the 512-entry hash table for all taps (cube, 4 x 800^2 x 3:
// 94 us, now 55; nearest, 4 x 800 x 700 x 4: 86, now 51).
// ---------------------------------------------------------------------------

constexpr int kWinWaves = 4;                  // waves per workgroup; a tile is 16 x (4 * kWinWaves) pixels
constexpr int kWinThreads = 64 * kWinWaves;

// Texels of a tile's windows together: what five workgroups per CU leave of
// the LDS at four channels (8 x 1024^2, trilinear: 237.8 us with 928, 239.7
// with 768, 313.8 with 992, where only four fit).  The bilinear filter has one slot a pixel and no
// level to absorb minification, so up to three channels it takes as many as
// the 10-bit window fields address (4 x 1000^2 x 3 at 1-3 texels a pixel:
// backward 338 -> 289 us against 768, before the bands).
template <int FILTER, int CT>
constexpr int win_texels() {
  return (FILTER == DR_FILTER_LINEAR || FILTER == DR_FILTER_NEAREST) && CT < 4 ? 1008
                                                                              : 232 * kWinWaves;
}

// Most bands of a box larger than the pool (bilinear): 289 -> 218 us at the
// same sizes; two, four, six or ten allowed differ by the noise (218-226),
// since a box of more than a few thousand texels holds few taps each.
constexpr int kWinBands = 4;

// Runs of a wave up to which the direct way adds lane by lane (1 x 512^2,
// trilinear, one tile a workgroup: 21 us for the kernel, 34 with the hash
// table; the bilinear case above takes the staged way: 189 us, 349 lane by
// lane).
constexpr int kWinFewRuns = 12;

// The texel of window coordinate t.
template <int BND>
__device__ __forceinline__ int win_texel(int t, int size) {
  if (BND != DR_BOUNDARY_WRAP) return t;
  const int r = t % size;
  return r < 0 ? r + size : r;
}

// t mod size for t >= 0, mostly below 2 * size.
__device__ __forceinline__ int wrap_up(int t, int size) {
  if (t >= size) t -= size;
  return t < size ? t : t % size;
}

// a * b, 0 where either is 0 whatever the other (an infinity, NaN): one
// instruction, whose intrinsic has no builtin in this compiler.
__device__ float mul0(float a, float b) __asm("llvm.amdgcn.fmul.legacy");

// Weight `tap` (0..3: 00, 10, 01, 11) of the wave-uniform lane `leader`.
__device__ __forceinline__ float leader_weight(const TapSlot& q, int leader, int tap) {
  const int a = __builtin_amdgcn_readlane(__float_as_int(q.w00), leader);
  const int b = __builtin_amdgcn_readlane(__float_as_int(q.w10), leader);
  const int c = __builtin_amdgcn_readlane(__float_as_int(q.w01), leader);
  const int d = __builtin_amdgcn_readlane(__float_as_int(q.w11), leader);
  return __int_as_float(tap == 0 ? a : tap == 1 ? b : tap == 2 ? c : d);
}

template <int FILTER, int CT, int BND, bool BIAS>
// Five waves per SIMD (the register budget this asks for costs a few
// spilled values; measured cheaper than four or six).
__global__ void __launch_bounds__(kWinThreads, 5) k_tex_bwd_win(TexBwdArgs A, int total_tiles) {
  constexpr int kWinTexels = win_texels<FILTER, CT>();
  // channel-major (win[c * kWinTexels + texel]): a wave's run tails on
  // neighbouring texels then add 8 bytes apart, spread over the banks,
  // rather than 8 * CT bytes apart on a few of them
  __shared__ double win[kWinTexels * CT];
  __shared__ __align__(16) int s_lmask[kWinWaves];  // per wave: the levels in use (bit mask)
  __shared__ int2 s_lbox[kWinWaves][kMaxLevels];     // per wave and level: packed box
  // Sums that are fp64 from the first term on: the nearest filter's and the
  // bilinear cube maps' runs, and their and the wrap mode's empty pixels
  // (other runs and empty pixels are summed in fp32 first).  Against fp32 sums:
  // cube, 4 x 800^2 x 3, 49 -> 55 us; nearest and bilinear wrap, no change.
  constexpr bool kWide = FILTER == DR_FILTER_NEAREST || BND == DR_BOUNDARY_CUBE;
  using RunT = std::conditional_t<kWide, double, float>;
  using AccT = std::conditional_t<kWide || BND == DR_BOUNDARY_WRAP, double, float>;
  __shared__ FootAccLds<CT, kWinWaves, AccT> s_acc;
  FootAcc<CT, AccT> acc;
  acc_init(acc);
  const int tid = threadIdx.x;
  for (int i = tid; i < kWinTexels * CT; i += kWinThreads) win[i] = 0.0;
  __syncthreads();

  const MipDesc& md = A.md;
  const bool mip = FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR || FILTER == DR_FILTER_LINEAR_MIPMAP_NEAREST;
  constexpr bool kCube = BND == DR_BOUNDARY_CUBE;
  constexpr bool kSameUv = BND == DR_BOUNDARY_WRAP || FILTER == DR_FILTER_NEAREST;
  constexpr bool kOneLevel = kCube || FILTER == DR_FILTER_NEAREST || FILTER == DR_FILTER_LINEAR;
  // Taps of a footprint.  The nearest filter has one, of weight 1 (its mask
  // goes into the cotangent): three more of weight 0 would put 0 * inf into
  // texels that it does not sample, and cost their LDS additions.
  constexpr int kTaps = FILTER == DR_FILTER_NEAREST ? 1 : 4;
  // A tap of weight zero may lie outside its box, and has a clamped place
  // there: it adds 0 (mul0), and what 0 * g is where a cotangent is not
  // finite goes to the tap's own texel, apart from the windows.  (So does the
  // product of a cotangent of zero and a weight that is not finite.)
  constexpr bool kOwnTaps = kTaps == 4 && (kCube || BND == DR_BOUNDARY_WRAP);
  constexpr int kRows = kTaps == 1 ? 1 : 2, kRowVals = (kTaps == 1 ? 1 : 2) * CT;  // texel rows
  const bool shared_tex = A.tex_stride == 0;
  const int wave = tid >> 6, lane = tid & 63;
  const int tiles = A.ntx * A.nty;

  int it = 0;
  // the tile's (n, ty, tx), advanced by the grid stride each step (scalar
  // adds; a division only when the stride crosses an image)
  const int G = (int)gridDim.x;
  const int Gy = G / A.ntx, Gx = G - Gy * A.ntx;
  int n = (int)blockIdx.x / tiles;
  int ty = ((int)blockIdx.x - n * tiles) / A.ntx;
  int tx = (int)blockIdx.x - n * tiles - ty * A.ntx;
  for (int bt = (int)blockIdx.x; bt < total_tiles; bt += G, ++it) {
    if (it > 0) {
      tx += Gx;
      ty += Gy;
      if (tx >= A.ntx) {
        tx -= A.ntx;
        ++ty;
      }
      if (ty >= A.nty) {
        const int q = ty / A.nty;
        n += q;
        ty -= q * A.nty;
      }
    }
    const int pw = tx * 16 + (lane & 15);  // 16x4 strip per wave, one pixel row per 16 lanes
    const int ph = ty * (4 * kWinWaves) + wave * 4 + (lane >> 4);
    const bool valid = pw < A.Wi && ph < A.Hi;
    const int64_t pix = ((int64_t)n * A.Hi + min(ph, A.Hi - 1)) * A.Wi + min(pw, A.Wi - 1);
    // cube maps: k is the face, one level each
    auto level_w = [&](int k) { return kOneLevel ? A.Wt : mip_w(md, k); };
    auto level_h = [&](int k) { return kOneLevel ? A.Ht : mip_h(md, k); };
    auto level_ptr = [&](int k) -> const float* {
      return k == 0 ? A.tex + n * A.tex_stride
                    : A.pyr + mip_off(md, k) + (shared_tex ? 0 : (int64_t)n * mip_h(md, k) * mip_w(md, k) * CT);
    };
    auto dlevel_ptr = [&](int k) -> float* {
      if (kCube) return A.d_tex + n * A.tex_stride + (int64_t)k * A.Ht * A.Wt * CT;
      return k == 0 ? A.d_tex + n * A.tex_stride
                    : A.d_pyr + mip_off(md, k) + (shared_tex ? 0 : (int64_t)n * mip_h(md, k) * mip_w(md, k) * CT);
    };

    // -- per pixel: footprints, gradients of uv / uvDA ------------------------
    float g[CT];
    if constexpr (CT == 4) {  // one vector load
      const float4 q4 = ld_nt4(A.d_out + pix * 4);
      g[0] = q4.x; g[1 % CT] = q4.y; g[2 % CT] = q4.z; g[3 % CT] = q4.w;
    } else {
      load_texel<CT>(A.d_out + pix * CT, CT, g);
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) g[c] = valid ? g[c] : 0.0f;
    float2 uvp = make_float2(0.0f, 0.0f);
    Bilin cb;
    int face = 0;
    if (kCube) {
      const float* d = A.uv + pix * 3;
      face = cube_bilin(d[0], d[1], d[2], A.Wt, A.Ht, cb);
    } else {
      uvp = ld_nt2(A.uv + pix * 2);
    }
    TapSlot q[2];
    float4 da_in = make_float4(0.f, 0.f, 0.f, 0.f), da = da_in;
    float s = 1.0f;
    bool scaled = false;
    // The second level's texels are read only when they count: a nonzero
    // weight, or (trilinear) a LOD inside (0, L-1) at an integer, where
    // d_lod needs its sample.  Magnified and background pixels (LOD clamped
    // to 0) skip them.
    bool need1 = false;
    bool lod0 = true;  // LOD clamped to 0: no d_lod sample is needed
    if (mip) {
      da_in = ld_nt4(A.uv_da + pix * 4);
      if (BIAS) {
        s = bias_scale(A.bias_map, pix, A.scale_bias, A.has_bias != 0);
        scaled = true;
      }
      da = scaled ? make_float4(da_in.x * s, da_in.y * s, da_in.z * s, da_in.w * s) : da_in;
      const Lod ld = mip_lod(da, A.Ht, A.Wt, md.L, FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR);
      q[0].k = ld.k0;
      q[0].scale = 1.0f - ld.frac;
      q[1].k = ld.k1;
      q[1].scale = ld.frac;
      need1 = ld.frac != 0.0f || (FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR && ld.k0 != 0);
      lod0 = FILTER != DR_FILTER_LINEAR_MIPMAP_LINEAR || (ld.k0 == 0 && ld.frac == 0.0f);
    } else {
      q[0].k = face;
      q[0].scale = 1.0f;
      q[1].k = 0;
      q[1].scale = 0.0f;
    }
    float dfx_total = 0.0f, dfy_total = 0.0f, samp[2] = {0.0f, 0.0f};
#pragma unroll
    for (int li = 0; li < 2; ++li) {
      if (li == 1 && !__ballot(valid && (q[1].scale != 0.0f || need1))) {
        // no lane weights or samples the second level (magnified and
        // background waves): its footprint would only be discarded
        q[1].ix0 = q[1].ix1 = q[1].iy0 = q[1].iy1 = 0;
        q[1].w00 = q[1].w10 = q[1].w01 = q[1].w11 = 0.0f;
        continue;
      }
      const int k = q[li].k, Hk = level_h(k), Wk = level_w(k);
      const Bilin b = kCube ? cb
                      : FILTER == DR_FILTER_NEAREST ? nearest_tap(uvp.x, uvp.y, Wk, Hk, BND)
                                                    : bilin(uvp.x, uvp.y, Wk, Hk, BND);
      float w00 = b.w00, w10 = b.w10, w01 = b.w01, w11 = b.w11;
      if (b.ix1 == b.ix0) { w00 += w10; w01 += w11; w10 = 0.0f; w11 = 0.0f; }
      if (b.iy1 == b.iy0) { w00 += w01; w10 += w11; w01 = 0.0f; w11 = 0.0f; }
      if (BND == DR_BOUNDARY_WRAP) {
        q[li].ix0 = win_coord(b.tx0, b.ix0); q[li].ix1 = q[li].ix0 + 1;
        q[li].iy0 = win_coord(b.ty0, b.iy0); q[li].iy1 = q[li].iy0 + 1;
      } else {
        q[li].ix0 = b.ix0; q[li].ix1 = b.ix1; q[li].iy0 = b.iy0; q[li].iy1 = b.iy1;
      }
      bool on = valid && q[li].scale != 0.0f;
      if constexpr (FILTER == DR_FILTER_NEAREST) {
        bool any = false;  // a nonzero value, or NaN (0 * inf outside the image)
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          g[c] *= b.w00;
          any = any || g[c] != 0.0f;
        }
        on = on && any;
        w00 = 1.0f;
        w10 = w01 = w11 = 0.0f;
      }
      q[li].w00 = on ? w00 : 0.0f; q[li].w10 = on ? w10 : 0.0f;
      q[li].w01 = on ? w01 : 0.0f; q[li].w11 = on ? w11 : 0.0f;
      // A footprint collapsed onto one texel (clamped at a corner; every
      // background pixel) has zero texel differences: its uv gradient is
      // zero and, at LOD 0, its sample is not needed.
      const bool flat = BND != DR_BOUNDARY_ZERO && b.ix0 == b.ix1 && b.iy0 == b.iy1 && lod0;
      if (!kCube && FILTER != DR_FILTER_NEAREST && valid && (li == 0 || need1) && !flat) {
        float dfx, dfy;
        duv_level<uint32_t>(level_ptr(k), Wk, CT, b, g, mip ? q[li].scale : 1.0f, dfx, dfy, samp[li]);
        dfx_total += dfx * (float)Wk;
        dfy_total += dfy * (float)Hk;
      }
    }
    if (valid && A.d_uv) {  // (cube and nearest: zero, Texture.swift:196-198, :234)
      if (kCube) {
        A.d_uv[pix * 3 + 0] = 0.0f;
        A.d_uv[pix * 3 + 1] = 0.0f;
        A.d_uv[pix * 3 + 2] = 0.0f;
      } else {
        st_nt2(A.d_uv + pix * 2, make_float2(dfx_total, dfy_total));
      }
    }
    if (mip && valid && (A.d_uv_da || A.d_bias)) {  // Texture.swift:1011-1102
      const float sx = da.x * (float)A.Wt, sy = da.y * (float)A.Wt;
      const float tx_ = da.z * (float)A.Ht, ty_ = da.w * (float)A.Ht;
      const float Asq = sx * sx + tx_ * tx_;
      const float Bsq = sy * sy + ty_ * ty_;
      const float rho_sq = fmaxf(Asq, Bsq);
      const float lod_raw = 0.5f * log2f(fmaxf(rho_sq, 1e-20f));
      float4 d_eff = make_float4(0.f, 0.f, 0.f, 0.f);
      if (!(lod_raw <= 0.0f || lod_raw >= (float)(md.L - 1))) {
        float d_lod;
        if (FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR) {
          d_lod = -samp[0] + samp[1];
        } else {
          const int k0 = f2i(floorf(lod_raw));
          const int k1 = min(k0 + 1, md.L - 1);
          float s0 = 0.0f, s1 = 0.0f, u0, u1;
          const Bilin b0 = bilin(uvp.x, uvp.y, mip_w(md, k0), mip_h(md, k0), BND);
          duv_level<uint32_t>(level_ptr(k0), mip_w(md, k0), CT, b0, g, 0.0f, u0, u1, s0);
          const Bilin b1 = bilin(uvp.x, uvp.y, mip_w(md, k1), mip_h(md, k1), BND);
          duv_level<uint32_t>(level_ptr(k1), mip_w(md, k1), CT, b1, g, 0.0f, u0, u1, s1);
          d_lod = -s0 + s1;
        }
        const float ln2 = 0.6931471805599453f;
        // A gradient: the hardware reciprocal (1 ulp) is well inside tolerance.
        const float dlod_drho_sq = __builtin_amdgcn_rcpf(2.0f * rho_sq * ln2);
        const float A_is_max = (Asq >= Bsq) ? 1.0f : 0.0f;
        const float B_is_max = 1.0f - A_is_max;
        d_eff = make_float4(d_lod * dlod_drho_sq * A_is_max * 2.0f * sx * (float)A.Wt,
                            d_lod * dlod_drho_sq * B_is_max * 2.0f * sy * (float)A.Wt,
                            d_lod * dlod_drho_sq * A_is_max * 2.0f * tx_ * (float)A.Ht,
                            d_lod * dlod_drho_sq * B_is_max * 2.0f * ty_ * (float)A.Ht);
      }
      if (A.d_uv_da) {
        const float4 o = scaled ? make_float4(d_eff.x * s, d_eff.y * s, d_eff.z * s, d_eff.w * s) : d_eff;
        st_nt4(A.d_uv_da + pix * 4, o);
      }
      if (BIAS && A.d_bias && A.bias_map) {
        const float gm = d_eff.x * da_in.x + d_eff.y * da_in.y + d_eff.z * da_in.z + d_eff.w * da_in.w;
        A.d_bias[pix] = gm * s * 0.6931471805599453f;
      }
    }

    // -- hot footprint of slot 0: groups on one texel go to the accumulator
    bool hot = false;
    {
      const bool on0 = q[0].w00 != 0.0f || q[0].w10 != 0.0f || q[0].w01 != 0.0f || q[0].w11 != 0.0f;
      const int Wk = level_w(q[0].k);
      const uint64_t key = ((uint64_t)q[0].k << 48) | (uint64_t)((int64_t)q[0].iy0 * Wk + q[0].ix0);
      const uint32_t key2 = ((uint32_t)(q[0].ix1 - q[0].ix0) << 16) ^ (uint32_t)(q[0].iy1 - q[0].iy0);
      // flat footprints only (all the weight on one texel: every background
      // pixel), in groups of any size: a few background pixels kept out of
      // the windows keep a tile that mixes them with the object from boxes
      // spanning both, which the windows cannot hold (0.299 -> 0.294 ms at 8 x
      // 1024^2, when such boxes' taps took an LDS hash table); other footprints,
      // however many lanes share them, take the windows' run sums
      // Wrap mode: an empty pixel's footprint (uv = 0) is the texture's four
      // corner texels, so pixels of one uv are grouped instead: those at uv
      // (0, 0), and any whose left or right neighbour has the same uv (a
      // background given another constant).  One uv on one level has one set
      // of weights, so the group's cotangents are summed and then weighted
      // (4 x 1000^2 x 3, bilinear, 55% of the pixels empty: 960 -> 92 us with
      // the windows' unwrapped coordinates).
      // The nearest filter's footprints are all one texel: grouped by uv too.
      bool flat;
      if (kSameUv) {
        const int ux = __float_as_int(uvp.x), uy = __float_as_int(uvp.y);
        // (every lane executes the shifts)
        const int lx = dpp_shift<0x111>(ux), ly = dpp_shift<0x111>(uy);
        const int rx = dpp_shift<0x101>(ux), ry = dpp_shift<0x101>(uy);
        const bool left = (lane & 15) != 0 && lx == ux && ly == uy;
        const bool right = (lane & 15) != 15 && rx == ux && ry == uy;
        flat = on0 && ((uvp.x == 0.0f && uvp.y == 0.0f) || left || right);
      } else {
        flat = on0 && q[0].ix0 == q[0].ix1 && q[0].iy0 == q[0].iy1;
      }
      uint64_t pending = __ballot(flat);
#pragma unroll 1
      for (int probe = 0; probe < 2 && pending; ++probe) {
        const int leader = probe_leader(pending, probe);  // wave-uniform: readlane
        const uint64_t lkey = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(key >> 32), leader) << 32) |
                              (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)key, leader);
        const uint32_t lkey2 = (uint32_t)__builtin_amdgcn_readlane((int)key2, leader);
        bool same;
        if (kSameUv)
          same = flat && !hot && q[0].k == __builtin_amdgcn_readlane(q[0].k, leader) &&
                 __float_as_int(uvp.x) == __builtin_amdgcn_readlane(__float_as_int(uvp.x), leader) &&
                 __float_as_int(uvp.y) == __builtin_amdgcn_readlane(__float_as_int(uvp.y), leader);
        else
          same = flat && !hot && key == lkey && key2 == lkey2;
        const uint64_t members = __ballot(same);
        pending &= ~members;
        const int lk = __builtin_amdgcn_readlane(q[0].k, leader);
        float* base = dlevel_ptr(lk);
        const int lW = level_w(lk);
        float* lp[4];
        const int lH = level_h(lk);
        const int lix0 = win_texel<BND>(__builtin_amdgcn_readlane(q[0].ix0, leader), lW);
        const int lix1 = win_texel<BND>(__builtin_amdgcn_readlane(q[0].ix1, leader), lW);
        const int liy0 = win_texel<BND>(__builtin_amdgcn_readlane(q[0].iy0, leader), lH);
        const int liy1 = win_texel<BND>(__builtin_amdgcn_readlane(q[0].iy1, leader), lH);
        lp[0] = base + ((int64_t)liy0 * lW + lix0) * CT;
        lp[1] = base + ((int64_t)liy0 * lW + lix1) * CT;
        lp[2] = base + ((int64_t)liy1 * lW + lix0) * CT;
        lp[3] = base + ((int64_t)liy1 * lW + lix1) * CT;
        const bool hit = acc.on && acc.p[0] == lp[0] && acc.p[1] == lp[1] && acc.p[2] == lp[2] &&
                         acc.p[3] == lp[3];
        if (!hit) {
          acc_flush(acc);
#pragma unroll
          for (int t = 0; t < 4; ++t) acc.p[t] = (float*)uni((uint64_t)lp[t]);
          acc.v = 0;
          acc.on = true;
        }
        // all the weight is on tap 0 (one texel; wrap mode: the group has one
        // set of four weights): four sums, one per channel
        AccT x[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float gc = g[c < CT ? c : 0] * q[0].scale;
          x[c] = (c < CT && same) ? (kSameUv ? gc : q[0].w00 * gc) : 0.0f;
        }
        const AccT z = wave_sum4(x);  // lane l: total of value l & 3
        const AccT zc = __shfl(z, (lane >> 2) & 3, kWave);
        if (kSameUv && kTaps == 4) {  // lane 4c + t: channel c, tap t
          const float wt = leader_weight(q[0], leader, lane & 3);
          if (lane < 4 * CT) acc.v += wt * zc;
        } else {
          if (lane < 4 * CT && (lane & 3) == 0) acc.v += zc;  // lane 4c: channel c, tap 0
        }
        if (same) hot = true;
      }
    }

    // -- per wave: the levels in use and the box on each; the block's windows
    //    cover every level any wave uses ------------------------------------
    const bool use0 = !hot && (q[0].w00 != 0.0f || q[0].w10 != 0.0f || q[0].w01 != 0.0f || q[0].w11 != 0.0f);
    const bool use1 = q[1].w00 != 0.0f || q[1].w10 != 0.0f || q[1].w01 != 0.0f || q[1].w11 != 0.0f;
    {
      const int lm = wave_or((use0 ? 1 << q[0].k : 0) | (use1 ? 1 << q[1].k : 0));
#pragma unroll 1
      for (int rem = lm; rem != 0; rem &= rem - 1) {  // uniform: one level at a time
        const int L = __builtin_ctz(rem);
        // texel coordinates fit in 16 bits (window path needs sizes <= 32767):
        // (x0, -x1) and (y0, -y1) are reduced as packed 16-bit minima
        int x0 = 32767, x1 = -32767, y0 = 32767, y1 = -32767;
#pragma unroll
        for (int li = 0; li < 2; ++li) {
          const bool u = li == 0 ? use0 : use1;
          if (!u || q[li].k != L) continue;
          int a0, a1, b0, b1;
          slot_box(q[li], a0, a1, b0, b1);
          x0 = min(x0, a0); x1 = max(x1, a1); y0 = min(y0, b0); y1 = max(y1, b1);
        }
        const int px = wave_min_pk16(pack16(x0, -x1));
        const int py = wave_min_pk16(pack16(y0, -y1));
        if (lane == 0) s_lbox[wave][L] = make_int2(px, py);
      }
      if (lane == 0) s_lmask[wave] = lm;
    }
    __syncthreads();
    // Level L's window, in lane L of each 16-lane row: the union of the
    // waves' boxes on L and its place in the pool (levels in ascending
    // order; a box larger than the pool is left out).  A lane then takes
    // its slots' windows from the lanes of their levels.
    const int4 wm = *reinterpret_cast<const int4*>(s_lmask);
    const int lmask = __builtin_amdgcn_readfirstlane(wm.x | wm.y | wm.z | wm.w);
    // (x0 | y0 << 16) and win_pack's word (a box in the pool has at most
    // kWinTexels texels, so each of its sides and its offset fit in 10 bits)
    int wxy, wsz;
    {
      const int L = lane & 15;
      int px = pack16(32767, 32767), py = px;
#pragma unroll
      for (int v = 0; v < kWinWaves; ++v) {
        const int mv = v == 0 ? wm.x : v == 1 ? wm.y : v == 2 ? wm.z : wm.w;
        if ((mv >> L) & 1) {
          const int2 b = s_lbox[v][L];
          px = pk16_min(px, b.x);
          py = pk16_min(py, b.y);
        }
      }
      const int x0 = unpack16_lo(px), x1 = -unpack16_hi(px);
      const int y0 = unpack16_lo(py), y1 = -unpack16_hi(py);
      const bool present = L < kMaxLevels && ((lmask >> L) & 1) && x1 >= x0 && y1 >= y0;
      const int fit = present ? win_fit(x1 - x0 + 1, y1 - y0 + 1, kWinTexels) : 0;
      // inclusive prefix sum of the fitting areas along the row
      int incl = fit;
      int t = dpp_shift<0x111>(incl);
      incl += t;
      t = dpp_shift<0x112>(incl);
      incl += t;
      t = dpp_shift<0x114>(incl);
      incl += t;
      t = dpp_shift<0x118>(incl);
      incl += t;
      const bool usable = fit > 0 && incl <= kWinTexels;
      static_assert(kWinTexels < 1024, "window sides and offsets are 10-bit fields");
      wxy = pack16(x0, y0);
      wsz = usable ? win_pack(x1 - x0 + 1, y1 - y0 + 1, incl - fit) : 0;
    }

    // -- accumulate: runs of one footprint along a pixel row are summed
    //    first (lanes of one LDS atomic on one address are serialised), the
    //    run's last lane adds the totals ----------------------------------------
    // The runs of slot li's footprints in the `u` lanes, and the longest one in
    // the wave.  Every lane executes it.
    auto slot_runs = [&](int li, bool u, int& maxlen) -> RowRun {
      // level and the four texel coordinates (each < 32767 on the window
      // path) fix the taps; an unused slot gets a key no footprint has
      const uint64_t key =
          !u ? (0x7FFFull << 45) | (uint64_t)lane
          : BND == DR_BOUNDARY_WRAP  // (the second coordinates follow from the first)
             ? ((uint64_t)q[li].k << 60) | ((uint64_t)(uint16_t)q[li].ix0 << 16) |
                   (uint16_t)q[li].iy0
             : ((uint64_t)q[li].k << 60) | ((uint64_t)q[li].ix0 << 45) |
                   ((uint64_t)q[li].ix1 << 30) | ((uint64_t)q[li].iy0 << 15) |
                   (uint64_t)q[li].iy1;
      const RowRun run = row_run(key);
      maxlen = wave_max(run.li - run.s + 1);
      return run;
    };
    // Their totals of taps t0, t0 + 1, ... (v: tap-major, CT values a tap), in
    // a run's last lane; zero in a lane without `u`.  Every lane executes it.
    auto run_totals = [&](int li, bool u, const RowRun& run, int maxlen, int t0, auto& v) {
      constexpr int n = sizeof(v) / sizeof(v[0]) / CT;
      const float sc = mip ? q[li].scale : 1.0f;
      const float wt[4] = {q[li].w00, q[li].w10, q[li].w01, q[li].w11};
      float gs[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) gs[c] = !u ? 0.0f : g[c] * sc;
#pragma unroll
      for (int t = 0; t < n; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          v[t * CT + c] = kTaps == 1 ? gs[c] : kOwnTaps ? mul0(wt[t0 + t], gs[c]) : wt[t0 + t] * gs[c];
      row_run_scan_n(run, v, maxlen);
    };
    // Taps summed at once: all four in fp32, one in fp64, whose four would
    // need twice the registers (cube, 4 x 800^2 x 4: 61 us, 76 with all four).
    constexpr int kAtOnce = kWide ? 1 : kTaps;
#pragma unroll
    for (int li = 0; li < 2; ++li) {
      const bool u = li == 0 ? use0 : use1;
      if (__ballot(u) == 0) continue;  // no lane uses this slot (uniform)
      const int k = q[li].k;
      // the window of level k (every lane executes the permutes)
      const int sxy = __builtin_amdgcn_ds_bpermute(k << 2, wxy);
      const int ssz = __builtin_amdgcn_ds_bpermute(k << 2, wsz);
      int maxlen;
      const RowRun run = slot_runs(li, u, maxlen);
      const bool adds = u && run.tail && ssz != 0;
      int o[4] = {0, 0, 0, 0};
      if (adds) {
        // window indices of the four taps.  The box holds every tap with a
        // nonzero weight in some lane of the run; a tap whose weight is zero
        // in all of them (a texel column or row with zero weight, outside
        // the image for the zero boundary) may lie outside it, and its
        // coordinates are clamped into the box, where it adds 0.
        const int wx = unpack16_lo(sxy), wy = unpack16_hi(sxy);
        const int ww = win_w(ssz), wh = win_h(ssz), sbase = win_at(ssz);
        const int cx0 = min(max(q[li].ix0 - wx, 0), ww - 1);
        const int cx1 = min(max(q[li].ix1 - wx, 0), ww - 1);
        const int r0 = sbase + min(max(q[li].iy0 - wy, 0), wh - 1) * ww;
        const int r1 = sbase + min(max(q[li].iy1 - wy, 0), wh - 1) * ww;
        o[0] = r0 + cx0; o[1] = r0 + cx1; o[2] = r1 + cx0; o[3] = r1 + cx1;  // < sbase + area
      }
#pragma unroll
      for (int t0 = 0; t0 < kTaps; t0 += kAtOnce) {
        RunT v[kAtOnce * CT];
        run_totals(li, u, run, maxlen, t0, v);
        if (adds) {
#pragma unroll
          for (int t = 0; t < kAtOnce; ++t)
#pragma unroll
            for (int c = 0; c < CT; ++c)
              atomicAdd(win + c * kWinTexels + o[t0 + t], (double)v[t * CT + c]);
        }
      }
    }
    __syncthreads();

    if constexpr (kOwnTaps) {
      // what mul0 left out: 0 * g, and w * 0, where the other is not finite
      bool bad = false;
#pragma unroll
      for (int c = 0; c < CT; ++c) bad = bad || 0.0f * g[c] != 0.0f;
#pragma unroll
      for (int li = 0; li < (mip ? 2 : 1); ++li)
        bad = bad || 0.0f * (q[li].w00 + q[li].w10 + q[li].w01 + q[li].w11) != 0.0f;
      if (__ballot(bad) != 0ull) {  // uniform
#pragma unroll
        for (int li = 0; li < (mip ? 2 : 1); ++li) {
          const TapSlot& ql = q[li];
          if (!(bad && (li == 0 ? use0 : use1))) continue;
          const int k = ql.k, Wk = level_w(k), Hk = level_h(k);
#pragma unroll 1
          for (int t = 0; t < 4; ++t) {
            const float w = t == 0 ? ql.w00 : t == 1 ? ql.w10 : t == 2 ? ql.w01 : ql.w11;
            const int X = win_texel<BND>((t & 1) ? ql.ix1 : ql.ix0, Wk);
            const int Y = win_texel<BND>((t & 2) ? ql.iy1 : ql.iy0, Hk);
            float* p = dlevel_ptr(k) + ((int64_t)Y * Wk + X) * CT;
#pragma unroll
            for (int c = 0; c < CT; ++c) {
              const float x = w * g[c];
              if ((w == 0.0f || g[c] == 0.0f) && x != 0.0f) unsafeAtomicAdd(p + c, x);
            }
          }
        }
      }
    }

    // -- write the windows out, row by row -----------------------------------
    // Level k's window of bw x bh texels from window coordinates (x0, y0),
    // at `at` in the pool, added to the level and cleared.
    auto flush_window = [&](int k, int x0, int y0, int bw, int bh, int at) {
      float* base = dlevel_ptr(k);
      const int Wk = level_w(k), Hk = level_h(k);
      // (wrap mode: the first texel reduced into the texture; a window's
      // later columns and rows wrap from there)
      const int bx0 = win_texel<BND>(x0, Wk), by0 = win_texel<BND>(y0, Hk);
      const int row = bw * CT;
      const int total = row * bh;
      double* wb = win + at;
      // consecutive lanes take consecutive channels of a texel, so the
      // device atomics of a row share cache lines; (r, cpos) of element i
      // advance by a uniform step instead of a division per element
      const int dr = kWinThreads / row, dc = kWinThreads - dr * row;
      int r = tid / row, cpos = tid - r * row;
      for (int i = tid; i < total; i += kWinThreads) {
        const int tx = cpos / CT, c = cpos - tx * CT;
        double* e = wb + c * kWinTexels + r * bw + tx;
        const double v = *e;
        if (v != 0.0) {
          if (BND == DR_BOUNDARY_WRAP) {
            const int X = wrap_up(bx0 + tx, Wk), Y = wrap_up(by0 + r, Hk);
            unsafeAtomicAdd(base + ((int64_t)Y * Wk + X) * CT + c, (float)v);
          } else {
            unsafeAtomicAdd(base + ((int64_t)(by0 + r) * Wk + bx0) * CT + cpos, (float)v);
          }
          *e = 0.0;
        }
        r += dr;
        cpos += dc;
        if (cpos >= row) {
          cpos -= row;
          ++r;
        }
      }
    };
    int nowin = 0;  // levels without a window (uniform)
#pragma unroll 1
    for (int rem = lmask; rem != 0; rem &= rem - 1) {  // uniform
      const int k = __builtin_ctz(rem);
      const int sz = __builtin_amdgcn_readlane(wsz, k);
      if (sz == 0) {
        nowin |= 1 << k;
        continue;
      }
      const int xy = __builtin_amdgcn_readlane(wxy, k);
      flush_window(k, unpack16_lo(xy), unpack16_hi(xy), win_w(sz), win_h(sz), win_at(sz));
    }
    // -- bilinear: a box larger than the pool (a texture minified by up to a
    //    few texels a pixel) goes through it in bands of whole rows: a band's
    //    rows share cache-line requests, where the direct way below costs two
    //    requests a pixel whatever the box
    if (!mip && !kCube && nowin != 0) {  // uniform: level 0 alone is in use
      int px = pack16(32767, 32767), py = px;
#pragma unroll
      for (int w = 0; w < kWinWaves; ++w) {
        const int mw = w == 0 ? wm.x : w == 1 ? wm.y : w == 2 ? wm.z : wm.w;
        if (mw & 1) {
          px = pk16_min(px, s_lbox[w][0].x);
          py = pk16_min(py, s_lbox[w][0].y);
        }
      }
      px = __builtin_amdgcn_readfirstlane(px);
      py = __builtin_amdgcn_readfirstlane(py);
      const int x0 = unpack16_lo(px), y0 = unpack16_lo(py);
      const int bw = -unpack16_hi(px) - x0 + 1, bh = -unpack16_hi(py) - y0 + 1;
      const int rows = win_rows(bw, kWinTexels);
      if (rows * kWinBands >= bh) {  // (rows 0: too wide)
        int maxlen;
        const RowRun run = slot_runs(0, use0, maxlen);
        const bool adds = use0 && run.tail;
        RunT v[kTaps * CT];
        run_totals(0, use0, run, maxlen, 0, v);
        const int cx0 = min(max(q[0].ix0 - x0, 0), bw - 1);
        const int cx1 = min(max(q[0].ix1 - x0, 0), bw - 1);
        // (a zero-weight row outside the box is clamped into it: adds 0)
        const int cy0 = min(max(q[0].iy0 - y0, 0), bh - 1);
        const int cy1 = min(max(q[0].iy1 - y0, 0), bh - 1);
#pragma unroll 1
        for (int b0 = 0; b0 < bh; b0 += rows) {
          const int nr = min(rows, bh - b0);
          __syncthreads();  // the pool is written out (and cleared)
#pragma unroll
          for (int row = 0; row < kRows; ++row) {
            const int r = (row == 0 ? cy0 : cy1) - b0;
            if (adds && (unsigned)r < (unsigned)nr) {
#pragma unroll
              for (int c = 0; c < CT; ++c) {
                atomicAdd(win + c * kWinTexels + r * bw + cx0, (double)v[row * kRowVals + c]);
                if constexpr (kTaps == 4)
                  atomicAdd(win + c * kWinTexels + r * bw + cx1, (double)v[row * kRowVals + CT + c]);
              }
            }
          }
          __syncthreads();
          flush_window(0, x0, y0 + b0, bw, nr, 0);
        }
        nowin = 0;
      }
    }
    // -- levels without a window: each run's two texel rows straight to
    //    memory.  A wave lays a row's kRowVals totals of its 64 lanes out in
    //    its part of the pool and issues them with consecutive lanes on
    //    consecutive addresses (one cache-line request a row instead of one a
    //    value: the atomic units take requests, about 21 G/s), so a minified
    //    texture without mip levels costs two requests a pixel.  A few runs
    //    (a mixed tile's) are added lane by lane: fewer instructions.
    if (nowin != 0) {
      __syncthreads();  // the windows are written out: the pool is free and zero
      double* st = win + wave * (kWinTexels * CT / kWinWaves);
      static_assert(kWinTexels / kWinWaves >= 2 * 64, "a wave's row of totals fits its part");
      bool staged = false;
#pragma unroll
      for (int li = 0; li < (mip ? 2 : 1); ++li) {
        const int k = q[li].k;
        const bool u = (li == 0 ? use0 : use1) && ((nowin >> k) & 1);
        if (__ballot(u) == 0) continue;
        int maxlen;
        const RowRun run = slot_runs(li, u, maxlen);
        const bool adds = u && run.tail;
        const int Wk = level_w(k), Hk = level_h(k);
        const int X0 = win_texel<BND>(q[li].ix0, Wk), X1 = win_texel<BND>(q[li].ix1, Wk);
        const int Y0 = win_texel<BND>(q[li].iy0, Hk), Y1 = win_texel<BND>(q[li].iy1, Hk);
        float* const lv = dlevel_ptr(k);
        const uint32_t o0 = ((uint32_t)Y0 * (uint32_t)Wk + (uint32_t)X0) * CT;
        const uint32_t o1 = ((uint32_t)Y1 * (uint32_t)Wk + (uint32_t)X0) * CT;
        const int dx = (X1 - X0) * CT;
        const bool few = __popcll(__ballot(adds)) <= kWinFewRuns;  // uniform
        staged = staged || !few;
#pragma unroll
        for (int row = 0; row < kRows; ++row) {
          RunT v[kRowVals];
          run_totals(li, u, run, maxlen, row * 2, v);
          float* const pr = lv + (row == 0 ? o0 : o1);
          if (few) {
            if (adds) {
#pragma unroll
              for (int j = 0; j < kRowVals; ++j) {
                const float x = (float)v[j];
                if (x != 0.0f) unsafeAtomicAdd(pr + (j < CT ? j : dx + j - CT), x);
              }
            }
            continue;
          }
          const uint64_t p = (uint64_t)pr;
#pragma unroll
          for (int j = 0; j < kRowVals; ++j) st[lane * kRowVals + j] = adds ? (double)v[j] : 0.0;
          __builtin_amdgcn_wave_barrier();  // (LDS is ordered within a wave)
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll 1
          for (int i = 0; i < kRowVals; ++i) {
            const int e = (i * 64 + lane) / kRowVals, j = (i * 64 + lane) - e * kRowVals;
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(e << 2, (int)(uint32_t)p);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(e << 2, (int)(p >> 32));
            const int ed = __builtin_amdgcn_ds_bpermute(e << 2, dx);
            const float x = (float)st[i * 64 + lane];
            if (x != 0.0f)
              unsafeAtomicAdd((float*)(((uint64_t)hi << 32) | lo) + (j < CT ? j : ed + j - CT), x);
          }
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
      }
      if (staged) {  // zero again before the next barrier
#pragma unroll
        for (int j = 0; j < kRowVals; ++j) st[lane * kRowVals + j] = 0.0;
      }
    }
  }
  acc_flush_group(acc, s_acc);
}

// ---------------------------------------------------------------------------
// More than four channels (feature textures).  The forward gives a thread
// four channels of a pixel, consecutive threads consecutive channels, so
// texel reads and output writes are whole cache lines; one thread per pixel
// walking its channels read four bytes a lane at a stride of C floats
// (2 x 768^2 x 16, trilinear: 286 -> 49 us, 42 without the level of weight 0).
// ---------------------------------------------------------------------------

// The bilinear sample of channels [c, c + nc) of one level, in tex_fwd_px's
// operation order.
__device__ __forceinline__ float4 sample_chunk(const float* __restrict__ lv, int Wk, int C,
                                               const Bilin& b, int c, int nc) {
  const int64_t r0 = (int64_t)b.iy0 * Wk, r1 = (int64_t)b.iy1 * Wk;
  const float4 a = ld_chunk(lv + (r0 + b.ix0) * C + c, nc), d = ld_chunk(lv + (r0 + b.ix1) * C + c, nc);
  const float4 e = ld_chunk(lv + (r1 + b.ix0) * C + c, nc), f = ld_chunk(lv + (r1 + b.ix1) * C + c, nc);
  return make_float4(b.w00 * a.x + b.w10 * d.x + b.w01 * e.x + b.w11 * f.x,
                     b.w00 * a.y + b.w10 * d.y + b.w01 * e.y + b.w11 * f.y,
                     b.w00 * a.z + b.w10 * d.z + b.w01 * e.z + b.w11 * f.z,
                     b.w00 * a.w + b.w10 * d.w + b.w01 * e.w + b.w11 * f.w);
}

template <int FILTER, int BND>
__global__ void __launch_bounds__(256) k_tex_fwd_many(
    const float* __restrict__ tex, const float* __restrict__ pyr, MipDesc md, int64_t tex_stride,
    int Ht, int Wt, int C, const float* __restrict__ uv, const float* __restrict__ uv_da,
    const float* __restrict__ bias_map, float scale_bias, int has_bias, int64_t, int Hi, int Wi,
    float* __restrict__ out) {
  const int ntx = (Wi + 15) >> 4, tiles = ntx * ((Hi + 15) >> 4);
  const int b = (int)blockIdx.x, n = b / tiles, tile = b - n * tiles;
  const int ty = tile / ntx, tx = tile - ty * ntx;
  const int G = (C + 3) >> 2;  // chunks of four channels
  const bool shared = tex_stride == 0;
  // (pixel, chunk) of item i = threadIdx.x, + 256, ... of 256 * G, which need
  // not fit 32 bits
  const int step = 256 / G, rest = 256 - step * G;
  int lp = (int)threadIdx.x / G, g = (int)threadIdx.x - lp * G;
  for (; lp < 256; lp += step, g += rest) {
    if (g >= G) {
      g -= G;
      if (++lp >= 256) break;
    }
    const int c = g * 4;  // first channel
    const int ph = ty * 16 + (lp >> 4), pw = tx * 16 + (lp & 15);
    if (ph >= Hi || pw >= Wi) continue;
    const int64_t pix = ((int64_t)n * Hi + ph) * Wi + pw;
    const int nc = min(4, C - c);
    float4 o;
    if (BND == DR_BOUNDARY_CUBE) {
      Bilin bl;
      const int face = cube_bilin(uv[pix * 3 + 0], uv[pix * 3 + 1], uv[pix * 3 + 2], Wt, Ht, bl);
      o = sample_chunk(tex + n * tex_stride + (int64_t)face * Ht * Wt * C, Wt, C, bl, c, nc);
    } else {
      const float2 uvp = *reinterpret_cast<const float2*>(uv + pix * 2);
      if (FILTER == DR_FILTER_NEAREST) {
        float ox, oy;
        const int ix = apply_boundary(f2i(floorf(uvp.x * (float)Wt)), Wt, BND, ox);
        const int iy = apply_boundary(f2i(floorf(uvp.y * (float)Ht)), Ht, BND, oy);
        const float mask = (1.0f - ox) * (1.0f - oy);
        o = ld_chunk(tex + n * tex_stride + ((int64_t)iy * Wt + ix) * C + c, nc);
        o = make_float4(o.x * mask, o.y * mask, o.z * mask, o.w * mask);
      } else if (FILTER == DR_FILTER_LINEAR) {
        o = sample_chunk(tex + n * tex_stride, Wt, C, bilin(uvp.x, uvp.y, Wt, Ht, BND), c, nc);
      } else {
        float4 da = *reinterpret_cast<const float4*>(uv_da + pix * 4);
        const float s = bias_scale(bias_map, pix, scale_bias, has_bias != 0);
        if (bias_map || has_bias) da = make_float4(da.x * s, da.y * s, da.z * s, da.w * s);
        const Lod ld = mip_lod(da, Ht, Wt, md.L, FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR);
        auto level = [&](int k) {
          const int Hk = mip_h(md, k), Wk = mip_w(md, k);
          const float* lv = k == 0 ? tex + n * tex_stride
                                   : pyr + mip_off(md, k) + (shared ? 0 : (int64_t)n * Hk * Wk * C);
          return sample_chunk(lv, Wk, C, bilin(uvp.x, uvp.y, Wk, Hk, BND), c, nc);
        };
        const float w0 = 1.0f - ld.frac, w1 = ld.frac;
        // (a level of weight 0 counts where its texels are not finite: 0 * inf
        // is NaN; it is read unless it is the first level again)
        const float4 s0 = level(ld.k0), s1 = ld.k1 != ld.k0 ? level(ld.k1) : s0;
        o = make_float4(w0 * s0.x + w1 * s1.x, w0 * s0.y + w1 * s1.y, w0 * s0.z + w1 * s1.z,
                        w0 * s0.w + w1 * s1.w);
      }
    }
    st_chunk(out + pix * C + c, o, nc);
  }
}

// ---------------------------------------------------------------------------
// Windowed backward for more than four channels: k_tex_bwd_win's boxes and
// pool, with the channels taken four at a time and as many of them in the
// pool at once as the tile's boxes leave room for, so a window's flush writes
// a texel's channels as one run of memory.  One footprint set-up serves all
// channels, and d_uv and the LOD's gradient sum over them in registers.  The
// general kernel's wave probes and one device atomic per tap and channel
// took 3,453 us at 2 x 768^2 x 16, trilinear; this takes 186 (181 without
// zero_taps and the terms of weight 0, which matter for values that are not
// finite; there, 188 with the direct way's cotangents loaded one pixel at a
// time, 264 at four waves per SIMD, which spills 46 registers, 211 with two and
// a pool twice the size).
// Cube maps: k is the face, one level each.
// ---------------------------------------------------------------------------

constexpr int kManyPool = 4096;  // doubles: 32 KiB (3072: 197 us, 5632: 204)
constexpr int kManyC = 128;      // channels the empty pixels' sums have room for

// The sum of an empty-pixel group (one uv, so one footprint and one set of
// weights), kept in LDS per wave and channel until another footprint takes
// its place (wave-uniform).
struct ManyHot {
  bool on;
  int ux, uy;           // the uv's bits
  float* base;          // the level
  int ix0, ix1, iy0, iy1, Wk;
  float w00, w10, w01, w11;
};

template <int TAPS>
__device__ __forceinline__ void hot_flush(const ManyHot& h, int C, const double* s) {
  for (int i = lane_id(); i < TAPS * C; i += 64) {
    const int t = i / C, c = i - t * C;
    const float w = t == 0 ? h.w00 : t == 1 ? h.w10 : t == 2 ? h.w01 : h.w11;
    const float v = (float)((double)w * s[c]);
    if (v != 0.0f)
      unsafeAtomicAdd(h.base + ((int64_t)((t & 2) ? h.iy1 : h.iy0) * h.Wk +
                                ((t & 1) ? h.ix1 : h.ix0)) * C + c, v);
  }
}

// The taps of weight zero of one pixel's footprints (a border's merged ones, a
// texel centre's, those outside the image; slot 0's unless it is in the hot
// sum): 0 * g is 0, or NaN where a cotangent is not finite, and then belongs
// to the tap's own texel, which need not be in any window.  So does NaN of a
// weight that is not finite and a cotangent of zero.  Computed from the inputs
// again, so that nothing of it is kept in registers through the channels
// (k_tex_bwd_many spills already).
template <int FILTER, int BND>
__device__ __forceinline__ void zero_taps(const TexBwdArgs& A, int n, int64_t pix, bool in_hot) {
  constexpr bool kCube = BND == DR_BOUNDARY_CUBE;
  constexpr bool mip = FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR || FILTER == DR_FILTER_LINEAR_MIPMAP_NEAREST;
  constexpr int kTaps = FILTER == DR_FILTER_NEAREST ? 1 : 4;
  asm volatile("" : "+v"(pix));  // (not the values computed before)
  const float* gp = A.d_out + pix * A.C;
  Lod ld;
  ld.k0 = ld.k1 = 0;
  ld.frac = 0.0f;
  if (mip) {
    float4 da = *reinterpret_cast<const float4*>(A.uv_da + pix * 4);
    if (A.bias_map || A.has_bias) {
      const float s = bias_scale(A.bias_map, pix, A.scale_bias, A.has_bias != 0);
      da = make_float4(da.x * s, da.y * s, da.z * s, da.w * s);
    }
    ld = mip_lod(da, A.Ht, A.Wt, A.md.L, FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR);
  }
#pragma unroll 1
  for (int li = in_hot ? 1 : 0; li < (mip ? 2 : 1); ++li) {
    if (li == 1 && ld.frac == 0.0f) continue;
    int k = li == 0 ? ld.k0 : ld.k1;
    const int Wk = kCube ? A.Wt : mip_w(A.md, k), Hk = kCube ? A.Ht : mip_h(A.md, k);
    Bilin b;
    if (kCube) {
      k = cube_bilin(A.uv[pix * 3 + 0], A.uv[pix * 3 + 1], A.uv[pix * 3 + 2], Wk, Hk, b);
    } else {
      const float u = A.uv[pix * 2 + 0], v = A.uv[pix * 2 + 1];
      b = FILTER == DR_FILTER_NEAREST ? nearest_tap(u, v, Wk, Hk, BND) : bilin(u, v, Wk, Hk, BND);
    }
    if (b.ix1 == b.ix0) { b.w00 += b.w10; b.w01 += b.w11; b.w10 = 0.0f; b.w11 = 0.0f; }
    if (b.iy1 == b.iy0) { b.w00 += b.w01; b.w10 += b.w11; b.w01 = 0.0f; b.w11 = 0.0f; }
    float* lv = kCube || k == 0 ? A.d_tex + n * A.tex_stride + (int64_t)k * Hk * Wk * A.C
                                : A.d_pyr + mip_off(A.md, k) +
                                      (A.tex_stride == 0 ? 0 : (int64_t)n * Hk * Wk * A.C);
#pragma unroll
    for (int t = 0; t < kTaps; ++t) {
      const float w = t == 0 ? b.w00 : t == 1 ? b.w10 : t == 2 ? b.w01 : b.w11;
      if (w != 0.0f && 0.0f * w == 0.0f) continue;
      float* p = lv + ((int64_t)((t & 2) ? b.iy1 : b.iy0) * Wk + ((t & 1) ? b.ix1 : b.ix0)) * A.C;
      for (int c = 0; c < A.C; ++c) {
        const float gc = gp[c], x = w * gc;
        if ((w == 0.0f || gc == 0.0f) && x != 0.0f) unsafeAtomicAdd(p + c, x);
      }
    }
  }
}

template <int FILTER, int BND>
__global__ void __launch_bounds__(256, 3) k_tex_bwd_many(TexBwdArgs A, int total_tiles) {
  __shared__ double win[kManyPool];  // channel-major: win[c * texels + texel]
  __shared__ double s_hot[4][kManyC];
  __shared__ __align__(16) int s_lmask[4];
  __shared__ int2 s_lbox[4][kMaxLevels];
  __shared__ uint64_t s_hbase[4];
  __shared__ int2 s_hkey[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int i = tid; i < kManyPool; i += 256) win[i] = 0.0;
  for (int i = tid; i < 4 * kManyC; i += 256) (&s_hot[0][0])[i] = 0.0;
  __syncthreads();
  constexpr bool kCube = BND == DR_BOUNDARY_CUBE;
  constexpr bool mip = FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR || FILTER == DR_FILTER_LINEAR_MIPMAP_NEAREST;
  constexpr int kTaps = FILTER == DR_FILTER_NEAREST ? 1 : 4;  // (k_tex_bwd_win)
  const MipDesc& md = A.md;
  const int C = A.C;
  // texels are read for the gradients of uv and the LOD only
  const bool want = !kCube && FILTER != DR_FILTER_NEAREST && (A.d_uv || A.d_uv_da || A.d_bias);
  const bool shared_tex = A.tex_stride == 0;
  const int tiles = A.ntx * A.nty;
  ManyHot hot;
  hot.on = false;
  hot.ux = hot.uy = hot.ix0 = hot.ix1 = hot.iy0 = hot.iy1 = hot.Wk = 0;
  hot.base = nullptr;
  hot.w00 = hot.w10 = hot.w01 = hot.w11 = 0.0f;
  for (int bt = (int)blockIdx.x; bt < total_tiles; bt += (int)gridDim.x) {
    const int n = bt / tiles, tile = bt - n * tiles;
    const int ty = tile / A.ntx, tx = tile - ty * A.ntx;
    const int pw = tx * 16 + (lane & 15), ph = ty * 16 + wave * 4 + (lane >> 4);
    const bool valid = pw < A.Wi && ph < A.Hi;
    const int64_t pix = ((int64_t)n * A.Hi + min(ph, A.Hi - 1)) * A.Wi + min(pw, A.Wi - 1);
    const float* gp = A.d_out + pix * C;
    auto level_w = [&](int k) { return kCube ? A.Wt : mip_w(md, k); };
    auto level_h = [&](int k) { return kCube ? A.Ht : mip_h(md, k); };
    // float offset of level (face) k within the image's texture or pyramid
    auto level_ptr = [&](int k) -> const float* {
      if (kCube) return A.tex + n * A.tex_stride + (int64_t)k * A.Ht * A.Wt * C;
      return k == 0 ? A.tex + n * A.tex_stride
                    : A.pyr + mip_off(md, k) + (shared_tex ? 0 : (int64_t)n * mip_h(md, k) * mip_w(md, k) * C);
    };
    auto dlevel_ptr = [&](int k) -> float* {
      if (kCube) return A.d_tex + n * A.tex_stride + (int64_t)k * A.Ht * A.Wt * C;
      return k == 0 ? A.d_tex + n * A.tex_stride
                    : A.d_pyr + mip_off(md, k) + (shared_tex ? 0 : (int64_t)n * mip_h(md, k) * mip_w(md, k) * C);
    };

    // -- per pixel: LOD and footprints ------------------------------------------
    TapSlot q[2];
    float fx[2] = {0.0f, 0.0f}, fy[2] = {0.0f, 0.0f};
    int tx1[2] = {0, 0}, ty1[2] = {0, 0};   // second column and row as texels
    int tx0[2] = {0, 0}, ty0[2] = {0, 0};   // first
    int mask[2] = {15, 15};                 // zero boundary: taps inside the image
    float4 da_in = make_float4(0.f, 0.f, 0.f, 0.f), da = da_in;
    float s = 1.0f;
    const bool scaled = mip && (A.bias_map != nullptr || A.has_bias);
    float2 uvp = make_float2(0.0f, 0.0f);
    q[0].k = q[1].k = 0;
    q[0].scale = 1.0f;
    q[1].scale = 0.0f;
    Bilin cb;
    if (kCube) {
      const float* d = A.uv + pix * 3;
      q[0].k = cube_bilin(d[0], d[1], d[2], A.Wt, A.Ht, cb);
    } else {
      uvp = ld_nt2(A.uv + pix * 2);
    }
    if (mip) {
      da_in = ld_nt4(A.uv_da + pix * 4);
      if (scaled) s = bias_scale(A.bias_map, pix, A.scale_bias, A.has_bias != 0);
      da = scaled ? make_float4(da_in.x * s, da_in.y * s, da_in.z * s, da_in.w * s) : da_in;
      const Lod ld = mip_lod(da, A.Ht, A.Wt, md.L, FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR);
      q[0].k = ld.k0;
      q[0].scale = 1.0f - ld.frac;
      q[1].k = ld.k1;
      q[1].scale = ld.frac;
    }
#pragma unroll
    for (int li = 0; li < (mip ? 2 : 1); ++li) {
      const int k = q[li].k, Hk = level_h(k), Wk = level_w(k);
      const Bilin b = kCube ? cb
                      : FILTER == DR_FILTER_NEAREST ? nearest_tap(uvp.x, uvp.y, Wk, Hk, BND)
                                                    : bilin(uvp.x, uvp.y, Wk, Hk, BND);
      float w00 = b.w00, w10 = b.w10, w01 = b.w01, w11 = b.w11;
      if (b.ix1 == b.ix0) { w00 += w10; w01 += w11; w10 = 0.0f; w11 = 0.0f; }
      if (b.iy1 == b.iy0) { w00 += w01; w10 += w11; w01 = 0.0f; w11 = 0.0f; }
      const bool on = valid && q[li].scale != 0.0f;
      q[li].w00 = on ? w00 : 0.0f; q[li].w10 = on ? w10 : 0.0f;
      q[li].w01 = on ? w01 : 0.0f; q[li].w11 = on ? w11 : 0.0f;
      fx[li] = b.fx; fy[li] = b.fy;
      tx0[li] = b.ix0; tx1[li] = b.ix1; ty0[li] = b.iy0; ty1[li] = b.iy1;
      if (BND == DR_BOUNDARY_ZERO)
        mask[li] = (b.m00 != 0.0f ? 1 : 0) | (b.m10 != 0.0f ? 2 : 0) | (b.m01 != 0.0f ? 4 : 0) |
                   (b.m11 != 0.0f ? 8 : 0);
      if (BND == DR_BOUNDARY_WRAP) {
        q[li].ix0 = win_coord(b.tx0, b.ix0); q[li].ix1 = q[li].ix0 + 1;
        q[li].iy0 = win_coord(b.ty0, b.iy0); q[li].iy1 = q[li].iy0 + 1;
      } else {
        q[li].ix0 = b.ix0; q[li].ix1 = b.ix1; q[li].iy0 = b.iy0; q[li].iy1 = b.iy1;
      }
    }
    if (!mip) {
      q[1].ix0 = q[1].ix1 = q[1].iy0 = q[1].iy1 = 0;
      q[1].w00 = q[1].w10 = q[1].w01 = q[1].w11 = 0.0f;
    }

    // -- empty pixels (k_tex_bwd_win): lanes of one uv, summed per wave --------
    bool use0 = q[0].w00 != 0.0f || q[0].w10 != 0.0f || q[0].w01 != 0.0f || q[0].w11 != 0.0f;
    const bool use1 = q[1].w00 != 0.0f || q[1].w10 != 0.0f || q[1].w01 != 0.0f || q[1].w11 != 0.0f;
    bool in_hot = false;  // slot 0's gradient is in the hot sum
    if (!kCube) {
      const int ux = __float_as_int(uvp.x), uy = __float_as_int(uvp.y);
      const int lx = dpp_shift<0x111>(ux), ly = dpp_shift<0x111>(uy);
      const int rx = dpp_shift<0x101>(ux), ry = dpp_shift<0x101>(uy);
      const bool left = (lane & 15) != 0 && lx == ux && ly == uy;
      const bool right = (lane & 15) != 15 && rx == ux && ry == uy;
      const uint64_t cand = __ballot(use0 && ((uvp.x == 0.0f && uvp.y == 0.0f) || left || right));
      if (cand != 0ull) {  // uniform; one group a wave and tile
        const int leader = __ffsll((long long)cand) - 1;
        const int lux = __builtin_amdgcn_readlane(ux, leader), luy = __builtin_amdgcn_readlane(uy, leader);
        const int lk = __builtin_amdgcn_readlane(q[0].k, leader);
        in_hot = use0 && ux == lux && uy == luy && q[0].k == lk;
        float* base = dlevel_ptr(lk);
        if (!(hot.on && hot.ux == lux && hot.uy == luy && hot.base == base)) {
          if (hot.on) {
            hot_flush<kTaps>(hot, C, s_hot[wave]);
            __builtin_amdgcn_wave_barrier();  // (other lanes' reads, then writes)
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            for (int c = lane; c < C; c += 64) s_hot[wave][c] = 0.0;
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
          }
          hot.on = true;
          hot.ux = lux;
          hot.uy = luy;
          hot.base = base;
          hot.Wk = level_w(lk);
          hot.ix0 = __builtin_amdgcn_readlane(tx0[0], leader);
          hot.ix1 = __builtin_amdgcn_readlane(tx1[0], leader);
          hot.iy0 = __builtin_amdgcn_readlane(ty0[0], leader);
          hot.iy1 = __builtin_amdgcn_readlane(ty1[0], leader);
          hot.w00 = leader_weight(q[0], leader, 0);
          hot.w10 = leader_weight(q[0], leader, 1);
          hot.w01 = leader_weight(q[0], leader, 2);
          hot.w11 = leader_weight(q[0], leader, 3);
        }
        for (int c = 0; c < C; c += 4) {
          const float4 g = in_hot ? ld_chunk(gp + c, min(4, C - c)) : make_float4(0.f, 0.f, 0.f, 0.f);
          const float x[4] = {g.x * q[0].scale, g.y * q[0].scale, g.z * q[0].scale, g.w * q[0].scale};
          const float z = wave_sum4(x);  // lane l: total of value l & 3
          if (lane < 4 && c + lane < C) s_hot[wave][c + lane] += (double)z;
        }
        if (in_hot) use0 = false;
      }
    }

    // Whether zero_taps has anything to add: a cotangent or a weight that is
    // not finite makes the uv gradient's terms so too, and where there are none
    // it looks itself at taps of weight zero, or not finite.
    bool odd = false;
#pragma unroll
    for (int li = 0; li < (mip ? 2 : 1); ++li)
      odd = odd || (!want && valid && q[li].scale != 0.0f && !(li == 0 && in_hot) &&
                        (q[li].w00 == 0.0f ||
                         (kTaps == 4 &&
                          (q[li].w10 == 0.0f || q[li].w01 == 0.0f || q[li].w11 == 0.0f ||
                           0.0f * (q[li].w00 + q[li].w10 + q[li].w01 + q[li].w11) != 0.0f))));

    // -- boxes of the levels in use, and their windows (k_tex_bwd_win) -----------
    {
      const int lm = wave_or((use0 ? 1 << q[0].k : 0) | (use1 ? 1 << q[1].k : 0));
#pragma unroll 1
      for (int rem = lm; rem != 0; rem &= rem - 1) {
        const int L = __builtin_ctz(rem);
        int x0 = 32767, x1 = -32767, y0 = 32767, y1 = -32767;
#pragma unroll
        for (int li = 0; li < 2; ++li) {
          const bool u = li == 0 ? use0 : use1;
          if (!u || q[li].k != L) continue;
          int a0, a1, b0, b1;
          slot_box(q[li], a0, a1, b0, b1);
          x0 = min(x0, a0); x1 = max(x1, a1); y0 = min(y0, b0); y1 = max(y1, b1);
        }
        const int px = wave_min_pk16(pack16(x0, -x1));
        const int py = wave_min_pk16(pack16(y0, -y1));
        if (lane == 0) s_lbox[wave][L] = make_int2(px, py);
      }
      if (lane == 0) s_lmask[wave] = lm;
    }
    __syncthreads();
    const int4 wm = *reinterpret_cast<const int4*>(s_lmask);
    const int lmask = __builtin_amdgcn_readfirstlane(wm.x | wm.y | wm.z | wm.w);
    // lane L of each 16-lane row: level L's box, and (below) its place
    int bx = 0, by = 0, bw = 0, bh = 0;
    {
      const int L = lane & 15;
      int px = pack16(32767, 32767), py = px;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int mv = v == 0 ? wm.x : v == 1 ? wm.y : v == 2 ? wm.z : wm.w;
        if ((mv >> L) & 1) {
          const int2 b = s_lbox[v][L];
          px = pk16_min(px, b.x);
          py = pk16_min(py, b.y);
        }
      }
      const int x0 = unpack16_lo(px), x1 = -unpack16_hi(px);
      const int y0 = unpack16_lo(py), y1 = -unpack16_hi(py);
      if (((lmask >> L) & 1) && x1 >= x0 && y1 >= y0) {
        bx = x0; by = y0; bw = x1 - x0 + 1; bh = y1 - y0 + 1;
      }
    }
    constexpr int kMaxTexels = kManyPool / 4;  // with four channels in the pool
    const int fit = win_fit(bw, bh, kMaxTexels);  // (no box: 0)
    int incl = fit;  // prefix sum of the fitting areas along the 16-lane row
    {
      int t = dpp_shift<0x111>(incl);
      incl += t;
      t = dpp_shift<0x112>(incl);
      incl += t;
      t = dpp_shift<0x114>(incl);
      incl += t;
      t = dpp_shift<0x118>(incl);
      incl += t;
    }
    const bool usable = fit > 0 && incl <= kMaxTexels;
    const int at = usable ? incl - fit : -1;  // first texel in the pool, -1: no window
    // texels of the windows, and the channels that then fit (a multiple of 4)
    const int texels = wave_max(usable ? incl : 0);
    const int cap_c = texels > 0 ? min((kManyPool / texels) & ~3, (C + 3) & ~3) : (C + 3) & ~3;
    // nowin: levels in use without a window
    int nowin = 0;
#pragma unroll 1
    for (int rem = lmask; rem != 0; rem &= rem - 1) {
      const int k = __builtin_ctz(rem);
      if (__builtin_amdgcn_readlane(at, k) < 0) nowin |= 1 << k;
    }

    // a slot's tap cells in the pool (clamped into its box: a zero-weight
    // tap outside it adds 0), -1 without a window, and its run
    int o[2][4];
    RowRun run[2];
    int maxlen[2] = {0, 0};
    bool adds[2] = {false, false};
#pragma unroll
    for (int li = 0; li < (mip ? 2 : 1); ++li) {
      const bool u = li == 0 ? use0 : use1;
      const int k = q[li].k;
      const int wx = __builtin_amdgcn_ds_bpermute(k << 2, bx), wy = __builtin_amdgcn_ds_bpermute(k << 2, by);
      const int ww = __builtin_amdgcn_ds_bpermute(k << 2, bw), wh = __builtin_amdgcn_ds_bpermute(k << 2, bh);
      const int wa = __builtin_amdgcn_ds_bpermute(k << 2, at);
      const int cx0 = min(max(q[li].ix0 - wx, 0), ww - 1), cx1 = min(max(q[li].ix1 - wx, 0), ww - 1);
      const int r0 = wa + min(max(q[li].iy0 - wy, 0), wh - 1) * ww;
      const int r1 = wa + min(max(q[li].iy1 - wy, 0), wh - 1) * ww;
      o[li][0] = r0 + cx0; o[li][1] = r0 + cx1; o[li][2] = r1 + cx0; o[li][3] = r1 + cx1;
      const uint64_t key = !u ? (0x7FFFull << 45) | (uint64_t)lane
                              // (a border's merged column or row has the first coordinate twice)
                              : ((uint64_t)k << 60) | ((uint64_t)(uint16_t)q[li].ix0 << 16) |
                                    (uint16_t)q[li].iy0 |
                                    ((uint64_t)(q[li].ix0 == q[li].ix1) << 32) |
                                    ((uint64_t)(q[li].iy0 == q[li].iy1) << 33);
      run[li] = row_run(key);
      maxlen[li] = wave_max(run[li].li - run[li].s + 1);
      adds[li] = u && run[li].tail && wa >= 0;
    }

    // -- channels: d_uv and the LOD samples, the windows' sums, their flush -----
    float dfx_total = 0.0f, dfy_total = 0.0f, samp[2] = {0.0f, 0.0f};
    float dfx[2] = {0.0f, 0.0f}, dfy[2] = {0.0f, 0.0f};
#pragma unroll 1
    for (int c0 = 0; c0 < C; c0 += cap_c) {
      const int c1 = min(C, c0 + cap_c);
#pragma unroll 1
      for (int c = c0; c < c1; c += 4) {
        const int nc = min(4, C - c);
        const float4 g4 = valid ? ld_chunk(gp + c, nc) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float g[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
        for (int li = 0; li < (mip ? 2 : 1); ++li) {
          // (also a level of weight 0, and a footprint on one texel: their
          // terms are 0 unless a texel is not finite)
          if (want && valid) {
            const int k = q[li].k, Wk = level_w(k);
            const float* lv = level_ptr(k) + c;
            const uint32_t ra = (uint32_t)ty0[li] * (uint32_t)Wk, rb = (uint32_t)ty1[li] * (uint32_t)Wk;
            const float4 A0 = ld_chunk(lv + (ra + (uint32_t)tx0[li]) * (uint32_t)C, nc);
            const float4 A1 = ld_chunk(lv + (ra + (uint32_t)tx1[li]) * (uint32_t)C, nc);
            const float4 A2 = ld_chunk(lv + (rb + (uint32_t)tx0[li]) * (uint32_t)C, nc);
            const float4 A3 = ld_chunk(lv + (rb + (uint32_t)tx1[li]) * (uint32_t)C, nc);
            const float a0[4] = {A0.x, A0.y, A0.z, A0.w}, a1[4] = {A1.x, A1.y, A1.z, A1.w};
            const float a2[4] = {A2.x, A2.y, A2.z, A2.w}, a3[4] = {A3.x, A3.y, A3.z, A3.w};
            const float u = fx[li], v = fy[li];
            const float sc = mip ? q[li].scale : 1.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float t00 = a0[j] * (float)(mask[li] & 1), t10 = a1[j] * (float)((mask[li] >> 1) & 1);
              const float t01 = a2[j] * (float)((mask[li] >> 2) & 1), t11 = a3[j] * (float)(mask[li] >> 3);
              const float gc = g[j] * sc;
              dfx[li] += gc * ((1.0f - v) * (t10 - t00) + v * (t11 - t01));
              dfy[li] += gc * ((1.0f - u) * (t01 - t00) + u * (t11 - t10));
              if (mip) {
                const float sample = (1.0f - u) * (1.0f - v) * t00 + u * (1.0f - v) * t10 +
                                     (1.0f - u) * v * t01 + u * v * t11;
                samp[li] += sample * g[j];
              }
            }
          }
          const bool us = li == 0 ? use0 : use1;
          if (__ballot(us) == 0ull) continue;
          const float sc = mip ? q[li].scale : 1.0f;
          const float wt[4] = {q[li].w00, q[li].w10, q[li].w01, q[li].w11};
          float v[kTaps * 4];
#pragma unroll
          for (int t = 0; t < kTaps; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[t * 4 + j] = us ? mul0(wt[t], g[j] * sc) : 0.0f;
          row_run_scan_n(run[li], v, maxlen[li]);
          if (adds[li]) {
            double* w = win + (c - c0) * texels;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              if (j < nc) {
#pragma unroll
                for (int t = 0; t < kTaps; ++t) atomicAdd(w + j * texels + o[li][t], (double)v[t * 4 + j]);
              }
            }
          }
        }
      }
      __syncthreads();
      // consecutive lanes take consecutive channels of a texel
      const int nch = c1 - c0;
      const float inv = __builtin_amdgcn_rcpf((float)nch);
#pragma unroll 1
      for (int rem = lmask & ~nowin; rem != 0; rem &= rem - 1) {  // uniform
        const int k = __builtin_ctz(rem);
        const int W = __builtin_amdgcn_readlane(bw, k), H = __builtin_amdgcn_readlane(bh, k);
        const int a0 = __builtin_amdgcn_readlane(at, k);
        float* base = dlevel_ptr(k) + c0;
        const int Wk = level_w(k), Hk = level_h(k);
        const int X0 = win_texel<BND>(__builtin_amdgcn_readlane(bx, k), Wk);
        const int Y0 = win_texel<BND>(__builtin_amdgcn_readlane(by, k), Hk);
        const float invw = __builtin_amdgcn_rcpf((float)W);
        for (int i = tid; i < W * H * nch; i += 256) {
          // i < 2^13: the products with the reciprocals stay clear of integers
          const int e = f2i(((float)i + 0.5f) * inv), ch = i - e * nch;
          const int r = f2i(((float)e + 0.5f) * invw), x = e - r * W;
          double* p = win + ch * texels + a0 + e;
          const double v = *p;
          if (v != 0.0) {
            int X = X0 + x, Y = Y0 + r;
            if (BND == DR_BOUNDARY_WRAP) {
              X = wrap_up(X, Wk);
              Y = wrap_up(Y, Hk);
            }
            unsafeAtomicAdd(base + ((int64_t)Y * Wk + X) * C + ch, (float)v);
            *p = 0.0;
          }
        }
      }
      __syncthreads();
    }

    // -- levels without a window: a pixel at a time, lanes on (tap, channel):
    //    a texel's channels in one request ------------------------------------
    if (nowin != 0) {
#pragma unroll
      for (int li = 0; li < (mip ? 2 : 1); ++li) {
        const int k = q[li].k;
        const bool u = (li == 0 ? use0 : use1) && ((nowin >> k) & 1);
        const float sc = mip ? q[li].scale : 1.0f;
        // four pixels a step: their cotangents are loaded together
        for (uint64_t m = __ballot(u); m != 0ull;) {
          int e[4];
          float w[4];
          const float* ge[4];
          float* p[4];
          const int t = lane >> 4;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool on = m != 0ull;  // uniform; past the last one: its lane again, weight 0
            e[r] = on ? __ffsll((long long)m) - 1 : e[r > 0 ? r - 1 : 0];
            m &= m - 1;
            const int kk = __builtin_amdgcn_readlane(k, e[r]), Wk = level_w(kk);
            w[r] = on ? leader_weight(q[li], e[r], t) *
                            __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc), e[r]))
                      : 0.0f;
            const int X = (t & 1) ? __builtin_amdgcn_readlane(tx1[li], e[r]) : __builtin_amdgcn_readlane(tx0[li], e[r]);
            const int Y = (t & 2) ? __builtin_amdgcn_readlane(ty1[li], e[r]) : __builtin_amdgcn_readlane(ty0[li], e[r]);
            const int ph_e = ty * 16 + wave * 4 + (e[r] >> 4), pw_e = tx * 16 + (e[r] & 15);
            ge[r] = A.d_out + (((int64_t)n * A.Hi + ph_e) * A.Wi + pw_e) * C;
            p[r] = dlevel_ptr(kk) + ((int64_t)Y * Wk + X) * C;
          }
          for (int c = lane & 15; c < C; c += 16) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = ge[r][c];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float x = w[r] * v[r];
              if (w[r] != 0.0f && x != 0.0f) unsafeAtomicAdd(p[r] + c, x);
            }
          }
        }
      }
    }

    if (want) odd = valid && 0.0f * (dfx[0] + dfy[0] + dfx[1] + dfy[1]) != 0.0f;
    if (odd) zero_taps<FILTER, BND>(A, n, pix, in_hot);

    // -- d_uv, d_uvDA, d_bias (Texture.swift:500-520, :979-1102) -----------------
    if (kCube) {
      if (A.d_uv && valid) {
        A.d_uv[pix * 3 + 0] = 0.0f;
        A.d_uv[pix * 3 + 1] = 0.0f;
        A.d_uv[pix * 3 + 2] = 0.0f;
      }
      continue;
    }
    if (!valid) continue;
#pragma unroll
    for (int li = 0; li < (mip ? 2 : 1); ++li) {
      dfx_total += dfx[li] * (float)level_w(q[li].k);
      dfy_total += dfy[li] * (float)level_h(q[li].k);
    }
    if (A.d_uv) st_nt2(A.d_uv + pix * 2, make_float2(dfx_total, dfy_total));
    if (!mip || (!A.d_uv_da && !A.d_bias)) continue;
    const float sx = da.x * (float)A.Wt, sy = da.y * (float)A.Wt;
    const float tx_ = da.z * (float)A.Ht, ty_ = da.w * (float)A.Ht;
    const float Asq = sx * sx + tx_ * tx_;
    const float Bsq = sy * sy + ty_ * ty_;
    const float rho_sq = fmaxf(Asq, Bsq);
    const float lod_raw = 0.5f * log2f(fmaxf(rho_sq, 1e-20f));
    float4 d_eff = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!(lod_raw <= 0.0f || lod_raw >= (float)(md.L - 1))) {
      float d_lod;
      if (FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR) {
        d_lod = -samp[0] + samp[1];
      } else {  // the trilinear surrogate's two levels
        const int k0 = f2i(floorf(lod_raw));
        const int k1 = min(k0 + 1, md.L - 1);
        float s0 = 0.0f, s1 = 0.0f;
        const Bilin b0 = bilin(uvp.x, uvp.y, mip_w(md, k0), mip_h(md, k0), BND);
        const Bilin b1 = bilin(uvp.x, uvp.y, mip_w(md, k1), mip_h(md, k1), BND);
        for (int c = 0; c < C; c += 4) {
          const int nc = min(4, C - c);
          const float4 g = ld_chunk(gp + c, nc);
          const float4 a = sample_chunk(level_ptr(k0), mip_w(md, k0), C, b0, c, nc);
          const float4 b = sample_chunk(level_ptr(k1), mip_w(md, k1), C, b1, c, nc);
          s0 += a.x * g.x; s0 += a.y * g.y; s0 += a.z * g.z; s0 += a.w * g.w;
          s1 += b.x * g.x; s1 += b.y * g.y; s1 += b.z * g.z; s1 += b.w * g.w;
        }
        d_lod = -s0 + s1;
      }
      const float ln2 = 0.6931471805599453f;
      const float dlod_drho_sq = 1.0f / (2.0f * rho_sq * ln2);
      const float A_is_max = (Asq >= Bsq) ? 1.0f : 0.0f;
      const float B_is_max = 1.0f - A_is_max;
      d_eff = make_float4(d_lod * dlod_drho_sq * A_is_max * 2.0f * sx * (float)A.Wt,
                          d_lod * dlod_drho_sq * B_is_max * 2.0f * sy * (float)A.Wt,
                          d_lod * dlod_drho_sq * A_is_max * 2.0f * tx_ * (float)A.Ht,
                          d_lod * dlod_drho_sq * B_is_max * 2.0f * ty_ * (float)A.Ht);
    }
    if (A.d_uv_da) {
      const float4 ov = scaled ? make_float4(d_eff.x * s, d_eff.y * s, d_eff.z * s, d_eff.w * s) : d_eff;
      st_nt4(A.d_uv_da + pix * 4, ov);
    }
    if (A.d_bias && A.bias_map) {
      const float gm = d_eff.x * da_in.x + d_eff.y * da_in.y + d_eff.z * da_in.z + d_eff.w * da_in.w;
      A.d_bias[pix] = gm * s * 0.6931471805599453f;
    }
  }
  // the waves' empty-pixel sums, those of one footprint together (one
  // workgroup's atomics on a texel instead of four waves')
  if (lane == 0) {
    s_hbase[wave] = hot.on ? (uint64_t)hot.base : 0ull;
    s_hkey[wave] = make_int2(hot.ux, hot.uy);
  }
  __syncthreads();
  if (!hot.on) return;
  auto same = [&](int w) {
    return s_hbase[w] == s_hbase[wave] && s_hkey[w].x == s_hkey[wave].x && s_hkey[w].y == s_hkey[wave].y;
  };
  for (int w = 0; w < wave; ++w)
    if (same(w)) return;  // an earlier wave writes this footprint
  for (int w = wave + 1; w < 4; ++w)
    if (same(w))
      for (int c = lane; c < C; c += 64) s_hot[wave][c] += s_hot[w][c];
  __builtin_amdgcn_wave_barrier();  // (LDS is ordered within a wave)
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  hot_flush<kTaps>(hot, C, s_hot[wave]);
}

// Texture.swift:156: level k = 2x2 mean of level k-1.  Builds up to five
// levels at once: each workgroup reduces a 32 x 32 patch of level s, four
// channels of it, through levels s+1..s+m in LDS (m <= 5; the sizes of
// levels s..s+m-1 are even, so the patches' outputs do not straddle).  More
// than four channels take a workgroup per four, neighbours in the grid (512^2 x
// 16: nine single-level launches, 66 us; two of these, 29 us).
constexpr int kMipMaxC = 4;
constexpr int kMipPatchLog = 5, kMipPatch = 1 << kMipPatchLog;

__global__ void __launch_bounds__(256) k_mip_block(const float* __restrict__ src,
                                                   float* __restrict__ pyr, MipDesc md, int s,
                                                   int m, int C, int64_t blocks) {
  __shared__ float buf[2][256 * kMipMaxC];
  if (block_xy() >= blocks) return;
  const int Ws = md.w[s];
  const int nbx = (Ws + kMipPatch - 1) / kMipPatch;
  const int per_n = nbx * ((md.h[s] + kMipPatch - 1) / kMipPatch);
  const int chunks = (C + kMipMaxC - 1) / kMipMaxC;
  int blk = (int)block_xy() / chunks;
  const int c0 = ((int)block_xy() - blk * chunks) * kMipMaxC, nc = min(kMipMaxC, C - c0);
  const int n = blk / per_n;
  blk -= n * per_n;
  const int by = blk / nbx, bx = blk - by * nbx;
  const float* lvl = src + (int64_t)n * md.h[s] * Ws * C + c0;
  int cur = 0;
  for (int j = 1; j <= m; ++j) {
    const int e = kMipPatch >> j;  // output edge at this step
    const int k = s + j;
    const int Wk = md.w[k], Hk = md.h[k];
    float* dst = pyr + md.off[k] + (int64_t)n * Hk * Wk * C + c0;
    for (int t = threadIdx.x; t < e * e * nc; t += blockDim.x) {
      const int q = t / nc, c = t - q * nc;
      const int y = q >> (kMipPatchLog - j), x = q & (e - 1);
      const int ox = bx * e + x, oy = by * e + y;
      if (ox >= Wk || oy >= Hk) continue;  // past the level's edge
      float a, b, d, f;
      if (j == 1) {
        const int sx = 2 * ox, sy = 2 * oy;
        a = lvl[((int64_t)sy * Ws + sx) * C + c];
        b = lvl[((int64_t)sy * Ws + sx + 1) * C + c];
        d = lvl[((int64_t)(sy + 1) * Ws + sx) * C + c];
        f = lvl[((int64_t)(sy + 1) * Ws + sx + 1) * C + c];
      } else {
        const int pe = 2 * e;
        const float* pb = buf[cur ^ 1];
        a = pb[((2 * y) * pe + 2 * x) * nc + c];
        b = pb[((2 * y) * pe + 2 * x + 1) * nc + c];
        d = pb[((2 * y + 1) * pe + 2 * x) * nc + c];
        f = pb[((2 * y + 1) * pe + 2 * x + 1) * nc + c];
      }
      const float v = (((a + b) + d) + f) * 0.25f;
      buf[cur][(y * e + x) * nc + c] = v;
      dst[((int64_t)oy * Wk + ox) * C + c] = v;
    }
    __syncthreads();
    cur ^= 1;
  }
}

// k_mip_block for four channels: one output texel per thread, 16-byte
// loads and stores, the same sums in the same order.
__global__ void __launch_bounds__(256) k_mip_block_c4(const float* __restrict__ src,
                                                      float* __restrict__ pyr, MipDesc md, int s,
                                                      int m, int64_t blocks) {
  __shared__ float4 buf[2][256];
  if (block_xy() >= blocks) return;
  const int Ws = md.w[s];
  const int nbx = (Ws + kMipPatch - 1) / kMipPatch;
  const int per_n = nbx * ((md.h[s] + kMipPatch - 1) / kMipPatch);
  const int n = (int)block_xy() / per_n, blk = (int)block_xy() - n * per_n;
  const int by = blk / nbx, bx = blk - by * nbx;
  const float4* lvl = reinterpret_cast<const float4*>(src) + (int64_t)n * md.h[s] * Ws;
  auto mean4 = [](float4 a, float4 b, float4 d, float4 f) {
    return make_float4((((a.x + b.x) + d.x) + f.x) * 0.25f, (((a.y + b.y) + d.y) + f.y) * 0.25f,
                       (((a.z + b.z) + d.z) + f.z) * 0.25f, (((a.w + b.w) + d.w) + f.w) * 0.25f);
  };
  int cur = 0;
  for (int j = 1; j <= m; ++j) {
    const int e = kMipPatch >> j;  // output edge at this step
    const int k = s + j;
    const int Wk = md.w[k], Hk = md.h[k];
    float4* dst = reinterpret_cast<float4*>(pyr + md.off[k]) + (int64_t)n * Hk * Wk;
    for (int t = threadIdx.x; t < e * e; t += blockDim.x) {
      const int y = t >> (kMipPatchLog - j), x = t & (e - 1);
      const int ox = bx * e + x, oy = by * e + y;
      if (ox >= Wk || oy >= Hk) continue;  // past the level's edge
      float4 v;
      if (j == 1) {
        const int sx = 2 * ox, sy = 2 * oy;
        v = mean4(lvl[(int64_t)sy * Ws + sx], lvl[(int64_t)sy * Ws + sx + 1],
                  lvl[(int64_t)(sy + 1) * Ws + sx], lvl[(int64_t)(sy + 1) * Ws + sx + 1]);
      } else {
        const int pe = 2 * e;
        const float4* pb = buf[cur ^ 1];
        v = mean4(pb[(2 * y) * pe + 2 * x], pb[(2 * y) * pe + 2 * x + 1],
                  pb[(2 * y + 1) * pe + 2 * x], pb[(2 * y + 1) * pe + 2 * x + 1]);
      }
      buf[cur][y * e + x] = v;
      dst[(int64_t)oy * Wk + ox] = v;
    }
    __syncthreads();
    cur ^= 1;
  }
}

// Backward of the pyramid (MLX autodiff of concatenate + mean): level k's
// total cotangent is its own gradient plus 1/4 of level k+1's total,
// accumulated from the coarsest level down; level 0's total is added to
// d_tex (which already holds level 0's own gradient).  Two passes: level 1's
// totals in place (each of its values walks its chain of ancestors), then
// level 0 adds a quarter of its parent's total.  A workgroup takes 256
// values, or vectors of V = 4 where C is a multiple of 4, of one row (or
// several whole rows, where they are shorter), so consecutive threads read
// consecutive memory; one thread per texel walking the whole chain for each of
// its channels took 71 us at 512^2 x 16, this takes 16.
template <int V>
struct alignas(4 * V) VecF {
  float v[V];
};

// How a level's rows of `vals` values are dealt to workgroups: 2^log threads a
// row (at most 256), bpr workgroups for each 256 >> log rows.
struct CollapseGrid {
  int64_t rows, vals, blocks;
  int log, bpr;
};

// i / d, i below n (uniform): in 32 bits where n allows.
__device__ __forceinline__ int64_t div_n(int64_t i, int64_t n, int d) {
  return n < (1ll << 31) ? (int)i / d : i / d;
}

// A thread's row and its value of the row; false: none.
__device__ __forceinline__ bool collapse_place(const CollapseGrid& g, int64_t& row, int64_t& i) {
  const int64_t b = block_xy();
  const int64_t r = g.bpr == 1 ? b : div_n(b, g.blocks, g.bpr);
  const int part = (int)(b - r * g.bpr);
  row = (r << (8 - g.log)) + ((int)threadIdx.x >> g.log);
  i = ((int64_t)part << g.log) + ((int)threadIdx.x & ((1 << g.log) - 1));
  return row < g.rows && i < g.vals;
}

template <int V>
__global__ void __launch_bounds__(256) k_mip_collapse1(float* __restrict__ d_pyr, MipDesc md,
                                                       int G, CollapseGrid cg) {
  int64_t row, i;  // row: n * H1 + y
  if (!collapse_place(cg, row, i)) return;
  const int H1 = md.h[1];
  const int x = (int)div_n(i, cg.vals, G), c = (int)(i - (int64_t)x * G);
  const int n = (int)div_n(row, cg.rows, H1), y = (int)(row - (int64_t)n * H1);
  VecF<V>* d = reinterpret_cast<VecF<V>*>(d_pyr);
  auto at = [&](int k) -> VecF<V>& {
    const int sh = k - 1;
    return d[md.off[k] / V + (((int64_t)n * md.h[k] + (y >> sh)) * md.w[k] + (x >> sh)) * G + c];
  };
  VecF<V> acc = at(md.L - 1);
  for (int k = md.L - 2; k >= 1; --k) {
    const VecF<V> o = at(k);
#pragma unroll
    for (int j = 0; j < V; ++j) acc.v[j] = o.v[j] + acc.v[j] * 0.25f;
  }
  at(1) = acc;
}

template <int V>
__global__ void __launch_bounds__(256) k_mip_collapse0(const float* __restrict__ d_pyr, MipDesc md,
                                                       int G, CollapseGrid cg,
                                                       float* __restrict__ d_tex) {
  int64_t row, i;  // row: n * H + y
  if (!collapse_place(cg, row, i)) return;
  const int H = md.h[0];
  const int x = (int)div_n(i, cg.vals, G), c = (int)(i - (int64_t)x * G);
  const int n = (int)div_n(row, cg.rows, H), y = (int)(row - (int64_t)n * H);
  const VecF<V> t = reinterpret_cast<const VecF<V>*>(
      d_pyr)[md.off[1] / V + (((int64_t)n * md.h[1] + (y >> 1)) * md.w[1] + (x >> 1)) * G + c];
  VecF<V>* dp = reinterpret_cast<VecF<V>*>(d_tex) + row * cg.vals + i;
  VecF<V> d = *dp;
#pragma unroll
  for (int j = 0; j < V; ++j) d.v[j] += t.v[j] * 0.25f;
  *dp = d;
}

template <int FILTER, int CT, int BND, bool BIAS>
hipError_t launch_tex_bwd_win_bb(const TexBwdArgs& args, int total_tiles, hipStream_t stream) {
  static int per_cu = 0;
  if (per_cu == 0) {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_tex_bwd_win<FILTER, CT, BND, BIAS>,
                                                     kWinThreads, 0) != hipSuccess ||
        b <= 0)
      b = 2;
    per_cu = b;
  }
  const int64_t resident = (int64_t)device_cu_count() * per_cu;
  const unsigned grid = (unsigned)(total_tiles < resident ? total_tiles : resident);
  hipLaunchKernelGGL((k_tex_bwd_win<FILTER, CT, BND, BIAS>), dim3(grid), dim3(kWinThreads), 0,
                     stream, args, total_tiles);
  return hipGetLastError();
}

template <int FILTER, int CT, int BND>
hipError_t launch_tex_bwd_win_b(const TexBwdArgs& args, int total_tiles, hipStream_t stream) {
  if constexpr (FILTER == DR_FILTER_LINEAR_MIPMAP_NEAREST || FILTER == DR_FILTER_LINEAR_MIPMAP_LINEAR) {
    if (args.bias_map || args.has_bias)
      return launch_tex_bwd_win_bb<FILTER, CT, BND, true>(args, total_tiles, stream);
  }
  return launch_tex_bwd_win_bb<FILTER, CT, BND, false>(args, total_tiles, stream);
}

// The boundary mode is a compile-time constant of the windowed kernel (the
// clamp and wrap footprints need no out-of-range masks).
template <int FILTER, int CT>
hipError_t launch_tex_bwd_win(const TexBwdArgs& args, int total_tiles, hipStream_t stream) {
  if (args.boundary == DR_BOUNDARY_CLAMP)
    return launch_tex_bwd_win_b<FILTER, CT, DR_BOUNDARY_CLAMP>(args, total_tiles, stream);
  if (args.boundary == DR_BOUNDARY_WRAP)
    return launch_tex_bwd_win_b<FILTER, CT, DR_BOUNDARY_WRAP>(args, total_tiles, stream);
  return launch_tex_bwd_win_b<FILTER, CT, DR_BOUNDARY_ZERO>(args, total_tiles, stream);
}

template <int FILTER, int BND>
hipError_t launch_tex_bwd_many(const TexBwdArgs& args, int total_tiles, hipStream_t stream) {
  static int per_cu = 0;
  if (per_cu == 0) {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_tex_bwd_many<FILTER, BND>, 256, 0) !=
            hipSuccess ||
        b <= 0)
      b = 2;
    per_cu = b;
  }
  const int64_t resident = (int64_t)device_cu_count() * per_cu;
  const unsigned grid = (unsigned)(total_tiles < resident ? total_tiles : resident);
  hipLaunchKernelGGL((k_tex_bwd_many<FILTER, BND>), dim3(grid), dim3(256), 0, stream, args,
                     total_tiles);
  return hipGetLastError();
}

template <int FILTER>
hipError_t launch_tex_bwd_many_b(const TexBwdArgs& args, int total_tiles, hipStream_t stream) {
  if (args.boundary == DR_BOUNDARY_CLAMP)
    return launch_tex_bwd_many<FILTER, DR_BOUNDARY_CLAMP>(args, total_tiles, stream);
  if (args.boundary == DR_BOUNDARY_WRAP)
    return launch_tex_bwd_many<FILTER, DR_BOUNDARY_WRAP>(args, total_tiles, stream);
  return launch_tex_bwd_many<FILTER, DR_BOUNDARY_ZERO>(args, total_tiles, stream);
}

// Launches the persistent backward with as many workgroups as fit on the
// device at once.
template <int FILTER, bool CUBE, int CT>
hipError_t launch_tex_bwd(const TexBwdArgs& args, int total_tiles, hipStream_t stream) {
  static int per_cu = 0;
  if (per_cu == 0) {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_tex_bwd<FILTER, CUBE, CT>, 256, 0) !=
            hipSuccess ||
        b <= 0)
      b = 2;
    per_cu = b;
  }
  const int64_t resident = (int64_t)device_cu_count() * per_cu;
  const unsigned grid = (unsigned)(total_tiles < resident ? total_tiles : resident);
  hipLaunchKernelGGL((k_tex_bwd<FILTER, CUBE, CT>), dim3(grid), dim3(256), 0, stream, args,
                     total_tiles);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// cube maps with mip filters, and the direction gradient
// ---------------------------------------------------------------------------
// An extension of the reference, which samples cube maps bilinearly only
// (Texture.swift:75-76) and returns a zero direction gradient (:196-198).
// Faces and face (u, v) as :620-635; the face (u, v) screen derivatives
// from the direction's (dx/dX, dx/dY, dy/dX, dy/dY, dz/dX, dz/dY) by the
// chain rule through u = (sc/ma + 1)/2, v = (tc/ma + 1)/2 with the face
// fixed; then the 2D LOD, clamped bilinear taps and two-rounding trilinear
// blend of :764-863 on the chosen face of each level.  The backward adds
// the direction gradient through the sample position and, for mip
// filters, through the LOD; the pyramid is every face's 2x2 box pyramid.

struct CubeSel {
  int face, as, at, am;  // axes of sc, tc, ma
  float ss, ts, ms;      // their signs
  float sc, tc, ma;
};

__device__ __forceinline__ CubeSel cube_select(float x, float y, float z) {
  CubeSel s;
  const float ax = fabsf(x), ay = fabsf(y), az = fabsf(z);
  if (ax >= ay && ax >= az) {
    s.am = 0; s.ms = x > 0.0f ? 1.0f : -1.0f; s.ma = ax;
    s.at = 1; s.ts = -1.0f; s.tc = -y;
    s.as = 2;
    if (x > 0.0f) { s.face = 0; s.ss = -1.0f; s.sc = -z; }
    else          { s.face = 1; s.ss = 1.0f;  s.sc = z; }
  } else if (ay >= az) {
    s.am = 1; s.ms = y > 0.0f ? 1.0f : -1.0f; s.ma = ay;
    s.as = 0; s.ss = 1.0f; s.sc = x;
    s.at = 2;
    if (y > 0.0f) { s.face = 2; s.ts = 1.0f;  s.tc = z; }
    else          { s.face = 3; s.ts = -1.0f; s.tc = -z; }
  } else {
    s.am = 2; s.ms = z > 0.0f ? 1.0f : -1.0f; s.ma = az;
    s.at = 1; s.ts = -1.0f; s.tc = -y;
    s.as = 0;
    if (z > 0.0f) { s.face = 4; s.ss = 1.0f;  s.sc = x; }
    else          { s.face = 5; s.ss = -1.0f; s.sc = -x; }
  }
  return s;
}

__device__ __forceinline__ float pick3(int a, float v0, float v1, float v2) {
  return a == 0 ? v0 : (a == 1 ? v1 : v2);
}

// The direction's screen derivatives as (d/dX, d/dY) per axis.
struct DirDA {
  float x[3], y[3];
};

// Face (u_X, u_Y, v_X, v_Y) from the direction's derivatives.
__device__ __forceinline__ float4 cube_face_da(const CubeSel& s, const DirDA& d) {
  const float inv = 0.5f / (s.ma * s.ma);
  const float sX = s.ss * pick3(s.as, d.x[0], d.x[1], d.x[2]);
  const float sY = s.ss * pick3(s.as, d.y[0], d.y[1], d.y[2]);
  const float tX = s.ts * pick3(s.at, d.x[0], d.x[1], d.x[2]);
  const float tY = s.ts * pick3(s.at, d.y[0], d.y[1], d.y[2]);
  const float mX = s.ms * pick3(s.am, d.x[0], d.x[1], d.x[2]);
  const float mY = s.ms * pick3(s.am, d.y[0], d.y[1], d.y[2]);
  return make_float4((sX * s.ma - s.sc * mX) * inv, (sY * s.ma - s.sc * mY) * inv,
                     (tX * s.ma - s.tc * mX) * inv, (tY * s.ma - s.tc * mY) * inv);
}

struct CubeArgs {
  const float* tex;  // [Nt, 6, Ht, Wt, C]
  const float* pyr;  // levels 1..L-1 of the Nt*6 faces
  MipDesc md;        // built for Nt*6 textures
  int64_t tex_stride;  // 6*Ht*Wt*C, or 0 for one shared cube map
  int Ht, Wt, C;
  const float* dir;      // [N, Hi, Wi, 3]
  const float* dir_da;   // [N, Hi, Wi, 6] (mip modes)
  const float* bias_map;
  float scale_bias;
  int has_bias;
  int64_t P;
  int HWi;
  int Wi;      // image width (the forward's 16x16 tiles)
  float* out;  // forward
  // backward
  const float* d_out;
  float* d_tex;
  float* d_pyr;
  float* d_dir;     // NULL: not requested
  int dir_grad;     // 0: d_dir is written as zeros (the reference's value)
  float* d_dir_da;
  float* d_bias;
};

__device__ __forceinline__ const float* cube_level(const CubeArgs& A, int n, int face, int k,
                                                   int Hk, int Wk) {
  if (k == 0) return A.tex + n * A.tex_stride + (int64_t)face * A.Ht * A.Wt * A.C;
  const int64_t nt = A.tex_stride ? n : 0;
  return A.pyr + mip_off(A.md, k) + (nt * 6 + face) * (int64_t)Hk * Wk * A.C;
}

__device__ __forceinline__ float* cube_dlevel(const CubeArgs& A, int n, int face, int k, int Hk,
                                              int Wk) {
  if (k == 0) return A.d_tex + n * A.tex_stride + (int64_t)face * A.Ht * A.Wt * A.C;
  const int64_t nt = A.tex_stride ? n : 0;
  return A.d_pyr + mip_off(A.md, k) + (nt * 6 + face) * (int64_t)Hk * Wk * A.C;
}

// Per-pixel set-up shared by both passes.
struct CubePx {
  CubeSel s;
  float u, v, inv_ma, bscale;
  bool scaled;
  DirDA dd, dd_in;  // folded (dd) and as given (dd_in)
  float4 da;        // face derivatives
  Lod ld;
};

template <int MODE>
__device__ __forceinline__ CubePx cube_px(const CubeArgs& A, int64_t pix) {
  CubePx p;
  // the direction, its derivatives and the bias are loaded together, ahead
  // of the face selection's branches (one round trip instead of two)
  const float* dp = A.dir + pix * 3;
  const float x = dp[0], y = dp[1], z = dp[2];
  float2 a = make_float2(0.f, 0.f), b = a, c = a;
  float bm = 0.0f;
  if (MODE > 0) {
    const float2* q = reinterpret_cast<const float2*>(A.dir_da + pix * 6);
    a = q[0];
    b = q[1];
    c = q[2];
    if (A.bias_map) bm = A.bias_map[pix];
  }
  p.s = cube_select(x, y, z);
  p.inv_ma = 1.0f / p.s.ma;
  p.u = (p.s.sc * p.inv_ma + 1.0f) * 0.5f;
  p.v = (p.s.tc * p.inv_ma + 1.0f) * 0.5f;
  p.ld.k0 = p.ld.k1 = 0;
  p.ld.frac = 0.0f;
  p.scaled = false;
  p.bscale = 1.0f;
  if (MODE > 0) {
    p.dd_in.x[0] = a.x; p.dd_in.y[0] = a.y;
    p.dd_in.x[1] = b.x; p.dd_in.y[1] = b.y;
    p.dd_in.x[2] = c.x; p.dd_in.y[2] = c.y;
    p.dd = p.dd_in;
    p.scaled = A.bias_map != nullptr || A.has_bias;
    if (p.scaled) {
      p.bscale = A.bias_map ? (A.has_bias ? exp2f(bm) * A.scale_bias : exp2f(bm)) : A.scale_bias;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        p.dd.x[i] = p.dd_in.x[i] * p.bscale;
        p.dd.y[i] = p.dd_in.y[i] * p.bscale;
      }
    }
    p.da = cube_face_da(p.s, p.dd);
    p.ld = mip_lod(p.da, A.Ht, A.Wt, A.md.L, MODE == 2);
  }
  return p;
}

// MODE: 1 = mip-nearest, 2 = trilinear (bilinear cube sampling is k_tex_fwd).
// One 16x16 pixel tile per workgroup (a 16x4 strip per wave), so a wave's
// texel gathers share cache lines along both image axes.
template <int MODE, int CT>
__global__ void __launch_bounds__(256) k_cube_fwd(CubeArgs A) {
  const int Wi = A.Wi, Hi = A.HWi / Wi;
  const int ntx = (Wi + 15) >> 4, tiles = ntx * ((Hi + 15) >> 4);
  const int b = (int)blockIdx.x, n = b / tiles, tile = b - n * tiles;
  const int ty = tile / ntx, tx = tile - ty * ntx;
  const int ph = ty * 16 + ((int)threadIdx.x >> 4), pw = tx * 16 + ((int)threadIdx.x & 15);
  if (ph >= Hi || pw >= Wi) return;
  const int64_t pix = ((int64_t)n * Hi + ph) * Wi + pw;
  const int C = dimC<CT>(A.C);
  const CubePx p = cube_px<MODE>(A, pix);
  float* op = A.out + pix * C;
  float acc[kMaxC];
  for (int li = 0; li < 2; ++li) {
    const int k = li == 0 ? p.ld.k0 : p.ld.k1;
    const int Hk = mip_h(A.md, k), Wk = mip_w(A.md, k);
    const float* lv = cube_level(A, n, p.s.face, k, Hk, Wk);
    const Bilin b = bilin(p.u, p.v, Wk, Hk, DR_BOUNDARY_CLAMP);
    const float wgt = li == 0 ? (1.0f - p.ld.frac) : p.ld.frac;
    if constexpr (CT > 0) {
      float t00[kMaxC], t10[kMaxC], t01[kMaxC], t11[kMaxC];
      load_texel<CT>(lv + ((int64_t)b.iy0 * Wk + b.ix0) * C, C, t00);
      load_texel<CT>(lv + ((int64_t)b.iy0 * Wk + b.ix1) * C, C, t10);
      load_texel<CT>(lv + ((int64_t)b.iy1 * Wk + b.ix0) * C, C, t01);
      load_texel<CT>(lv + ((int64_t)b.iy1 * Wk + b.ix1) * C, C, t11);
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const float sample = b.w00 * t00[c] + b.w10 * t10[c] + b.w01 * t01[c] + b.w11 * t11[c];
        acc[c] = li == 0 ? wgt * sample : acc[c] + wgt * sample;
      }
    } else {
      for (int c = 0; c < C; ++c) {
        const float t00 = lv[((int64_t)b.iy0 * Wk + b.ix0) * C + c];
        const float t10 = lv[((int64_t)b.iy0 * Wk + b.ix1) * C + c];
        const float t01 = lv[((int64_t)b.iy1 * Wk + b.ix0) * C + c];
        const float t11 = lv[((int64_t)b.iy1 * Wk + b.ix1) * C + c];
        const float sample = b.w00 * t00 + b.w10 * t10 + b.w01 * t01 + b.w11 * t11;
        op[c] = li == 0 ? wgt * sample : op[c] + wgt * sample;
      }
    }
  }
  if constexpr (CT > 0) {
#pragma unroll
    for (int c = 0; c < CT; ++c) op[c] = acc[c];
  }
}

// MODE: 0 = bilinear (only with the direction gradient), 1 / 2 as above.
// One pixel of the backward; every lane of the wave calls it (the scatter
// groups lanes across the wave), `valid` marks the lanes with a pixel.
template <int MODE, int CT>
__device__ __forceinline__ void cube_bwd_px(const CubeArgs& A, int64_t pix, bool valid, int n,
                                            FootAcc<(CT > 0 ? CT : 1)>& acc0,
                                            CubeTable<CT>& tab) {
  const int C = dimC<CT>(A.C);
  const float* gp = A.d_out + pix * C;
  float g[CT > 0 ? CT : 1];
  if constexpr (CT > 0) load_texel<CT>(gp, C, g);  // pix is clamped into the image
  const CubePx p = cube_px<MODE>(A, pix);
  if constexpr (CT > 0) {
#pragma unroll
    for (int c = 0; c < CT; ++c) g[c] = valid ? g[c] : 0.0f;
  }
  const float* gsrc = CT > 0 ? g : gp;  // run-time C reads d_out directly
  const CubeSel& s = p.s;
  // Trilinear with the LOD inside (0, L-1): the LOD gradient needs both
  // levels' samples (:1011-1102), and those levels are the two the filter
  // blends (the same LOD expression), so the texels read here serve it too.
  float lod_raw = 0.0f, Asq = 0.0f, Bsq = 0.0f;
  bool lod_in = false;
  if (MODE > 0) {
    const float sx = p.da.x * (float)A.Wt, sy = p.da.y * (float)A.Wt;
    const float tx_ = p.da.z * (float)A.Ht, ty_ = p.da.w * (float)A.Ht;
    Asq = sx * sx + tx_ * tx_;
    Bsq = sy * sy + ty_ * ty_;
    lod_raw = 0.5f * log2f(fmaxf(fmaxf(Asq, Bsq), 1e-20f));
    lod_in = lod_raw > 0.0f && lod_raw < (float)(A.md.L - 1);
  }
  const bool lod_here = MODE == 2 && valid && lod_in;
  // sample position gradient (:934-999) and the pyramid scatter (:870-932);
  // a level of zero weight adds nothing and is skipped (uniformly per wave)
  float du = 0.0f, dv = 0.0f, d_lod = 0.0f;
  for (int li = 0; li < (MODE == 0 ? 1 : 2); ++li) {
    const int k = li == 0 ? p.ld.k0 : p.ld.k1;
    const float scale = MODE == 0 ? 1.0f : (li == 0 ? (1.0f - p.ld.frac) : p.ld.frac);
    const bool on = valid && scale != 0.0f;
    const bool rd = on || lod_here;  // the texels are read
    if (__ballot(rd) == 0ull) continue;
    const int Hk = mip_h(A.md, k), Wk = mip_w(A.md, k);
    const float* lv = cube_level(A, n, s.face, k, Hk, Wk);
    float* dl = cube_dlevel(A, n, s.face, k, Hk, Wk);
    const Bilin b = bilin(p.u, p.v, Wk, Hk, DR_BOUNDARY_CLAMP);
    if (__ballot(on)) {
      if (li == 0)
        scatter_footprint<CT, true, CubeTable<CT>>(on, dl, Wk, C, b, gsrc, scale, acc0, tab);
      else
        scatter_footprint<CT, false, CubeTable<CT>>(on, dl, Wk, C, b, gsrc, scale, acc0, tab);
    }
    if (!rd) continue;
    const float sign = li == 0 ? -1.0f : 1.0f;
    float dfx = 0.0f, dfy = 0.0f;
    // a texel's channels in one load (CT > 0) rather than one per channel
    // (4096 x 256^2, 6 x 512^2 x 3: 37.7 -> 36.1 ms)
    float q00[kMaxC], q10[kMaxC], q01[kMaxC], q11[kMaxC];
    if constexpr (CT > 0) {
      load_texel<CT>(lv + ((int64_t)b.iy0 * Wk + b.ix0) * C, C, q00);
      load_texel<CT>(lv + ((int64_t)b.iy0 * Wk + b.ix1) * C, C, q10);
      load_texel<CT>(lv + ((int64_t)b.iy1 * Wk + b.ix0) * C, C, q01);
      load_texel<CT>(lv + ((int64_t)b.iy1 * Wk + b.ix1) * C, C, q11);
    }
    for (int c = 0; c < C; ++c) {
      const float t00 = CT > 0 ? q00[c] : lv[((int64_t)b.iy0 * Wk + b.ix0) * C + c];
      const float t10 = CT > 0 ? q10[c] : lv[((int64_t)b.iy0 * Wk + b.ix1) * C + c];
      const float t01 = CT > 0 ? q01[c] : lv[((int64_t)b.iy1 * Wk + b.ix0) * C + c];
      const float t11 = CT > 0 ? q11[c] : lv[((int64_t)b.iy1 * Wk + b.ix1) * C + c];
      const float gs = gsrc[c] * scale;
      dfx += gs * ((1.0f - b.fy) * (t10 - t00) + b.fy * (t11 - t01));
      dfy += gs * ((1.0f - b.fx) * (t01 - t00) + b.fx * (t11 - t10));
      if (lod_here) {
        const float sample = b.w00 * t00 + b.w10 * t10 + b.w01 * t01 + b.w11 * t11;
        d_lod += sign * sample * gsrc[c];
      }
    }
    du += dfx * (float)Wk;
    dv += dfy * (float)Hk;
  }
  if (!valid) return;
  const float* g_ = gsrc;
  const float inv2 = 0.5f / (s.ma * s.ma);
  // d u / d dir = inv2 * (ss*ma e_as - sc*ms e_am), likewise v; the axes
  // are distinct, so each sum below lands in its own component
  const float g_as = du * (s.ss * s.ma * inv2);
  const float g_at = dv * (s.ts * s.ma * inv2);
  const float g_am = -((du * s.sc + dv * s.tc) * s.ms * inv2);
  float gdd_x[3] = {0.0f, 0.0f, 0.0f}, gdd_y[3] = {0.0f, 0.0f, 0.0f};
  float l_as = 0.0f, l_at = 0.0f, l_am = 0.0f;
  if (MODE > 0) {
    const float sx = p.da.x * (float)A.Wt, sy = p.da.y * (float)A.Wt;
    const float tx_ = p.da.z * (float)A.Ht, ty_ = p.da.w * (float)A.Ht;
    const float rho_sq = fmaxf(Asq, Bsq);
    if (lod_in) {
      if (MODE == 1) {  // mip-nearest: the LOD's two levels are not the one sampled
        const int j0 = f2i(floorf(lod_raw));
        const int j1 = min(j0 + 1, A.md.L - 1);
        for (int li = 0; li < 2; ++li) {
          const int k = li == 0 ? j0 : j1;
          const float sign = li == 0 ? -1.0f : 1.0f;
          const int Hk = mip_h(A.md, k), Wk = mip_w(A.md, k);
          const float* lv = cube_level(A, n, s.face, k, Hk, Wk);
          const Bilin b = bilin(p.u, p.v, Wk, Hk, DR_BOUNDARY_CLAMP);
          for (int c = 0; c < C; ++c) {
            const float t00 = lv[((int64_t)b.iy0 * Wk + b.ix0) * C + c];
            const float t10 = lv[((int64_t)b.iy0 * Wk + b.ix1) * C + c];
            const float t01 = lv[((int64_t)b.iy1 * Wk + b.ix0) * C + c];
            const float t11 = lv[((int64_t)b.iy1 * Wk + b.ix1) * C + c];
            const float sample = b.w00 * t00 + b.w10 * t10 + b.w01 * t01 + b.w11 * t11;
            d_lod += sign * sample * g_[c];
          }
        }
      }
      const float ln2 = 0.6931471805599453f;
      const float dlod_drho_sq = 1.0f / (2.0f * rho_sq * ln2);
      const float A_is_max = (Asq >= Bsq) ? 1.0f : 0.0f;
      const float B_is_max = 1.0f - A_is_max;
      const float duX = d_lod * dlod_drho_sq * A_is_max * 2.0f * sx * (float)A.Wt;
      const float duY = d_lod * dlod_drho_sq * B_is_max * 2.0f * sy * (float)A.Wt;
      const float dvX = d_lod * dlod_drho_sq * A_is_max * 2.0f * tx_ * (float)A.Ht;
      const float dvY = d_lod * dlod_drho_sq * B_is_max * 2.0f * ty_ * (float)A.Ht;
      const DirDA& d6 = p.dd;
      const float sX = s.ss * pick3(s.as, d6.x[0], d6.x[1], d6.x[2]);
      const float sY = s.ss * pick3(s.as, d6.y[0], d6.y[1], d6.y[2]);
      const float tX = s.ts * pick3(s.at, d6.x[0], d6.x[1], d6.x[2]);
      const float tY = s.ts * pick3(s.at, d6.y[0], d6.y[1], d6.y[2]);
      const float mX = s.ms * pick3(s.am, d6.x[0], d6.x[1], d6.x[2]);
      const float mY = s.ms * pick3(s.am, d6.y[0], d6.y[1], d6.y[2]);
      // through the direction derivatives: u_X = inv2 * (sX*ma - sc*mX), ...
      const float ex_as = duX * s.ss * s.ma * inv2, ey_as = duY * s.ss * s.ma * inv2;
      const float ex_at = dvX * s.ts * s.ma * inv2, ey_at = dvY * s.ts * s.ma * inv2;
      const float ex_am = -((duX * s.sc + dvX * s.tc) * s.ms * inv2);
      const float ey_am = -((duY * s.sc + dvY * s.tc) * s.ms * inv2);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        gdd_x[i] = i == s.as ? ex_as : (i == s.at ? ex_at : ex_am);
        gdd_y[i] = i == s.as ? ey_as : (i == s.at ? ey_at : ey_am);
      }
      // through the direction: d u_X / d sc = -inv2*mX,
      // d u_X / d ma = inv2*sX - 2*u_X/ma, likewise for the others
      l_as = -((duX * mX + duY * mY) * s.ss * inv2);
      l_at = -((dvX * mX + dvY * mY) * s.ts * inv2);
      l_am = s.ms * (duX * (sX * inv2 - 2.0f * p.da.x * p.inv_ma) +
                     duY * (sY * inv2 - 2.0f * p.da.y * p.inv_ma) +
                     dvX * (tX * inv2 - 2.0f * p.da.z * p.inv_ma) +
                     dvY * (tY * inv2 - 2.0f * p.da.w * p.inv_ma));
    }
  }
  if (A.d_dir) {
    float o[3] = {0.0f, 0.0f, 0.0f};
    if (A.dir_grad) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const float a = i == s.as ? g_as : (i == s.at ? g_at : g_am);
        const float l = i == s.as ? l_as : (i == s.at ? l_at : l_am);
        o[i] = a + l;
      }
    }
    float* dd_o = A.d_dir + pix * 3;
    dd_o[0] = o[0];
    dd_o[1] = o[1];
    dd_o[2] = o[2];
  }
  if (MODE > 0 && A.d_dir_da) {
    float2* q = reinterpret_cast<float2*>(A.d_dir_da + pix * 6);
    const float sc_ = p.scaled ? p.bscale : 1.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) q[i] = make_float2(gdd_x[i] * sc_, gdd_y[i] * sc_);
  }
  if (MODE > 0 && A.d_bias && A.bias_map) {
    float gm = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) gm = gm + gdd_x[i] * p.dd_in.x[i] + gdd_y[i] * p.dd_in.y[i];
    A.d_bias[pix] = gm * p.bscale * 0.6931471805599453f;
  }
}

// Persistent 16x16 pixel tiles, one pixel per thread: each tile's d_tex /
// d_pyramid contributions are summed in the LDS table (large groups of
// lanes on one footprint across the wave first, the most frequent one in a
// per-wave accumulator kept across tiles), then written out.
template <int MODE, int CT>
__global__ void __launch_bounds__(256) k_cube_bwd(CubeArgs A, int Hi, int Wi, int ntx,
                                                  int total_tiles) {
  __shared__ CubeTable<CT> tab;
  __shared__ FootAccLds<(CT > 0 ? CT : 1), 4> s_acc;
  FootAcc<(CT > 0 ? CT : 1)> acc0;
  acc_init(acc0);
  cube_table_clear<CT>(tab);
  __syncthreads();
  const int tiles = ntx * ((Hi + 15) >> 4);
  for (int t = (int)blockIdx.x; t < total_tiles; t += (int)gridDim.x) {
    const int n = t / tiles, tile = t - n * tiles;
    const int ty = tile / ntx, tx = tile - ty * ntx;
    const int ph = ty * 16 + ((int)threadIdx.x >> 4), pw = tx * 16 + ((int)threadIdx.x & 15);
    const bool valid = ph < Hi && pw < Wi;
    const int64_t pix = ((int64_t)n * Hi + min(ph, Hi - 1)) * Wi + min(pw, Wi - 1);
    cube_bwd_px<MODE, CT>(A, pix, valid, n, acc0, tab);
    __syncthreads();
    cube_table_flush<CT>(tab);
  }
  acc_flush_group(acc0, s_acc);
}

}  // namespace dr

using namespace dr;

static int build_desc(int Ht, int Wt, int C, int Nt, int L, MipDesc& md) {
  DR_CHECK_ARG(L >= 1 && L <= kMaxLevels, "texture: mip level count out of range");
  md.L = L;
  md.nc = (int64_t)Nt * C;
  int h = Ht, w = Wt;
  int64_t off = 0;
  for (int k = 0; k < L; ++k) {
    md.h[k] = h;
    md.w[k] = w;
    md.off[k] = k == 0 ? 0 : off;
    if (k > 0) off += (int64_t)Nt * h * w * C;
    if (k + 1 < L) {
      DR_CHECK_ARG(h >= 2 && w >= 2 && h % 2 == 0 && w % 2 == 0,
                   "texture: mip levels need even sizes down to the last level");
      h /= 2;
      w /= 2;
    }
  }
  for (int k = L; k < kMaxLevels; ++k) {
    md.h[k] = md.w[k] = 1;
    md.off[k] = 0;
  }
  return DR_OK;
}

extern "C" int dr_texture_mip_levels(int H, int W, int max_level, int32_t* level_h,
                                     int32_t* level_w) {
  int n = 0;
  if (level_h) level_h[n] = H;
  if (level_w) level_w[n] = W;
  ++n;
  while (H >= 2 && W >= 2 && H % 2 == 0 && W % 2 == 0 && n < 32) {
    if (max_level >= 0 && n > max_level) break;
    H /= 2;
    W /= 2;
    if (level_h) level_h[n] = H;
    if (level_w) level_w[n] = W;
    ++n;
  }
  return n;
}

extern "C" int64_t dr_texture_mip_size(int Nt, int H, int W, int C, int L) {
  int64_t s = 0;
  for (int k = 1; k < L; ++k) {
    H /= 2;
    W /= 2;
    s += (int64_t)Nt * H * W * C;
  }
  return s;
}

extern "C" int dr_texture_build_mip(const float* tex, int Nt, int H, int W, int C, int L,
                                    float* pyramid, dr_stream_t stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  (void)hipGetLastError();
  DR_CHECK_ARG(tex && Nt >= 1 && C >= 1, "texture_build_mip: bad arguments");
  MipDesc md;
  int st = build_desc(H, W, C, Nt, L, md);
  if (st) return st;
  if (L > 1) DR_CHECK_ARG(pyramid != nullptr, "texture_build_mip: null pyramid");
  for (int sl = 0; sl < L - 1;) {
    const int m = (L - 1 - sl) < 5 ? (L - 1 - sl) : 5;
    const float* src = sl == 0 ? tex : pyramid + md.off[sl];
    const int64_t patches = (int64_t)((md.h[sl] + kMipPatch - 1) / kMipPatch) *
                            ((md.w[sl] + kMipPatch - 1) / kMipPatch) * Nt;
    const int64_t blocks = patches * ((C + kMipMaxC - 1) / kMipMaxC);
    DR_CHECK_ARG(blocks < ((int64_t)1 << 31), "texture_build_mip: texture too large");
    {
      DR_TIMED("k_mip_block", stream);
      if (C == 4 && (((uintptr_t)src | (uintptr_t)pyramid) & 15) == 0)
        hipLaunchKernelGGL(k_mip_block_c4, grid_xy(blocks), dim3(256), 0, stream, src, pyramid, md,
                           sl, m, blocks);
      else
        hipLaunchKernelGGL(k_mip_block, grid_xy(blocks), dim3(256), 0, stream, src, pyramid, md, sl,
                           m, C, blocks);
    }
    DR_CHECK_LAUNCH();
    sl += m;
  }
  return DR_OK;
}

static int check_tex(const float* tex, const float* pyr, int Nt, int N, int Ht, int Wt, int C,
                     int L, const float* uv, const float* uv_da, int filter, int boundary,
                     MipDesc& md) {
  DR_CHECK_ARG(tex && uv && N >= 1 && Ht >= 1 && Wt >= 1 && C >= 1, "texture: bad arguments");
  DR_CHECK_ARG(Nt == 1 || Nt == N, "texture: tex batch dim incompatible with uv batch");
  DR_CHECK_ARG(filter >= 0 && filter <= 3 && boundary >= 0 && boundary <= 3,
               "texture: bad filter / boundary");
  const bool cube = boundary == DR_BOUNDARY_CUBE;
  DR_CHECK_ARG(!cube || filter != DR_FILTER_NEAREST,
               "texture: cube textures support the linear and mipmap filterModes");
  const int ntex = cube ? Nt * 6 : Nt;  // a cube map is six face textures
  const bool mip = filter >= DR_FILTER_LINEAR_MIPMAP_NEAREST;
  if (mip) {
    DR_CHECK_ARG(uv_da != nullptr, "texture: mipmap filterModes require uvDA");
    DR_CHECK_ARG(L == 1 || pyr != nullptr, "texture: mip pyramid missing");
    return build_desc(Ht, Wt, C, ntex, L, md);
  }
  return build_desc(Ht, Wt, C, ntex, 1, md);
}

#define DR_TEX_C_DISPATCH(KERNEL, F, BNDV, GRID, ...)                                        \
  do {                                                                                        \
    switch (C) {                                                                              \
      case 1: hipLaunchKernelGGL((KERNEL<F, BNDV, 1>), GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      case 2: hipLaunchKernelGGL((KERNEL<F, BNDV, 2>), GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      case 3: hipLaunchKernelGGL((KERNEL<F, BNDV, 3>), GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      case 4: hipLaunchKernelGGL((KERNEL<F, BNDV, 4>), GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
      default: hipLaunchKernelGGL((k_tex_fwd_many<F, BNDV>), GRID, dim3(256), 0, stream, __VA_ARGS__); break; \
    }                                                                                         \
  } while (0)

#define DR_TEX_B_DISPATCH(KERNEL, F, GRID, ...)                                                          \
  do {                                                                                                  \
    if (boundary == DR_BOUNDARY_CLAMP) DR_TEX_C_DISPATCH(KERNEL, F, DR_BOUNDARY_CLAMP, GRID, __VA_ARGS__); \
    else if (boundary == DR_BOUNDARY_WRAP) DR_TEX_C_DISPATCH(KERNEL, F, DR_BOUNDARY_WRAP, GRID, __VA_ARGS__); \
    else DR_TEX_C_DISPATCH(KERNEL, F, DR_BOUNDARY_ZERO, GRID, __VA_ARGS__);                             \
  } while (0)

#define DR_TEX_DISPATCH(KERNEL, GRID, ...)                                                              \
  do {                                                                                                  \
    if (boundary == DR_BOUNDARY_CUBE) DR_TEX_C_DISPATCH(KERNEL, DR_FILTER_LINEAR, DR_BOUNDARY_CUBE, GRID, __VA_ARGS__); \
    else if (filter == DR_FILTER_NEAREST) DR_TEX_B_DISPATCH(KERNEL, DR_FILTER_NEAREST, GRID, __VA_ARGS__); \
    else if (filter == DR_FILTER_LINEAR) DR_TEX_B_DISPATCH(KERNEL, DR_FILTER_LINEAR, GRID, __VA_ARGS__); \
    else if (filter == DR_FILTER_LINEAR_MIPMAP_NEAREST) DR_TEX_B_DISPATCH(KERNEL, DR_FILTER_LINEAR_MIPMAP_NEAREST, GRID, __VA_ARGS__); \
    else DR_TEX_B_DISPATCH(KERNEL, DR_FILTER_LINEAR_MIPMAP_LINEAR, GRID, __VA_ARGS__);   \
  } while (0)

// d_tex += the pyramid's gradient (the backward of the 2x2 means).
static int mip_collapse(float* d_pyr, const MipDesc& md, int ntex, int Ht, int Wt, int C,
                        float* d_tex, hipStream_t stream) {
  DR_TIMED("k_mip_collapse", stream);
  const bool vec = C % 4 == 0 && (((uintptr_t)d_pyr | (uintptr_t)d_tex) & 15) == 0;
  const int G = vec ? C / 4 : C;  // values of a texel
  auto deal = [&](int h, int w) {
    CollapseGrid g;
    g.rows = (int64_t)ntex * h;
    g.vals = (int64_t)w * G;
    g.log = 0;
    while (g.log < 8 && (1 << g.log) < g.vals) ++g.log;
    g.bpr = (int)((g.vals + (1 << g.log) - 1) >> g.log);
    const int per = 256 >> g.log;  // rows of a workgroup
    g.blocks = (g.rows + per - 1) / per * g.bpr;
    return g;
  };
  if (md.L >= 3) {
    const CollapseGrid g = deal(md.h[1], md.w[1]);
    if (vec)
      hipLaunchKernelGGL(k_mip_collapse1<4>, grid_xy(g.blocks), dim3(256), 0, stream, d_pyr, md, G, g);
    else
      hipLaunchKernelGGL(k_mip_collapse1<1>, grid_xy(g.blocks), dim3(256), 0, stream, d_pyr, md, G, g);
    DR_CHECK_LAUNCH();
  }
  const CollapseGrid g = deal(Ht, Wt);
  if (vec)
    hipLaunchKernelGGL(k_mip_collapse0<4>, grid_xy(g.blocks), dim3(256), 0, stream, d_pyr, md, G, g, d_tex);
  else
    hipLaunchKernelGGL(k_mip_collapse0<1>, grid_xy(g.blocks), dim3(256), 0, stream, d_pyr, md, G, g, d_tex);
  DR_CHECK_LAUNCH();
  return DR_OK;
}

static CubeArgs cube_args(const float* tex, const float* pyr, const MipDesc& md,
                          int64_t tex_stride, int Ht, int Wt, int C, const float* dir,
                          const float* dir_da, const float* bias_map, float scale_bias,
                          int has_bias, int64_t P, int HWi) {
  CubeArgs A{};
  A.tex = tex;
  A.pyr = pyr;
  A.md = md;
  A.tex_stride = tex_stride;
  A.Ht = Ht;
  A.Wt = Wt;
  A.C = C;
  A.dir = dir;
  A.dir_da = dir_da;
  A.bias_map = bias_map;
  A.scale_bias = scale_bias;
  A.has_bias = has_bias;
  A.P = P;
  A.HWi = HWi;
  return A;
}

#define DR_CUBE_DISPATCH(KERNEL, MODE, GRID, ARGS)                                           \
  do {                                                                                        \
    switch (C) {                                                                              \
      case 1: hipLaunchKernelGGL((KERNEL<MODE, 1>), GRID, dim3(256), 0, stream, ARGS); break; \
      case 2: hipLaunchKernelGGL((KERNEL<MODE, 2>), GRID, dim3(256), 0, stream, ARGS); break; \
      case 3: hipLaunchKernelGGL((KERNEL<MODE, 3>), GRID, dim3(256), 0, stream, ARGS); break; \
      case 4: hipLaunchKernelGGL((KERNEL<MODE, 4>), GRID, dim3(256), 0, stream, ARGS); break; \
      default: hipLaunchKernelGGL((KERNEL<MODE, 0>), GRID, dim3(256), 0, stream, ARGS); break; \
    }                                                                                         \
  } while (0)

extern "C" int dr_texture_fwd(const float* tex, const float* pyramid, int Nt, int Ht, int Wt,
                              int C, int L, const float* uv, const float* uv_da,
                              const float* bias_map, float bias, int filter, int boundary, int N,
                              int Hi, int Wi, float* out, dr_stream_t stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  (void)hipGetLastError();
  MipDesc md;
  int st = check_tex(tex, pyramid, Nt, N, Ht, Wt, C, L, uv, uv_da, filter, boundary, md);
  if (st) return st;
  DR_CHECK_ARG(out != nullptr && Hi >= 1 && Wi >= 1, "texture: bad output");
  const bool cube = boundary == DR_BOUNDARY_CUBE;
  const int64_t tex_stride = Nt == 1 ? 0 : (int64_t)(cube ? 6 : 1) * Ht * Wt * C;
  const int64_t P = (int64_t)N * Hi * Wi;
  const float scale_bias = exp2f(bias);
  const int has_bias = bias != 0.0f;
  const dim3 grid(grid_for(P, 256));
  if (cube && filter >= DR_FILTER_LINEAR_MIPMAP_NEAREST) {
    CubeArgs A = cube_args(tex, pyramid, md, tex_stride, Ht, Wt, C, uv, uv_da, bias_map,
                           scale_bias, has_bias, P, Hi * Wi);
    A.out = out;
    A.Wi = Wi;
    const int64_t tiles = (int64_t)N * ((Hi + 15) / 16) * ((Wi + 15) / 16);
    DR_CHECK_ARG(tiles <= INT32_MAX, "texture: too many pixel tiles");
    const dim3 tgrid((unsigned)tiles);
    DR_TIMED("k_cube_fwd", stream);
    if (filter == DR_FILTER_LINEAR_MIPMAP_LINEAR) DR_CUBE_DISPATCH(k_cube_fwd, 2, tgrid, A);
    else DR_CUBE_DISPATCH(k_cube_fwd, 1, tgrid, A);
    DR_CHECK_LAUNCH();
    return DR_OK;
  }
  const int64_t px_tiles = (int64_t)N * ((Hi + 15) / 16) * ((Wi + 15) / 16);
  DR_CHECK_ARG(px_tiles < ((int64_t)1 << 31), "texture: too many pixels");
  DR_TIMED("k_tex_fwd", stream);
  DR_TEX_DISPATCH(k_tex_fwd, dim3((unsigned)px_tiles), tex, pyramid, md, tex_stride, Ht, Wt, C, uv,
                  uv_da, bias_map, scale_bias, has_bias, P, Hi, Wi, out);
  DR_CHECK_LAUNCH();
  return DR_OK;
}

// The cube backward's persistent tiles: as many workgroups as fit at once.
template <int MODE, int CT>
static hipError_t launch_cube_bwd(const CubeArgs& A, int Hi, int Wi, int ntx, int total_tiles,
                                  hipStream_t stream) {
  static int per_cu = 0;
  if (per_cu == 0) {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_cube_bwd<MODE, CT>, 256, 0) !=
            hipSuccess ||
        b <= 0)
      b = 2;
    per_cu = b;
  }
  const int64_t resident = (int64_t)device_cu_count() * per_cu;
  const unsigned grid = (unsigned)(total_tiles < resident ? total_tiles : resident);
  hipLaunchKernelGGL((k_cube_bwd<MODE, CT>), dim3(grid), dim3(256), 0, stream, A, Hi, Wi, ntx,
                     total_tiles);
  return hipGetLastError();
}

// Where the backward keeps the mip pyramid's gradient: the library's
// per-stream scratch (grown with hipMalloc as needed), or a fixed buffer of
// `cap` floats (dr_texture_bwd_noalloc).
struct DPyrBuf {
  float* fixed;
  int64_t cap;
};

static int dpyr_get(const DPyrBuf& buf, int64_t np, hipStream_t stream, float*& d_pyr) {
  if (buf.fixed) {
    DR_CHECK_ARG(np <= buf.cap, "texture_bwd_noalloc: the mip pyramid gradient needs " +
                                    std::to_string(np) + " floats, above the fixed " +
                                    std::to_string(buf.cap) + " (use dr_texture_bwd)");
    d_pyr = buf.fixed;
    return DR_OK;
  }
  Scratch* sc = scratch_for(stream);
  if (!sc) return scratch_fail();
  d_pyr = (float*)scratch_get(sc, stream, SLOT_DPYR, (size_t)np * sizeof(float));
  return d_pyr ? DR_OK : scratch_fail();
}

// The cube extension's backward: k_cube_bwd (a tile's d_tex and d_pyramid sums
// in an LDS table), then the pyramid collapse over the Nt*6 faces.  The first
// `zero_tex` floats of d_tex are cleared first (0: accumulate), after the
// pyramid gradient's buffer is known to fit, so a refused call leaves d_tex
// untouched.
static int cube_bwd(const float* tex, const float* pyramid, const MipDesc& md, int64_t tex_stride,
                    int Nt, int Ht, int Wt, int C, const float* dir, const float* dir_da,
                    const float* bias_map, float bias, int filter, int N, int Hi, int Wi,
                    const float* d_out, float* d_tex, int64_t zero_tex, float* d_dir,
                    float* d_dir_da, float* d_bias_map, unsigned flags, const DPyrBuf& pbuf,
                    hipStream_t stream) {
  const bool mip = filter >= DR_FILTER_LINEAR_MIPMAP_NEAREST;
  float* d_pyr = nullptr;
  if (mip && md.L > 1) {
    const int64_t np = dr_texture_mip_size(Nt * 6, Ht, Wt, C, md.L);
    const int st = dpyr_get(pbuf, np, stream, d_pyr);
    if (st) return st;
    if (zero_tex) DR_CHECK_HIP(fill2_async(d_tex, zero_tex, d_pyr, np, 0.0f, stream));
    else DR_CHECK_HIP(fill_async(d_pyr, 0.0f, np, stream));
  } else if (zero_tex) {
    DR_CHECK_HIP(fill_async(d_tex, 0.0f, zero_tex, stream));
  }
  const int64_t P = (int64_t)N * Hi * Wi;
  CubeArgs A = cube_args(tex, pyramid, md, tex_stride, Ht, Wt, C, dir, dir_da, bias_map,
                         exp2f(bias), bias != 0.0f, P, Hi * Wi);
  A.d_out = d_out;
  A.d_tex = d_tex;
  A.d_pyr = d_pyr;
  A.d_dir = d_dir;
  A.dir_grad = (flags & DR_CUBE_DIR_GRAD) ? 1 : 0;
  A.d_dir_da = mip ? d_dir_da : nullptr;
  A.d_bias = mip ? d_bias_map : nullptr;
  const int ntx = (Wi + 15) / 16;
  const int64_t total_tiles = (int64_t)N * ntx * ((Hi + 15) / 16);
  DR_CHECK_ARG(total_tiles < ((int64_t)1 << 31), "texture_bwd: too many pixels");
  {
    DR_TIMED("k_cube_bwd", stream);
    hipError_t e = hipSuccess;
#define DR_CB(MODEV, CTV) e = launch_cube_bwd<MODEV, CTV>(A, Hi, Wi, ntx, (int)total_tiles, stream)
#define DR_CB_C(MODEV)                 \
  switch (C) {                         \
    case 1: DR_CB(MODEV, 1); break;    \
    case 2: DR_CB(MODEV, 2); break;    \
    case 3: DR_CB(MODEV, 3); break;    \
    case 4: DR_CB(MODEV, 4); break;    \
    default: DR_CB(MODEV, 0); break;   \
  }
    if (filter == DR_FILTER_LINEAR_MIPMAP_LINEAR) DR_CB_C(2)
    else if (filter == DR_FILTER_LINEAR_MIPMAP_NEAREST) DR_CB_C(1)
    else DR_CB_C(0)
#undef DR_CB_C
#undef DR_CB
    DR_CHECK_HIP(e);
  }
  DR_CHECK_LAUNCH();
  if (d_pyr) return mip_collapse(d_pyr, md, Nt * 6, Ht, Wt, C, d_tex, stream);
  return DR_OK;
}

static int texture_bwd(const float* tex, const float* pyramid, int Nt, int Ht, int Wt, int C,
                       int L, const float* uv, const float* uv_da, const float* bias_map,
                       float bias, int filter, int boundary, int N, int Hi, int Wi,
                       const float* d_out, float* d_tex, float* d_uv, float* d_uv_da,
                       float* d_bias_map, unsigned flags, const DPyrBuf& pbuf,
                       hipStream_t stream) {
  (void)hipGetLastError();
  MipDesc md;
  int st = check_tex(tex, pyramid, Nt, N, Ht, Wt, C, L, uv, uv_da, filter, boundary, md);
  if (st) return st;
  DR_CHECK_ARG(d_out && d_tex && Hi >= 1 && Wi >= 1, "texture_bwd: null tensor");
  const bool cube = boundary == DR_BOUNDARY_CUBE;
  const int64_t tex_stride = Nt == 1 ? 0 : (int64_t)(cube ? 6 : 1) * Ht * Wt * C;
  const int64_t ntex = (int64_t)Nt * (cube ? 6 : 1) * Ht * Wt * C;
  const bool zero_tex = !(flags & DR_ACCUMULATE);
  if (cube && (filter >= DR_FILTER_LINEAR_MIPMAP_NEAREST || (flags & DR_CUBE_DIR_GRAD))) {
    return cube_bwd(tex, pyramid, md, tex_stride, Nt, Ht, Wt, C, uv, uv_da, bias_map, bias,
                    filter, N, Hi, Wi, d_out, d_tex, zero_tex ? ntex : 0, d_uv, d_uv_da,
                    d_bias_map, flags, pbuf, stream);
  }
  const bool mip = !cube && filter >= DR_FILTER_LINEAR_MIPMAP_NEAREST;
  float* d_pyr = nullptr;
  if (mip && md.L > 1) {
    const int64_t np = dr_texture_mip_size(Nt, Ht, Wt, C, md.L);
    st = dpyr_get(pbuf, np, stream, d_pyr);
    if (st) return st;
    // d_tex and the coarser levels' accumulator are zeroed in one launch
    if (zero_tex) DR_CHECK_HIP(fill2_async(d_tex, ntex, d_pyr, np, 0.0f, stream));
    else DR_CHECK_HIP(fill_async(d_pyr, 0.0f, np, stream));
  } else if (zero_tex) {
    DR_CHECK_HIP(fill_async(d_tex, 0.0f, ntex, stream));
  }
  const int ntx = (Wi + 15) / 16, nty = (Hi + 15) / 16;
  TexBwdArgs args;
  args.tex = tex;
  args.pyr = pyramid;
  args.md = md;
  args.tex_stride = tex_stride;
  args.Ht = Ht;
  args.Wt = Wt;
  args.C = C;
  args.boundary = boundary;
  args.has_bias = bias != 0.0f;
  args.uv = uv;
  args.uv_da = uv_da;
  args.bias_map = bias_map;
  args.scale_bias = exp2f(bias);
  args.N = N;
  args.Hi = Hi;
  args.Wi = Wi;
  args.ntx = ntx;
  args.nty = nty;
  args.d_out = d_out;
  args.d_tex = d_tex;
  args.d_pyr = d_pyr;
  args.d_uv = d_uv;
  args.d_uv_da = mip ? d_uv_da : nullptr;
  args.d_bias = mip ? d_bias_map : nullptr;
  const int64_t total_tiles = (int64_t)N * ntx * nty;
  DR_CHECK_ARG(total_tiles < (int64_t)1 << 31, "texture_bwd: too many pixels");
  // Persistent tiles: each wave keeps its footprint accumulator across the
  // tiles it visits.
  {
    DR_TIMED("k_tex_bwd", stream);
    hipError_t e = hipSuccess;
#define DR_TB(F, CUBEV, CTV) e = launch_tex_bwd<F, CUBEV, CTV>(args, (int)total_tiles, stream)
#define DR_TB_C(F, CUBEV)                  \
  switch (C) {                             \
    case 1: DR_TB(F, CUBEV, 1); break;     \
    case 2: DR_TB(F, CUBEV, 2); break;     \
    case 3: DR_TB(F, CUBEV, 3); break;     \
    case 4: DR_TB(F, CUBEV, 4); break;     \
    default: DR_TB(F, CUBEV, 0); break;    \
  }
    // the windowed kernel's tiles are 16 x (4 * kWinWaves) pixels
    TexBwdArgs wargs = args;
    wargs.nty = (Hi + 4 * kWinWaves - 1) / (4 * kWinWaves);
    const int wtiles = (int)((int64_t)N * ntx * wargs.nty);
#define DR_TW(F)                                                   \
  switch (C) {                                                     \
    case 1: e = launch_tex_bwd_win<F, 1>(wargs, wtiles, stream); break; \
    case 2: e = launch_tex_bwd_win<F, 2>(wargs, wtiles, stream); break; \
    case 3: e = launch_tex_bwd_win<F, 3>(wargs, wtiles, stream); break; \
    default: e = launch_tex_bwd_win<F, 4>(wargs, wtiles, stream); break; \
  }
    const bool windowed = C <= 4 && Wt <= 32767 && Ht <= 32767;  // window boxes use 16-bit texel coordinates
    // more channels: while the empty pixels' sums have room, texel
    // coordinates fit 16 bits and a level's floats 32
    const bool many = C > 4 && C <= kManyC && Wt <= 32767 && Ht <= 32767 &&
                      (uint64_t)Ht * Wt * C < (1ull << 32);
    if (many && cube)
      e = launch_tex_bwd_many<DR_FILTER_LINEAR, DR_BOUNDARY_CUBE>(args, (int)total_tiles, stream);
    else if (many && filter == DR_FILTER_NEAREST)
      e = launch_tex_bwd_many_b<DR_FILTER_NEAREST>(args, (int)total_tiles, stream);
    else if (many && filter == DR_FILTER_LINEAR)
      e = launch_tex_bwd_many_b<DR_FILTER_LINEAR>(args, (int)total_tiles, stream);
    else if (many && filter == DR_FILTER_LINEAR_MIPMAP_NEAREST)
      e = launch_tex_bwd_many_b<DR_FILTER_LINEAR_MIPMAP_NEAREST>(args, (int)total_tiles, stream);
    else if (many)
      e = launch_tex_bwd_many_b<DR_FILTER_LINEAR_MIPMAP_LINEAR>(args, (int)total_tiles, stream);
    else if (windowed && cube)
      switch (C) {
        case 1: e = launch_tex_bwd_win_bb<DR_FILTER_LINEAR, 1, DR_BOUNDARY_CUBE, false>(wargs, wtiles, stream); break;
        case 2: e = launch_tex_bwd_win_bb<DR_FILTER_LINEAR, 2, DR_BOUNDARY_CUBE, false>(wargs, wtiles, stream); break;
        case 3: e = launch_tex_bwd_win_bb<DR_FILTER_LINEAR, 3, DR_BOUNDARY_CUBE, false>(wargs, wtiles, stream); break;
        default: e = launch_tex_bwd_win_bb<DR_FILTER_LINEAR, 4, DR_BOUNDARY_CUBE, false>(wargs, wtiles, stream); break;
      }
    else if (windowed && filter == DR_FILTER_NEAREST) DR_TW(DR_FILTER_NEAREST)
    else if (windowed && filter == DR_FILTER_LINEAR) DR_TW(DR_FILTER_LINEAR)
    else if (windowed && filter == DR_FILTER_LINEAR_MIPMAP_NEAREST) DR_TW(DR_FILTER_LINEAR_MIPMAP_NEAREST)
    else if (windowed) DR_TW(DR_FILTER_LINEAR_MIPMAP_LINEAR)
    else if (cube) DR_TB_C(DR_FILTER_LINEAR, true)
    else if (filter == DR_FILTER_NEAREST) DR_TB_C(DR_FILTER_NEAREST, false)
    else if (filter == DR_FILTER_LINEAR) DR_TB_C(DR_FILTER_LINEAR, false)
    else if (filter == DR_FILTER_LINEAR_MIPMAP_NEAREST) DR_TB_C(DR_FILTER_LINEAR_MIPMAP_NEAREST, false)
    else DR_TB_C(DR_FILTER_LINEAR_MIPMAP_LINEAR, false)
#undef DR_TW
#undef DR_TB_C
#undef DR_TB
    DR_CHECK_HIP(e);
  }
  if (d_pyr) return mip_collapse(d_pyr, md, Nt, Ht, Wt, C, d_tex, stream);
  return DR_OK;
}

extern "C" int dr_texture_bwd(const float* tex, const float* pyramid, int Nt, int Ht, int Wt,
                              int C, int L, const float* uv, const float* uv_da,
                              const float* bias_map, float bias, int filter, int boundary, int N,
                              int Hi, int Wi, const float* d_out, float* d_tex, float* d_uv,
                              float* d_uv_da, float* d_bias_map, unsigned flags,
                              dr_stream_t stream_) {
  return texture_bwd(tex, pyramid, Nt, Ht, Wt, C, L, uv, uv_da, bias_map, bias, filter, boundary,
                     N, Hi, Wi, d_out, d_tex, d_uv, d_uv_da, d_bias_map, flags,
                     DPyrBuf{nullptr, 0}, (hipStream_t)stream_);
}

// ---- dr_texture_bwd without allocation --------------------------------------
// The pyramid gradient lives in one fixed device array instead of the
// library's per-stream scratch.  In host code `scratch` names a host-side
// stand-in: its device address on each GPU comes from hipGetSymbolAddress
// (with that GPU current), kept per device, and only that address is used.

static __device__ __align__(256) float scratch[DR_TEXTURE_BWD_NOALLOC_FLOATS];

static std::mutex g_noalloc_mu;
static float* g_noalloc_ptr[64] = {};

static int noalloc_scratch(float*& ptr) {
  int dev = 0;
  DR_CHECK_HIP(hipGetDevice(&dev));
  DR_CHECK_ARG(dev >= 0 && dev < 64, "texture_bwd_noalloc: device index above 63");
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* p = nullptr;
    DR_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    DR_CHECK_ARG(p != nullptr, "texture_bwd_noalloc: no device address for the scratch array");
    g_noalloc_ptr[dev] = (float*)p;
  }
  ptr = g_noalloc_ptr[dev];
  return DR_OK;
}

extern "C" int dr_texture_bwd_noalloc(const float* tex, const float* pyramid, int Nt, int Ht,
                                      int Wt, int C, int L, const float* uv, const float* uv_da,
                                      const float* bias_map, float bias, int filter, int boundary,
                                      int N, int Hi, int Wi, const float* d_out, float* d_tex,
                                      float* d_uv, float* d_uv_da, float* d_bias_map,
                                      unsigned flags, dr_stream_t stream_) {
  float* ptr = nullptr;
  const int st = noalloc_scratch(ptr);
  if (st) return st;
  return texture_bwd(tex, pyramid, Nt, Ht, Wt, C, L, uv, uv_da, bias_map, bias, filter, boundary,
                     N, Hi, Wi, d_out, d_tex, d_uv, d_uv_da, d_bias_map, flags,
                     DPyrBuf{ptr, (int64_t)DR_TEXTURE_BWD_NOALLOC_FLOATS}, (hipStream_t)stream_);
}
