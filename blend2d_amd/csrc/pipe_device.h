// Device fetchers and composition operators.
//
// Fetch: solid, linear/radial/conic gradient LUT lookup, affine pattern with
// nearest or bilinear filtering, translated pattern at an integer or
// fractional offset (pipeline/reference/fetchgeneric_p.h).  The
// reference steps each fetcher per pixel and per row; all of them are pure
// functions of the pixel position except the conic gradient, whose per-row
// origin accumulates in double precision from the first row of the fill call
// (fetchgeneric_p.h:1172-1173, 1227-1230).  That accumulation is reproduced.
//
// Composite: SRC_COPY / SRC_OVER / PLUS (pipeline/reference/compopgeneric_p.h)
// and MULTIPLY / SCREEN (pipeline/jit/compoppart.cpp:4291-4460, 4592-4628)
// with Blend2D's 8-bit div255 rounding (pixelgeneric_p.h:386-389).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_types.h"

namespace b2amd {
namespace pipe {

__device__ __forceinline__ uint32_t div255(uint32_t x) {
  uint32_t u = x + 0x80u;
  return ((u + ((u >> 8) & 0xFFu)) >> 8) & 0xFFu;
}

// div255 of two 16-bit lanes at once (bits 0-15 and 16-31, each <= 255 * 255):
// every intermediate of a lane stays below 65536, so no carry crosses lanes.
__device__ __forceinline__ uint32_t div255x2(uint32_t x) {
  const uint32_t u = x + 0x00800080u;
  return ((u + ((u >> 8) & 0x00FF00FFu)) >> 8) & 0x00FF00FFu;
}

// x86 cvttss2si / cvtss2si: out-of-range and NaN produce INT32_MIN.
__device__ __forceinline__ int32_t trunc_f32_to_i32(float v) {
  if (!(v >= -2147483648.0f && v < 2147483648.0f)) return INT32_MIN;
  return (int32_t)v;
}
__device__ __forceinline__ int32_t rint_f32_to_i32(float v) {
  if (!(v >= -2147483648.0f && v < 2147483648.0f)) return INT32_MIN;
  return (int32_t)__builtin_rintf(v);
}

// bayer_matrix_16x16 (tables/tables_p.h:448-469): dither thresholds of
// pixel (x & 15, y & 15), row by row.
__constant__ uint8_t kBayer16[256] = {
    0, 191,  48, 239,  12, 203,  60, 251,   3, 194,  51, 242,  15, 206,  63, 254,
  127,  64, 175, 112, 139,  76, 187, 124, 130,  67, 178, 115, 142,  79, 190, 127,
   32, 223,  16, 207,  44, 235,  28, 219,  35, 226,  19, 210,  47, 238,  31, 222,
  159,  96, 143,  80, 171, 108, 155,  92, 162,  99, 146,  83, 174, 111, 158,  95,
    8, 199,  56, 247,   4, 195,  52, 243,  11, 202,  59, 250,   7, 198,  55, 246,
  135,  72, 183, 120, 131,  68, 179, 116, 138,  75, 186, 123, 134,  71, 182, 119,
   40, 231,  24, 215,  36, 227,  20, 211,  43, 234,  27, 218,  39, 230,  23, 214,
  167, 104, 151,  88, 163, 100, 147,  84, 170, 107, 154,  91, 166, 103, 150,  87,
    2, 193,  50, 241,  14, 205,  62, 253,   1, 192,  49, 240,  13, 204,  61, 252,
  129,  66, 177, 114, 141,  78, 189, 126, 128,  65, 176, 113, 140,  77, 188, 125,
   34, 225,  18, 209,  46, 237,  30, 221,  33, 224,  17, 208,  45, 236,  29, 220,
  161,  98, 145,  82, 173, 110, 157,  94, 160,  97, 144,  81, 172, 109, 156,  93,
   10, 201,  58, 249,   6, 197,  54, 245,   9, 200,  57, 248,   5, 196,  53, 244,
  137,  74, 185, 122, 133,  70, 181, 118, 136,  73, 184, 121, 132,  69, 180, 117,
   42, 233,  26, 217,  38, 229,  22, 213,  41, 232,  25, 216,  37, 228,  21, 212,
  169, 106, 153,  90, 165, 102, 149,  86, 168, 105, 152,  89, 164, 101, 148,  85};

__device__ __forceinline__ uint64_t pa_norm(int32_t tw, int32_t rx, int32_t ox, uint64_t v) {
  uint32_t x = (uint32_t)((int32_t)(v >> 32) % tw);
  if ((int32_t)x < 0) x += (uint32_t)rx;
  if ((int32_t)x > ox) x -= (uint32_t)rx;
  return ((uint64_t)x << 32) | (v & 0xFFFFFFFFull);
}

__device__ __forceinline__ int32_t pa_index(int32_t v, int32_t mn, int32_t mx, int32_t cor) {
  if (v < mn) v = mn;
  if (v > mx) v = cor;
  return v ^ (v >> 31);
}

// N pixels per lane, one command for the whole wave.  What a command and its
// style hold is uniform, so it is read through the constant address space
// (scalar loads into SGPRs) and its branches are scalar; pixels are kept as two
// pairs of 16-bit lanes (blue and red, green and alpha) for the packed 16-bit
// instructions.

#define B2AMD_CONST __attribute__((address_space(4)))
template<typename T> using CPtr = const B2AMD_CONST T*;
template<typename T> __device__ __forceinline__ CPtr<T> cptr(const T* p) { return (CPtr<T>)(uintptr_t)p; }

// Memory reached through an address that was stored as an integer: tells the
// compiler that it is global memory (flat accesses also occupy the LDS path).
#define B2AMD_GLOBAL __attribute__((address_space(1)))
using GBytes = const B2AMD_GLOBAL uint8_t*;
__device__ __forceinline__ GBytes global_bytes(uint64_t address) { return (GBytes)address; }

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 as_pair(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ uint32_t as_u32(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ u16x2 both(uint32_t v) { const uint16_t h = (uint16_t)v; return u16x2{h, h}; }

// Byte k of v in both lanes (k a constant).
__device__ __forceinline__ u16x2 byte_pair(uint32_t v, int k) {
  return as_pair(__builtin_amdgcn_perm(0u, v, 0x0C000C00u | (uint32_t)k * 0x00010001u));
}

struct Px { u16x2 rb, ag; };
__device__ __forceinline__ Px px_of(uint32_t v) { return Px{as_pair(v & 0x00FF00FFu), as_pair((v >> 8) & 0x00FF00FFu)}; }
__device__ __forceinline__ uint32_t px_bits(Px p) { return as_u32(p.rb) | (as_u32(p.ag) << 8); }

// div255 of each lane: bits 8..15 of u + (u >> 8) with u = x + 128.  Lanes
// that wrap past 65535 keep exactly the bits that the 32-bit form masks out
// with & 0xFF, so the two agree for every product.
__device__ __forceinline__ u16x2 div255p(u16x2 x) {
  const u16x2 u = x + (uint16_t)0x80;
  return (u + (u >> (uint16_t)8)) >> (uint16_t)8;
}

// Source pixels under masks m (the same in both lanes), onto destination
// pixels d.  m == 0 leaves a
// pixel as it is under every operator.  `carry`: the source may hold a colour
// above its alpha (an image with any contents); SRC_OVER's final sum then
// carries from one byte into the next, as the reference's addition of the
// whole 32-bit pixel does.
template<int N>
__device__ __forceinline__ void composite32_n(uint32_t op, Px d[N], const Px s[N], const u16x2 m[N], bool carry) {
  switch (op) {
    case kOpSrcCopy:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = m[k], im = (uint16_t)0xFF - mm;
        d[k].rb = div255p(d[k].rb * im + s[k].rb * mm);
        d[k].ag = div255p(d[k].ag * im + s[k].ag * mm);
      }
      break;
    case kOpSrcOver:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = m[k];
        const u16x2 srb = div255p(s[k].rb * mm), sag = div255p(s[k].ag * mm);
        const u16x2 ia = (uint16_t)0xFF - sag.yy;
        d[k].rb = srb + div255p(d[k].rb * ia);
        d[k].ag = sag + div255p(d[k].ag * ia);
      }
      if (carry) {
#pragma unroll
        for (int k = 0; k < N; k++) d[k] = px_of(as_u32(d[k].rb) + (as_u32(d[k].ag) << 8));
      }
      break;
    case kOpPlus:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = m[k], top = both(255u);
        d[k].rb = __builtin_elementwise_min(d[k].rb + div255p(s[k].rb * mm), top);
        d[k].ag = __builtin_elementwise_min(d[k].ag + div255p(s[k].ag * mm), top);
      }
      break;
    case kOpMultiply:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = m[k];
        const u16x2 srb = div255p(s[k].rb * mm), sag = div255p(s[k].ag * mm);
        const u16x2 ia = (uint16_t)0xFF - sag.yy, ida = (uint16_t)0xFF - d[k].ag.yy;
        d[k].rb = div255p(d[k].rb * (srb + ia) + srb * ida);
        d[k].ag = div255p(d[k].ag * (sag + ia) + sag * ida);
      }
      break;
    case kOpScreen:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = m[k];
        const u16x2 srb = div255p(s[k].rb * mm), sag = div255p(s[k].ag * mm);
        d[k].rb = div255p(d[k].rb * ((uint16_t)0xFF - srb)) + srb;
        d[k].ag = div255p(d[k].ag * ((uint16_t)0xFF - sag)) + sag;
      }
      break;
    default:
      break;
  }
}

// SRC_OVER under full masks: the source needs no scaling.
template<int N>
__device__ __forceinline__ void src_over_full(Px d[N], const Px s[N], bool carry) {
#pragma unroll
  for (int k = 0; k < N; k++) {
    const u16x2 ia = (uint16_t)0xFF - s[k].ag.yy;
    d[k].rb = s[k].rb + div255p(d[k].rb * ia);
    d[k].ag = s[k].ag + div255p(d[k].ag * ia);
  }
  if (carry) {
#pragma unroll
    for (int k = 0; k < N; k++) d[k] = px_of(as_u32(d[k].rb) + (as_u32(d[k].ag) << 8));
  }
}

// A solid colour under one mask over the whole wave: everything that depends
// on the source alone is formed once in scalar registers, per pixel only the
// destination terms remain.  SRC_OVER and SRC_COPY.
template<int N>
__device__ __forceinline__ void composite32_flat(uint32_t op, Px d[N], uint32_t color, uint32_t m) {
  if (m == 255u && (op == kOpSrcCopy || (color >> 24) == 255u)) {   // the colour itself
#pragma unroll
    for (int k = 0; k < N; k++) d[k] = px_of(color);
    return;
  }
  const uint32_t s_rb = (color & 0x00FF00FFu) * m, s_ag = ((color >> 8) & 0x00FF00FFu) * m;
  if (op == kOpSrcOver) {
    const uint32_t s1_rb = div255x2(s_rb), s1_ag = div255x2(s_ag);
    const u16x2 ia = both((s1_ag >> 16) ^ 0xFFu);
#pragma unroll
    for (int k = 0; k < N; k++) {
      d[k].rb = as_pair(s1_rb) + div255p(d[k].rb * ia);
      d[k].ag = as_pair(s1_ag) + div255p(d[k].ag * ia);
    }
  }
  else {
    const u16x2 im = both(m ^ 0xFFu);
#pragma unroll
    for (int k = 0; k < N; k++) {
      d[k].rb = div255p(d[k].rb * im + as_pair(s_rb));
      d[k].ag = div255p(d[k].ag * im + as_pair(s_ag));
    }
  }
}

// The same on pairs of neighbouring A8 pixels; sa: source alpha.
template<int P>
__device__ __forceinline__ void composite8_n(uint32_t op, u16x2 d[P], const u16x2 sa[P], const u16x2 m[P]) {
  switch (op) {
    case kOpSrcCopy:
#pragma unroll
      for (int k = 0; k < P; k++) d[k] = div255p(d[k] * ((uint16_t)0xFF - m[k]) + sa[k] * m[k]);
      break;
    case kOpSrcOver:
#pragma unroll
      for (int k = 0; k < P; k++) {
        const u16x2 s1 = div255p(sa[k] * m[k]);
        d[k] = s1 + div255p(d[k] * ((uint16_t)0xFF - s1));
      }
      break;
    case kOpPlus:
#pragma unroll
      for (int k = 0; k < P; k++) d[k] = __builtin_elementwise_min(d[k] + div255p(sa[k] * m[k]), both(255u));
      break;
    default:
      break;
  }
}

// v mod d for 0 <= v < 2^22, 1 <= d (inv = 1 / d to one part in 2^22): the
// float quotient is off by at most one.
__device__ __forceinline__ uint32_t mod_small(uint32_t v, uint32_t d, float inv) {
  int32_t r = (int32_t)(v - (uint32_t)((float)v * inv) * d);
  r = r < 0 ? r + (int32_t)d : r;
  return (uint32_t)(r >= (int32_t)d ? r - (int32_t)d : r);
}

// Translated pattern: texel row / column of pattern coordinate p + t.  Pad
// clamps; repeat and reflect keep t in [0, period) and p is a pixel position,
// so their sum lies in [0, 2^18).
__device__ __forceinline__ uint32_t sp_wrap(int32_t p, int32_t t, int32_t period, int32_t size, float inv) {
  if (period == 0) {
    const int32_t v = __builtin_elementwise_add_sat(p, t);
    return (uint32_t)(v < 0 ? 0 : v > size - 1 ? size - 1 : v);
  }
  const uint32_t v = mod_small((uint32_t)(p + t), (uint32_t)period, inv);
  return v >= (uint32_t)size ? (uint32_t)period - 1u - v : v;
}

// Affine pattern, one axis: the pattern coordinates of N consecutive pixels
// from `v` (32.32) on, `step` apart, each normalized as pa_norm does.  The
// normalized coordinate is the only one congruent to it in (ox - r, ox], so
// the first is reduced with a float quotient and each next one by at most one
// period (with a period the step lies in [0, period); pad has none and keeps
// the coordinate).  That needs coordinates and a step below 2^22 in magnitude;
// a wave with a lane further out takes the division.
template<int N>
__device__ __forceinline__ void pa_walk(uint64_t v, uint64_t step, int32_t tw, int32_t r, int32_t ox, uint64_t out[N]) {
  constexpr int32_t kNear = 1 << 22;
  const int32_t hi = (int32_t)(v >> 32), last = (int32_t)((v + (uint64_t)(N - 1) * step) >> 32);
  const int32_t st = (int32_t)(step >> 32);
  const bool near_ok = hi > -kNear && hi < kNear && last > -kNear && last < kNear && st > -kNear && st < kNear;
  if (__ballot(!near_ok) == 0ull) {
    if (r == 0) {
#pragma unroll
      for (int k = 0; k < N; k++) out[k] = v + (uint64_t)k * step;
      return;
    }
    const float inv = __builtin_amdgcn_rcpf((float)tw);
    const int32_t q = (int32_t)__builtin_floorf((float)hi * inv);
    int32_t x = hi - q * tw;              // in [-tw, 2 tw)
    x = x > ox ? x - r : x;
    x = x > ox ? x - r : x;
    x = x <= ox - r ? x + r : x;
    uint64_t p = ((uint64_t)(uint32_t)x << 32) | (uint32_t)v;
    out[0] = p;
#pragma unroll
    for (int k = 1; k < N; k++) {
      p += step;
      int32_t h = (int32_t)(p >> 32);
      h = h > ox ? h - r : h;
      p = ((uint64_t)(uint32_t)h << 32) | (uint32_t)p;
      out[k] = p;
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < N; k++) out[k] = pa_norm(tw, r, ox, v + (uint64_t)k * step);
}

// N consecutive words at a 4-byte aligned address.
template<int N>
__device__ __forceinline__ void wide_load(const B2AMD_GLOBAL uint32_t* p, uint32_t out[N]) {
  if constexpr (N == 1) {
    out[0] = *p;
  }
  else {
    typedef uint32_t words __attribute__((ext_vector_type(N), aligned(4)));
    const words v = *(const B2AMD_GLOBAL words*)p;
#pragma unroll
    for (int k = 0; k < N; k++) out[k] = v[k];
  }
}

__device__ __forceinline__ uint32_t texel_at(GBytes row, uint32_t fmt, uint32_t x) {
  if (fmt == kFmtA8) return (uint32_t)row[x] * 0x01010101u;
  const uint32_t v = ((const B2AMD_GLOBAL uint32_t*)row)[x];
  return fmt == kFmtXRGB32 ? v | 0xFF000000u : v;
}

// Bilinear blend of four texels, rows first (8-bit weights): each 16-bit lane
// stays below 65536.
__device__ __forceinline__ uint32_t blend4(uint32_t t00, uint32_t t01, uint32_t t10, uint32_t t11, uint32_t wx, uint32_t wy) {
  const Px a = px_of(t00), b = px_of(t01), c = px_of(t10), e = px_of(t11);
  const u16x2 y1 = both(wy), y0 = both(256u - wy), x1 = both(wx), x0 = both(256u - wx);
  const uint16_t sh = 8;
  const u16x2 rb = (((a.rb * y0 + b.rb * y1) >> sh) * x0 + ((c.rb * y0 + e.rb * y1) >> sh) * x1) >> sh;
  const u16x2 ag = (((a.ag * y0 + b.ag * y1) >> sh) * x0 + ((c.ag * y0 + e.ag * y1) >> sh) * x1) >> sh;
  return px_bits(Px{rb, ag});
}

// Translated pattern: the texels of pixels px .. px + N - 1 from a row.
// Neighbours by one wide load (4-byte aligned); lanes whose pixels meet an edge
// of the image take them one by one.  Steps between texels are at most one up,
// so the ends being N - 1 apart means that all lie in a line.
template<int N>
__device__ __forceinline__ void aligned_texels(GBytes row, uint32_t fmt, int px, int32_t tx, int32_t rx, int32_t w, float inv_x,
                                               uint32_t out[N]) {
  const uint32_t x0 = sp_wrap(px, tx, rx, w, inv_x), xl = sp_wrap(px + N - 1, tx, rx, w, inv_x);
  if (N > 1 && fmt != kFmtA8 && xl == x0 + (uint32_t)(N - 1)) {
    wide_load<N>((const B2AMD_GLOBAL uint32_t*)row + x0, out);
    if (fmt == kFmtXRGB32) {
#pragma unroll
      for (int k = 0; k < N; k++) out[k] |= 0xFF000000u;
    }
    return;
  }
  out[0] = texel_at(row, fmt, x0);
#pragma unroll
  for (int k = 1; k < N; k++) out[k] = texel_at(row, fmt, k == N - 1 ? xl : sp_wrap(px + k, tx, rx, w, inv_x));
}

// The texels of pixels px .. px + N from two rows, the same way.
template<int N>
__device__ __forceinline__ void neighbour_texels(GBytes row0, GBytes row1, uint32_t fmt, int px, int32_t tx, int32_t rx,
                                                 int32_t w, float inv_x, uint32_t a[N + 1], uint32_t b[N + 1]) {
  const uint32_t x0 = sp_wrap(px, tx, rx, w, inv_x), xn = sp_wrap(px + N, tx, rx, w, inv_x);
  if (fmt == kFmtPRGB32 && xn == x0 + (uint32_t)N) {
    const B2AMD_GLOBAL uint32_t* const pa = (const B2AMD_GLOBAL uint32_t*)row0 + x0;
    const B2AMD_GLOBAL uint32_t* const pb = (const B2AMD_GLOBAL uint32_t*)row1 + x0;
    wide_load<N>(pa, a);
    wide_load<N>(pb, b);
    a[N] = pa[N];
    b[N] = pb[N];
    return;
  }
#pragma unroll
  for (int k = 0; k <= N; k++) {
    const uint32_t x = k == 0 ? x0 : k == N ? xn : sp_wrap(px + k, tx, rx, w, inv_x);
    a[k] = texel_at(row0, fmt, x);
    b[k] = texel_at(row1, fmt, x);
  }
}

// fetchgeneric_p.h:601-687: four texels under weights that sum to at most 256.
__device__ __forceinline__ uint32_t weigh4(uint32_t t00, uint32_t t10, uint32_t t01, uint32_t t11, u16x2 wa, u16x2 wb, u16x2 wc,
                                           u16x2 wd) {
  const Px a = px_of(t00), b = px_of(t10), c = px_of(t01), e = px_of(t11);
  const u16x2 rb = a.rb * wa + c.rb * wc + b.rb * wb + e.rb * wd;
  const u16x2 ag = a.ag * wa + c.ag * wc + b.ag * wb + e.ag * wd;
  return px_bits(Px{rb >> (uint16_t)8, ag >> (uint16_t)8});
}

// Styles that fetch_rows takes: translated patterns of 32-bit pixels.
__device__ __forceinline__ bool fetches_rows(uint32_t kind, uint32_t fmt) {
  return kind == kFetchPatternAligned ? fmt != kFmtA8 : kind == kFetchPatternFxFy && fmt == kFmtPRGB32;
}

// fetch_n of four pixels in each of R rows from y on (uniform): all rows' loads
// are in flight together, and with a fractional offset each texel row is read
// once.
template<int R>
__device__ __forceinline__ void fetch_rows(CPtr<DevStyle> s, uint32_t kind, int y, int px, const DevImage* images, uint32_t fmt,
                                           uint32_t out[R][4]) {
  const CPtr<DevImage> im = cptr(images + s->img);
  const GBytes base = global_bytes(im->ptr);
  const int64_t stride = im->stride;
  const int32_t w = s->sp_w, h = s->sp_h, rx = s->sp_rx, ry = s->sp_ry, tx = s->sp_tx, ty = s->sp_ty;
  const float inv_y = ry ? __builtin_amdgcn_rcpf((float)ry) : 0.0f, inv_x = rx ? __builtin_amdgcn_rcpf((float)rx) : 0.0f;
  const uint32_t x0 = sp_wrap(px, tx, rx, w, inv_x);
  if (kind == kFetchPatternAligned) {
    const bool line = sp_wrap(px + 3, tx, rx, w, inv_x) == x0 + 3u;
    if (line) {
#pragma unroll
      for (int r = 0; r < R; r++)
        wide_load<4>((const B2AMD_GLOBAL uint32_t*)(base + (int64_t)sp_wrap(y + r, ty, ry, h, inv_y) * stride) + x0, out[r]);
    }
    else {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t x = sp_wrap(px + k, tx, rx, w, inv_x);
#pragma unroll
        for (int r = 0; r < R; r++)
          out[r][k] = ((const B2AMD_GLOBAL uint32_t*)(base + (int64_t)sp_wrap(y + r, ty, ry, h, inv_y) * stride))[x];
      }
    }
    if (fmt == kFmtXRGB32) {
#pragma unroll
      for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < 4; k++) out[r][k] |= 0xFF000000u;
    }
    return;
  }
  uint32_t t[R + 1][5];
  const bool line = sp_wrap(px + 4, tx, rx, w, inv_x) == x0 + 4u;
  if (line) {
#pragma unroll
    for (int r = 0; r <= R; r++) {
      const B2AMD_GLOBAL uint32_t* const row =
        (const B2AMD_GLOBAL uint32_t*)(base + (int64_t)sp_wrap(y + r, ty, ry, h, inv_y) * stride) + x0;
      wide_load<4>(row, t[r]);
      t[r][4] = row[4];
    }
  }
  else {
#pragma unroll
    for (int k = 0; k <= 4; k++) {
      const uint32_t x = sp_wrap(px + k, tx, rx, w, inv_x);
#pragma unroll
      for (int r = 0; r <= R; r++)
        t[r][k] = ((const B2AMD_GLOBAL uint32_t*)(base + (int64_t)sp_wrap(y + r, ty, ry, h, inv_y) * stride))[x];
    }
  }
  const u16x2 wa = both(s->sp_wa), wb = both(s->sp_wb), wc = both(s->sp_wc), wd = both(s->sp_wd);
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int k = 0; k < 4; k++) out[r][k] = weigh4(t[r][k], t[r][k + 1], t[r + 1][k], t[r + 1][k + 1], wa, wb, wc, wd);
}

// The source pixels px .. px + N - 1 of row y (per lane) of a non-solid style
// (uniform).  Every address read lies inside the gradient table or the image
// for any pixel position, so pixels that end up with no coverage may be
// fetched too.
template<int N, bool kDither>
__device__ __forceinline__ void fetch_n(CPtr<DevStyle> s, uint32_t kind, int y, int px, int fill_row0, uint32_t ref_band_h,
                                        const uint32_t* __restrict__ luts, const DevImage* images, uint32_t fmt,
                                        uint32_t out[N]) {
  if (kind <= kFetchConic) {
    uint32_t idx[N];
    const uint32_t extend = s->extend, maxi = s->maxi, rori = s->rori;
    auto index = [&](uint32_t i) {
      if (extend == 0) {
        const int32_t v = (int32_t)i;
        return (uint32_t)(v < 0 ? 0 : v > (int32_t)maxi ? (int32_t)maxi : v);
      }
      const uint32_t a = i & maxi, b = a ^ rori;
      return b < a ? b : a;
    };
    if (kind == kFetchLinear) {
      const uint64_t dt = s->lin_dt;
      uint64_t pt = s->lin_pt0 + (uint64_t)(uint32_t)y * s->lin_dy + (uint64_t)(uint32_t)px * dt;
#pragma unroll
      for (int k = 0; k < N; k++) {
        idx[k] = index((uint32_t)(pt >> 32));
        pt += dt;
      }
    }
    else if (kind == kFetchRadial) {
      const double yd = (double)y;
      const double ptx = s->rad_yx * yd + s->rad_tx;
      const double pty = s->rad_yy * yd + s->rad_ty;
      const double b = yd * s->rad_by + s->rad_b0;
      const double sq_dist = ptx * ptx + pty * pty;
      const double sq_inv2a = s->rad_sq_inv2a;
      const float f0 = (float)(b * s->rad_inv2a);
      const float f1 = (float)((s->rad_amul4 * (sq_dist - s->rad_sq_fr) + b * b) * sq_inv2a);
      const float f2 = (float)((yd * s->rad_ddy + s->rad_dd0) * sq_inv2a);
      const float bd = s->rad_bd, ddd = s->rad_ddd;
#pragma unroll
      for (int k = 0; k < N; k++) {
        const float fx = (float)(px + k);
        const float a = __builtin_sqrtf(__builtin_fabsf((fx * fx) * ddd + (fx * f2 + f1)));
        idx[k] = index((uint32_t)trunc_f32_to_i32((fx * bd + f0) + a));
      }
    }
    else {
      // First row of the reference fill call that covers `y`: analytic fills
      // run per band (first band starts at the path's first row), box fills
      // start at the box's first row.
      int ys = fill_row0;
      if (ref_band_h) {
        const int band_start = y & ~(int)(ref_band_h - 1u);   // a power of two
        if (band_start > ys) ys = band_start;
      }
      const double yx = s->con_yx, yy = s->con_yy;
      double tpx = s->con_tx + yx * (double)ys;
      double tpy = s->con_ty + yy * (double)ys;
      for (int k = ys; k < y; k++) { tpx += yx; tpy += yy; }
      const float ayf = (float)tpy;
      const float f0 = (float)tpx;
      const float f2 = __builtin_signbit(ayf) ? s->con_n1 : 0.0f;
      const float ay = __builtin_fabsf(ayf);
      const float q0 = s->con_q[0], q1 = s->con_q[1], q2 = s->con_q[2], q3 = s->con_q[3];
      const float n2 = s->con_n2, n4 = s->con_n4, off = s->con_offset, xx = s->con_xx;
      const int32_t cmax = s->con_maxi;
      const uint32_t cror = (uint32_t)s->con_rori;
#pragma unroll
      for (int k = 0; k < N; k++) {
        const float xv = (float)(px + k) * xx + f0;
        const float ax = __builtin_fabsf(xv);
        const float xy_min = ay < ax ? ay : ax;
        const float xy_max = ax < ay ? ay : ax;
        const float sv = (ax == xy_min) ? n4 : 0.0f;
        const float p = xy_min / xy_max;
        const float p_sq = p * p;
        float v = p_sq * q3 + q2;
        v = v * p_sq + q1;
        v = v * p_sq + q0;
        v = __builtin_fabsf(v * p - sv);
        v = __builtin_fabsf(v - (__builtin_signbit(xv) ? n2 : 0.0f));
        v = __builtin_fabsf(v - f2) + off;
        const int32_t i = rint_f32_to_i32(v);
        idx[k] = (uint32_t)(i > cmax ? cmax : i) & cror;
      }
    }
    const uint32_t* __restrict__ table = luts + s->lut;
    if (kDither && s->dither) {
#pragma unroll
      for (int k = 0; k < N; k++) {
        uint2 e;
        __builtin_memcpy(&e, table + 2u * idx[k], 8);   // 4-byte aligned
        const uint32_t dd = kBayer16[(((uint32_t)y & 15u) << 4) | ((uint32_t)(px + k) & 15u)];
        const uint32_t a = e.y >> 24;
        uint32_t r = ((e.y & 0xFFFFu) + dd) >> 8;
        uint32_t g = ((e.x >> 16) + dd) >> 8;
        uint32_t b = ((e.x & 0xFFFFu) + dd) >> 8;
        r = r < a ? r : a;
        g = g < a ? g : a;
        b = b < a ? b : a;
        out[k] = (a << 24) | (r << 16) | (g << 8) | b;
      }
      return;
    }
#pragma unroll
    for (int k = 0; k < N; k++) out[k] = table[idx[k]];
    return;
  }

  const CPtr<DevImage> im = cptr(images + s->img);
  const GBytes base = global_bytes(im->ptr);
  const int64_t stride = im->stride;
  if (kind == kFetchPatternAligned || kind == kFetchPatternFxFy) {
    const int32_t w = s->sp_w, h = s->sp_h, rx = s->sp_rx, ry = s->sp_ry, tx = s->sp_tx, ty = s->sp_ty;
    const float inv_y = ry ? __builtin_amdgcn_rcpf((float)ry) : 0.0f, inv_x = rx ? __builtin_amdgcn_rcpf((float)rx) : 0.0f;
    const GBytes row0 = base + (int64_t)sp_wrap(y, ty, ry, h, inv_y) * stride;
    if (kind == kFetchPatternAligned) {
      aligned_texels<N>(row0, fmt, px, tx, rx, w, inv_x, out);
      return;
    }
    // columns x + tx and the next of rows y + ty and the next, weighted wa
    // (x0 y0), wb (x1 y0), wc (x0 y1), wd (x1 y1)
    const GBytes row1 = base + (int64_t)sp_wrap(y + 1, ty, ry, h, inv_y) * stride;
    uint32_t a[N + 1], b[N + 1];
    neighbour_texels<N>(row0, row1, fmt, px, tx, rx, w, inv_x, a, b);
    const u16x2 wa = both(s->sp_wa), wb = both(s->sp_wb), wc = both(s->sp_wc), wd = both(s->sp_wd);
#pragma unroll
    for (int k = 0; k < N; k++) out[k] = weigh4(a[k], a[k + 1], b[k], b[k + 1], wa, wb, wc, wd);
    return;
  }

  // affine
  uint64_t ux[N], uy[N];
  pa_walk<N>(s->pa_tx + s->pa_yx * (uint64_t)(uint32_t)y + s->pa_xx * (uint64_t)(uint32_t)px, s->pa_xx, s->pa_tw, s->pa_rx,
             s->pa_ox, ux);
  pa_walk<N>(s->pa_ty + s->pa_yy * (uint64_t)(uint32_t)y + s->pa_xy * (uint64_t)(uint32_t)px, s->pa_xy, s->pa_th, s->pa_ry,
             s->pa_oy, uy);
  const int32_t minx = s->pa_minx, miny = s->pa_miny, maxx = s->pa_maxx, maxy = s->pa_maxy;
  const int32_t corx = s->pa_corx, cory = s->pa_cory;
  if (kind == kFetchPatternNN) {
#pragma unroll
    for (int k = 0; k < N; k++)
      out[k] = texel_at(base + (int64_t)pa_index((int32_t)(uy[k] >> 32), miny, maxy, cory) * stride, fmt,
                        (uint32_t)pa_index((int32_t)(ux[k] >> 32), minx, maxx, corx));
    return;
  }
  uint32_t t00[N], t01[N], t10[N], t11[N];
  uint32_t x0[N], x1[N];
  bool apart = fmt == kFmtA8 || im->w < 2u;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int32_t ix = (int32_t)(ux[k] >> 32);
    x0[k] = (uint32_t)pa_index(ix, minx, maxx, corx);
    x1[k] = (uint32_t)pa_index(ix + 1, minx, maxx, corx);
    apart |= x0[k] - x1[k] + 1u > 2u;
  }
  if (__ballot(apart) == 0ull) {
    // the two texels of a row are neighbours or the same one: an 8-byte load
    // holds both (half the loads; the pair at the row's end starts a texel
    // before it)
    const uint32_t last = im->w - 2u;
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int32_t iy = (int32_t)(uy[k] >> 32);
      const uint32_t xl = min(min(x0[k], x1[k]), last);
      uint32_t a[2], b[2];
      wide_load<2>((const B2AMD_GLOBAL uint32_t*)(base + (int64_t)pa_index(iy, miny, maxy, cory) * stride) + xl, a);
      wide_load<2>((const B2AMD_GLOBAL uint32_t*)(base + (int64_t)pa_index(iy + 1, miny, maxy, cory) * stride) + xl, b);
      t00[k] = x0[k] == xl ? a[0] : a[1];
      t10[k] = x1[k] == xl ? a[0] : a[1];
      t01[k] = x0[k] == xl ? b[0] : b[1];
      t11[k] = x1[k] == xl ? b[0] : b[1];
    }
    if (fmt == kFmtXRGB32) {
#pragma unroll
      for (int k = 0; k < N; k++) {
        t00[k] |= 0xFF000000u;
        t01[k] |= 0xFF000000u;
        t10[k] |= 0xFF000000u;
        t11[k] |= 0xFF000000u;
      }
    }
  }
  else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int32_t iy = (int32_t)(uy[k] >> 32);
      const GBytes r0 = base + (int64_t)pa_index(iy, miny, maxy, cory) * stride;
      const GBytes r1 = base + (int64_t)pa_index(iy + 1, miny, maxy, cory) * stride;
      t00[k] = texel_at(r0, fmt, x0[k]);
      t01[k] = texel_at(r1, fmt, x0[k]);
      t10[k] = texel_at(r0, fmt, x1[k]);
      t11[k] = texel_at(r1, fmt, x1[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < N; k++) out[k] = blend4(t00[k], t01[k], t10[k], t11[k], (uint32_t)ux[k] >> 24, (uint32_t)uy[k] >> 24);
}

}  // namespace pipe
}  // namespace b2amd
