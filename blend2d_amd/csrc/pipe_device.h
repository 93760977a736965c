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

__device__ __forceinline__ uint32_t ch(uint32_t p, int i) { return (p >> (i * 8)) & 0xFFu; }

// div255 of two 16-bit lanes at once (bits 0-15 and 16-31, each <= 255 * 255):
// every intermediate of a lane stays below 65536, so no carry crosses lanes.
__device__ __forceinline__ uint32_t div255x2(uint32_t x) {
  const uint32_t u = x + 0x00800080u;
  return ((u + ((u >> 8) & 0x00FF00FFu)) >> 8) & 0x00FF00FFu;
}

// Per-lane min(v, 255) of two lanes holding values <= 510.
__device__ __forceinline__ uint32_t sat255x2(uint32_t v) {
  const uint32_t o = v & 0x01000100u;
  return (v | (o - (o >> 8))) & 0x00FF00FFu;
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

// Translated pattern, texel row of pattern row v (fetchgeneric_p.h:80-165):
// pad clamps to [0, h-1]; repeat wraps by h; reflect wraps by 2h and mirrors
// the second half.
__device__ __forceinline__ uint32_t sp_row(const DevStyle& s, int64_t v) {
  const int64_t h = (int64_t)s.sp_h;
  if (s.sp_ry == 0) return (uint32_t)(v < 0 ? 0 : v > h - 1 ? h - 1 : v);
  int64_t r = v % s.sp_ry;
  if (r < 0) r += s.sp_ry;
  if (r >= h) r = s.sp_ry - 1 - r;
  return (uint32_t)r;
}

// Translated pattern, texel column of pattern column u
// (fetchgeneric_p.h:187-352): pad clamps; a period rx (repeat: w, reflect:
// 2w) wraps, and a wrapped position v >= w maps to rx - 1 - v.  For repeat
// and reflect the offset is kept in [0, rx), so u >= 0 there.
__device__ __forceinline__ uint32_t sp_col(const DevStyle& s, int64_t u) {
  const int64_t w = (int64_t)s.sp_w;
  if (s.sp_rx == 0) return (uint32_t)(u < 0 ? 0 : u > w - 1 ? w - 1 : u);
  uint32_t v = (uint32_t)u % (uint32_t)s.sp_rx;
  if (v >= (uint32_t)w) v = (uint32_t)s.sp_rx - 1u - v;
  return v;
}

// Per (command, row) fetch state.
struct Row {
  uint64_t a, b;       // linear: pt at x = 0; pattern: tx, ty of the row;
                       // gradients: the row in b (dither thresholds)
  float f0, f1, f2;    // radial: b, d, dd;  conic: tx, ay, by
};

__device__ __forceinline__ Row row_setup(const DevStyle& s, int y, int fill_row0, uint32_t ref_band_h) {
  Row r;
  r.a = 0; r.b = (uint32_t)y; r.f0 = 0.f; r.f1 = 0.f; r.f2 = 0.f;
  switch (s.kind) {
    case kFetchLinear:
      r.a = s.lin_pt0 + (uint64_t)(uint32_t)y * s.lin_dy;
      break;
    case kFetchRadial: {
      double yd = (double)y;
      double ptx = s.rad_yx * yd + s.rad_tx;
      double pty = s.rad_yy * yd + s.rad_ty;
      double b = yd * s.rad_by + s.rad_b0;
      double sq_dist = ptx * ptx + pty * pty;
      r.f0 = (float)(b * s.rad_inv2a);
      r.f1 = (float)((s.rad_amul4 * (sq_dist - s.rad_sq_fr) + b * b) * s.rad_sq_inv2a);
      r.f2 = (float)((yd * s.rad_ddy + s.rad_dd0) * s.rad_sq_inv2a);
      break;
    }
    case kFetchConic: {
      // First row of the reference fill call that covers `y`: analytic fills
      // run per band (first band starts at the path's first row), box fills
      // start at the box's first row.
      int ys = fill_row0;
      if (ref_band_h) {
        int band_start = (y / (int)ref_band_h) * (int)ref_band_h;
        if (band_start > ys) ys = band_start;
      }
      double tpx = s.con_tx + s.con_yx * (double)ys;
      double tpy = s.con_ty + s.con_yy * (double)ys;
      for (int k = ys; k < y; k++) { tpx += s.con_yx; tpy += s.con_yy; }
      float ay = (float)tpy;
      r.f0 = (float)tpx;
      r.f2 = __builtin_signbit(ay) ? s.con_n1 : 0.0f;
      r.f1 = __builtin_fabsf(ay);
      break;
    }
    case kFetchPatternNN:
    case kFetchPatternBI:
      r.a = s.pa_tx + s.pa_yx * (uint64_t)(uint32_t)y;
      r.b = s.pa_ty + s.pa_yy * (uint64_t)(uint32_t)y;
      break;
    case kFetchPatternAligned:
    case kFetchPatternFxFy:
      // texel rows of this row and of the next one (FxFy)
      r.a = sp_row(s, (int64_t)y + s.sp_ty);
      r.b = sp_row(s, (int64_t)y + 1 + s.sp_ty);
      break;
    default:
      break;
  }
  return r;
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

// Gradient table entry `i` at pixel (x, row y): the 32-bit entry, or for a
// dithered gradient the 64-bit one with the pixel's Bayer threshold added to
// each colour channel before it is cut to 8 bits, limited by alpha
// (FetchGradientBase<DITHER>::fetch_pixel, fetchgeneric_p.h:899-934).
// kDither = false (frames without dithered gradients) leaves the dither path
// out of the code, and its registers out of the render kernels.
template<bool kDither>
__device__ __forceinline__ uint32_t lut_px(const DevStyle& s, const uint32_t* __restrict__ luts, uint32_t i, int x,
                                           uint32_t y) {
  if (!kDither || !s.dither) return luts[s.lut + i];
  const uint32_t lo = luts[s.lut + 2u * i], hi = luts[s.lut + 2u * i + 1u];
  const uint32_t dd = kBayer16[((y & 15u) << 4) | ((uint32_t)x & 15u)];
  const uint32_t a = hi >> 24;
  uint32_t r = ((hi & 0xFFFFu) + dd) >> 8;
  uint32_t g = ((lo >> 16) + dd) >> 8;
  uint32_t b = ((lo & 0xFFFFu) + dd) >> 8;
  r = r < a ? r : a;
  g = g < a ? g : a;
  b = b < a ? b : a;
  return (a << 24) | (r << 16) | (g << 8) | b;
}

__device__ __forceinline__ uint32_t grad_index(uint32_t idx, const DevStyle& s) {
  if (s.extend == 0) {
    int32_t i = (int32_t)idx;
    if (i < 0) i = 0;
    if (i > (int32_t)s.maxi) i = (int32_t)s.maxi;
    return (uint32_t)i;
  }
  uint32_t a = idx & s.maxi, b = a ^ s.rori;
  return b < a ? b : a;
}

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

__device__ __forceinline__ uint32_t texel(const DevImage& im, uint32_t fmt, int32_t x, int32_t y) {
  const uint8_t* row = (const uint8_t*)im.ptr + (int64_t)y * im.stride;
  if (fmt == kFmtA8) return (uint32_t)row[x] * 0x01010101u;
  uint32_t v = ((const uint32_t*)row)[x];
  if (fmt == kFmtXRGB32) v |= 0xFF000000u;
  return v;
}

template<bool kDither = false>
__device__ __forceinline__ uint32_t fetch(const DevStyle& s, const Row& r, int x, const uint32_t* __restrict__ luts,
                                          const DevImage* __restrict__ images, uint32_t src_fmt) {
  switch (s.kind) {
    case kFetchSolid:
      return s.solid;
    case kFetchLinear: {
      uint64_t pt = r.a + (uint64_t)(uint32_t)x * s.lin_dt;
      return lut_px<kDither>(s, luts, grad_index((uint32_t)(pt >> 32), s), x, (uint32_t)r.b);
    }
    case kFetchRadial: {
      float fx = (float)x;
      float sq_x = fx * fx;
      float a = __builtin_sqrtf(__builtin_fabsf(sq_x * s.rad_ddd + (fx * r.f2 + r.f1)));
      float v = (fx * s.rad_bd + r.f0) + a;
      return lut_px<kDither>(s, luts, grad_index((uint32_t)trunc_f32_to_i32(v), s), x, (uint32_t)r.b);
    }
    case kFetchConic: {
      float fx = (float)x;
      float xv = fx * s.con_xx + r.f0;
      float ax = __builtin_fabsf(xv);
      float ay = r.f1;
      float xy_min = ay < ax ? ay : ax;
      float xy_max = ax < ay ? ay : ax;
      float sv = (ax == xy_min) ? s.con_n4 : 0.0f;
      float p = xy_min / xy_max;
      float p_sq = p * p;
      float v = p_sq * s.con_q[3] + s.con_q[2];
      v = v * p_sq + s.con_q[1];
      v = v * p_sq + s.con_q[0];
      v = __builtin_fabsf(v * p - sv);
      v = __builtin_fabsf(v - (__builtin_signbit(xv) ? s.con_n2 : 0.0f));
      v = __builtin_fabsf(v - r.f2) + s.con_offset;
      int32_t i = rint_f32_to_i32(v);
      if (i > s.con_maxi) i = s.con_maxi;
      return lut_px<kDither>(s, luts, (uint32_t)i & (uint32_t)s.con_rori, x, (uint32_t)r.b);
    }
    case kFetchPatternNN:
    case kFetchPatternBI: {
      const DevImage& im = images[s.img];
      uint64_t px = pa_norm(s.pa_tw, s.pa_rx, s.pa_ox, r.a + s.pa_xx * (uint64_t)(uint32_t)x);
      uint64_t py = pa_norm(s.pa_th, s.pa_ry, s.pa_oy, r.b + s.pa_xy * (uint64_t)(uint32_t)x);
      int32_t ix = (int32_t)(px >> 32), iy = (int32_t)(py >> 32);
      if (s.kind == kFetchPatternNN)
        return texel(im, src_fmt, pa_index(ix, s.pa_minx, s.pa_maxx, s.pa_corx), pa_index(iy, s.pa_miny, s.pa_maxy, s.pa_cory));
      int32_t x0 = pa_index(ix, s.pa_minx, s.pa_maxx, s.pa_corx);
      int32_t y0 = pa_index(iy, s.pa_miny, s.pa_maxy, s.pa_cory);
      int32_t x1 = pa_index(ix + 1, s.pa_minx, s.pa_maxx, s.pa_corx);
      int32_t y1 = pa_index(iy + 1, s.pa_miny, s.pa_maxy, s.pa_cory);
      uint32_t wx = (uint32_t)(px & 0xFFFFFFFFull) >> 24;
      uint32_t wy = (uint32_t)(py & 0xFFFFFFFFull) >> 24;
      uint32_t iw = 256 - wx, ih = 256 - wy;
      uint32_t t00 = texel(im, src_fmt, x0, y0), t01 = texel(im, src_fmt, x0, y1);
      uint32_t t10 = texel(im, src_fmt, x1, y0), t11 = texel(im, src_fmt, x1, y1);
      uint32_t out = 0;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        uint32_t p0 = ((ch(t00, c) * ih + ch(t01, c) * wy) >> 8) & 0xFFu;
        uint32_t p1 = ((ch(t10, c) * ih + ch(t11, c) * wy) >> 8) & 0xFFu;
        out |= (((p0 * iw + p1 * wx) >> 8) & 0xFFu) << (c * 8);
      }
      return out;
    }
    case kFetchPatternAligned:
      return texel(images[s.img], src_fmt, (int32_t)sp_col(s, (int64_t)x + s.sp_tx), (int32_t)r.a);
    case kFetchPatternFxFy: {
      // fetchgeneric_p.h:601-687: columns x0 = x + tx and x1 = x0 + 1 of rows
      // y0, y1, weighted wa (x0 y0), wb (x1 y0), wc (x0 y1), wd (x1 y1).  The
      // weights sum to at most 256, so each 16-bit lane of the R/B and A/G
      // pairs stays below 65536.
      const DevImage& im = images[s.img];
      const int32_t x0 = (int32_t)sp_col(s, (int64_t)x + s.sp_tx), x1 = (int32_t)sp_col(s, (int64_t)x + 1 + s.sp_tx);
      const uint32_t t00 = texel(im, src_fmt, x0, (int32_t)r.a), t01 = texel(im, src_fmt, x0, (int32_t)r.b);
      const uint32_t t10 = texel(im, src_fmt, x1, (int32_t)r.a), t11 = texel(im, src_fmt, x1, (int32_t)r.b);
      const uint32_t m = 0x00FF00FFu;
      const uint32_t rb = (t00 & m) * s.sp_wa + (t01 & m) * s.sp_wc + (t10 & m) * s.sp_wb + (t11 & m) * s.sp_wd;
      const uint32_t ag = ((t00 >> 8) & m) * s.sp_wa + ((t01 >> 8) & m) * s.sp_wc +
                          ((t10 >> 8) & m) * s.sp_wb + ((t11 >> 8) & m) * s.sp_wd;
      return ((rb >> 8) & m) | (ag & ~m);
    }
    default:
      return 0;
  }
}

// One PRGB32 destination pixel.
__device__ __forceinline__ uint32_t composite32(uint32_t op, uint32_t d, uint32_t s, uint32_t m) {
  uint32_t r = 0;
  switch (op) {
    // SRC_COPY, SRC_OVER and PLUS work on the R/B and A/G channel pairs
    // (two 16-bit lanes per register); per channel the arithmetic is the
    // scalar div255 form.
    case kOpSrcCopy: {
      const uint32_t im = m ^ 0xFFu;
      const uint32_t rb = div255x2((d & 0x00FF00FFu) * im + (s & 0x00FF00FFu) * m);
      const uint32_t ag = div255x2(((d >> 8) & 0x00FF00FFu) * im + ((s >> 8) & 0x00FF00FFu) * m);
      return rb | (ag << 8);
    }
    case kOpSrcOver: {
      const uint32_t s1 = div255x2((s & 0x00FF00FFu) * m) | (div255x2(((s >> 8) & 0x00FF00FFu) * m) << 8);
      const uint32_t ia = (s1 >> 24) ^ 0xFFu;
      const uint32_t t = div255x2((d & 0x00FF00FFu) * ia) | (div255x2(((d >> 8) & 0x00FF00FFu) * ia) << 8);
      return s1 + t;
    }
    case kOpPlus: {
      const uint32_t rb = sat255x2((d & 0x00FF00FFu) + div255x2((s & 0x00FF00FFu) * m));
      const uint32_t ag = sat255x2(((d >> 8) & 0x00FF00FFu) + div255x2(((s >> 8) & 0x00FF00FFu) * m));
      return rb | (ag << 8);
    }
    case kOpMultiply: {
      uint32_t s1[4];
#pragma unroll
      for (int i = 0; i < 4; i++) s1[i] = div255(ch(s, i) * m);
      uint32_t da = ch(d, 3);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        uint32_t v = ch(d, i) * ((s1[i] + (s1[3] ^ 0xFFu)) & 0xFFFFu) + s1[i] * (da ^ 0xFFu);
        r |= div255(v & 0xFFFFu) << (i * 8);
      }
      return r;
    }
    case kOpScreen: {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        uint32_t s1 = div255(ch(s, i) * m);
        r |= ((div255(ch(d, i) * (s1 ^ 0xFFu)) + s1) & 0xFFu) << (i * 8);
      }
      return r;
    }
    default:
      return d;
  }
}

// One A8 destination pixel; `sa` is the source alpha.
__device__ __forceinline__ uint32_t composite8(uint32_t op, uint32_t d, uint32_t sa, uint32_t m) {
  switch (op) {
    case kOpSrcCopy: return div255(d * (m ^ 0xFFu) + sa * m);
    case kOpSrcOver: {
      uint32_t s1 = div255(sa * m);
      return (s1 + div255(d * (s1 ^ 0xFFu))) & 0xFFu;
    }
    case kOpPlus: {
      uint32_t v = d + div255(sa * m);
      return v > 255u ? 255u : v;
    }
    default:
      return d;
  }
}

// ---------------------------------------------------------------------------
// The render kernel's form of the same: N pixels per lane, one command for the
// whole wave.  What a command and its style hold is uniform, so it is read
// through the constant address space (scalar loads into SGPRs) and its
// branches are scalar; pixels are kept as two pairs of 16-bit lanes (blue and
// red, green and alpha) for the packed 16-bit instructions.
// ---------------------------------------------------------------------------

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

// Source pixels under masks m, onto destination pixels d: composite32 on
// pairs.  m == 0 leaves a pixel as it is under every operator.  `carry`: the
// source may hold a colour above its alpha (an image with any contents);
// SRC_OVER's final sum then carries from one byte into the next as the 32-bit
// addition of composite32 does.
template<int N>
__device__ __forceinline__ void composite32_n(uint32_t op, Px d[N], const Px s[N], const uint32_t m[N], bool carry) {
  switch (op) {
    case kOpSrcCopy:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = both(m[k]), im = (uint16_t)0xFF - mm;
        d[k].rb = div255p(d[k].rb * im + s[k].rb * mm);
        d[k].ag = div255p(d[k].ag * im + s[k].ag * mm);
      }
      break;
    case kOpSrcOver:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = both(m[k]);
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
        const u16x2 mm = both(m[k]), top = both(255u);
        d[k].rb = __builtin_elementwise_min(d[k].rb + div255p(s[k].rb * mm), top);
        d[k].ag = __builtin_elementwise_min(d[k].ag + div255p(s[k].ag * mm), top);
      }
      break;
    case kOpMultiply:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = both(m[k]);
        const u16x2 srb = div255p(s[k].rb * mm), sag = div255p(s[k].ag * mm);
        const u16x2 ia = (uint16_t)0xFF - sag.yy, ida = (uint16_t)0xFF - d[k].ag.yy;
        d[k].rb = div255p(d[k].rb * (srb + ia) + srb * ida);
        d[k].ag = div255p(d[k].ag * (sag + ia) + sag * ida);
      }
      break;
    case kOpScreen:
#pragma unroll
      for (int k = 0; k < N; k++) {
        const u16x2 mm = both(m[k]);
        const u16x2 srb = div255p(s[k].rb * mm), sag = div255p(s[k].ag * mm);
        d[k].rb = div255p(d[k].rb * ((uint16_t)0xFF - srb)) + srb;
        d[k].ag = div255p(d[k].ag * ((uint16_t)0xFF - sag)) + sag;
      }
      break;
    default:
      break;
  }
}

// A solid colour under one mask over the whole wave: everything that depends
// on the source alone is formed once in scalar registers, per pixel only the
// destination terms remain.  SRC_OVER and SRC_COPY.
template<int N>
__device__ __forceinline__ void composite32_flat(uint32_t op, Px d[N], uint32_t color, uint32_t m) {
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

// composite8 on pairs of neighbouring A8 pixels.
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
  typedef uint32_t words __attribute__((ext_vector_type(N == 1 ? 2 : N), aligned(4)));
  const words v = *(const B2AMD_GLOBAL words*)p;
#pragma unroll
  for (int k = 0; k < N; k++) out[k] = v[k];
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
      const uint32_t x0 = sp_wrap(px, tx, rx, w, inv_x), x3 = sp_wrap(px + N - 1, tx, rx, w, inv_x);
      if (fmt != kFmtA8 && N > 1) {
        // N neighbouring texels: one wide load (4-byte aligned)
        const bool run = x3 == x0 + (uint32_t)(N - 1);
        if (__ballot(!run) == 0ull) {
          wide_load<N>((const B2AMD_GLOBAL uint32_t*)row0 + x0, out);
          if (fmt == kFmtXRGB32) {
#pragma unroll
            for (int k = 0; k < N; k++) out[k] |= 0xFF000000u;
          }
          return;
        }
      }
      out[0] = texel_at(row0, fmt, x0);
#pragma unroll
      for (int k = 1; k < N; k++) out[k] = texel_at(row0, fmt, k == N - 1 ? x3 : sp_wrap(px + k, tx, rx, w, inv_x));
      return;
    }
    // fetchgeneric_p.h:601-687: columns x0 = x + tx and x1 = x0 + 1 of rows
    // y0, y1, weighted wa (x0 y0), wb (x1 y0), wc (x0 y1), wd (x1 y1), which
    // sum to at most 256
    const GBytes row1 = base + (int64_t)sp_wrap(y + 1, ty, ry, h, inv_y) * stride;
    uint32_t a[N + 1], b[N + 1];
#pragma unroll
    for (int k = 0; k <= N; k++) {
      const uint32_t x = sp_wrap(px + k, tx, rx, w, inv_x);
      a[k] = texel_at(row0, fmt, x);
      b[k] = texel_at(row1, fmt, x);
    }
    const u16x2 wa = both(s->sp_wa), wb = both(s->sp_wb), wc = both(s->sp_wc), wd = both(s->sp_wd);
#pragma unroll
    for (int k = 0; k < N; k++) {
      const Px t00 = px_of(a[k]), t01 = px_of(b[k]), t10 = px_of(a[k + 1]), t11 = px_of(b[k + 1]);
      const u16x2 rb = t00.rb * wa + t01.rb * wc + t10.rb * wb + t11.rb * wd;
      const u16x2 ag = t00.ag * wa + t01.ag * wc + t10.ag * wb + t11.ag * wd;
      out[k] = px_bits(Px{rb >> (uint16_t)8, ag >> (uint16_t)8});
    }
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
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int32_t ix = (int32_t)(ux[k] >> 32), iy = (int32_t)(uy[k] >> 32);
    const uint32_t x0 = (uint32_t)pa_index(ix, minx, maxx, corx), x1 = (uint32_t)pa_index(ix + 1, minx, maxx, corx);
    const GBytes r0 = base + (int64_t)pa_index(iy, miny, maxy, cory) * stride;
    const GBytes r1 = base + (int64_t)pa_index(iy + 1, miny, maxy, cory) * stride;
    t00[k] = texel_at(r0, fmt, x0);
    t01[k] = texel_at(r1, fmt, x0);
    t10[k] = texel_at(r0, fmt, x1);
    t11[k] = texel_at(r1, fmt, x1);
  }
#pragma unroll
  for (int k = 0; k < N; k++) out[k] = blend4(t00[k], t01[k], t10[k], t11[k], (uint32_t)ux[k] >> 24, (uint32_t)uy[k] >> 24);
}

}  // namespace pipe
}  // namespace b2amd
