// Coverage cells of one edge segment on one pixel row, in closed form.
//
// The reference rasterizes an edge by walking it scanline by scanline with
// two incremental divisions (raster/analyticrasterizer_p.h:289-1165): one
// steps x down the row boundaries, the other steps y across the column
// boundaries, each rounding its quotient to the nearest value.  A tile of
// the render kernel needs one row of one edge at a time, so this file
// evaluates those two sequences directly at any index instead of stepping
// to it:
//
//   x on the row boundary y = 256 k     X(k) = x0 +- floor(((256 k - y0) dx + ceil(dy / 2)) / dy)
//   y on the column boundary x = 256 m  Y(m) = y0 + floor((|256 m - x0| dy + ceil(dx / 2)) / dx)
//
// (both are the fixed points of the reference's lift / remainder / error
// accumulators, whose error term starts at floor(d / 2) - 1; the start and
// end rows use the edge's own end points).  Within a row the edge enters at
// X(r) and leaves at X(r + 1); every cell between gets the cover of the y
// interval between the column crossings around it and the area of its x
// extent.  How the crossing y is taken relative to the row differs with the
// slope, as in the reference: an edge at least as tall as wide (at most one
// crossing per row) keeps it modulo 256, a flatter one as is.
//
// Only prefix sums of a row's cells are ever used (the coverage of pixel x
// is the sum of cells 0..x), so a tile keeps the cells inside it and folds
// every cell left of it into one backdrop value, its cover << 9; the area a
// cell left of the tile carries into the first cell of the tile cancels out
// of every prefix sum inside the tile and is dropped on both sides.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define B2AMD_HD __host__ __device__ __forceinline__
#else
#define B2AMD_HD inline
#endif

namespace b2amd {
namespace ras {

// 1 / d to within two units in the last place, d > 0.
B2AMD_HD double recip(int32_t d) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double x = (double)d;
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
#else
  return 1.0 / (double)d;
#endif
}

// floor(n / d) for an integral n, 0 <= n < 2^49, and inv = recip(d).  The
// exact (n + 1/2) / d lies at least 1 / (2 d) away from every integer, and
// the computed product is off by less than 2^-50 of itself (two ulps of inv
// and one rounding): less than 1 / (2 d) while n < 2^49, so truncating it
// gives the floor.  The dividends here stay below 2^24 * 2^24 + 2^24.
B2AMD_HD int32_t div_floor(double n, double inv) { return (int32_t)((n + 0.5) * inv); }

// A line moving left is handled as its mirror image (x -> -x) moving right:
// the reference starts a cell right of a boundary point when moving right and
// left of it when moving left, and measures the area from the other side, so
// the two directions are exact mirror images.
struct Edge {
  int32_t x0, y0, x1, y1;  // 24.8, y0 < y1, x0 <= x1 (mirrored when `left`)
  int32_t dx, dy;          // x1 - x0, y1 - y0
  bool left;               // x shrinks downwards
  int32_t row0, row1;      // first and last pixel row it touches
  bool steep;              // dy >= dx: at most one column crossing per row
};

// Returns false for edges that add nothing (horizontal).  Coordinates lie
// within the canvas, at most 65535 pixels a side: the edge builder clips.
B2AMD_HD bool edge_init(Edge& e, int32_t x0, int32_t y0, int32_t x1, int32_t y1) {
  if (y0 >= y1) return false;
  e.left = x1 < x0;
  e.x0 = e.left ? -x0 : x0; e.y0 = y0;
  e.x1 = e.left ? -x1 : x1; e.y1 = y1;
  e.dx = e.x1 - e.x0;
  e.dy = y1 - y0;
  e.row0 = y0 >> 8;
  e.row1 = (y1 - 1) >> 8;
  e.steep = e.dy >= e.dx;
  return true;
}

// x where the edge crosses the row boundary y = 256 k, row0 < k <= row1;
// inv_dy = recip(e.dy).
B2AMD_HD int32_t x_at_row_boundary(const Edge& e, double inv_dy, int32_t k) {
  const uint32_t half = (uint32_t)(uint64_t)(e.dy - (e.dy >> 1));
  return e.x0 + div_floor(__builtin_fma((double)(256 * k - e.y0), (double)e.dx, (double)half), inv_dy);
}

// Product of two values below 2^23 in magnitude that fits 32 bits.
B2AMD_HD int32_t mul_small(int32_t a, int32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __mul24(a, b);
#else
  return a * b;
#endif
}

// v * sgn for sgn = +1 or -1.
B2AMD_HD int32_t with_sign(int32_t v, int32_t sgn) { return (v ^ (sgn >> 31)) - (sgn >> 31); }

// Row `r` (row0 <= r <= row1) of edge `e`, with cover sign `sgn` (+1 or -1),
// against a tile whose pixel columns are [x_left, x_left + width): calls
// sink(i, v) to add v to tile cell i (0 <= i < width) and returns the
// backdrop, the cover << 9 of the row's cells left of the tile.
template<typename Sink>
B2AMD_HD uint32_t emit_row(const Edge& e, int32_t r, int32_t x_left, int32_t width, int32_t sgn, Sink&& sink) {
  const int32_t row_y = 256 * r;
  const int32_t ytop = r == e.row0 ? e.y0 - row_y : 0;
  const int32_t ybot = r == e.row1 ? e.y1 - row_y : 256;
  // the tile's cells in the direction of travel: [w0, w1]
  const int32_t w0 = e.left ? -(x_left + width) : x_left, w1 = w0 + width - 1;

  const double inv_dy = recip(e.dy);
  const int32_t xt = x_at_row_boundary(e, inv_dy, r), xb = x_at_row_boundary(e, inv_dy, r + 1);
  const int32_t xe = r == e.row0 ? e.x0 : xt;
  const int32_t xx = r == e.row1 ? e.x1 : xb;

  // First and last cell, entry and exit offset in them.  A point on a
  // boundary starts the cell right of it and ends the cell left of it.
  const int32_t ce = xe >> 8, cx = (xx - 1) >> 8 > ce ? (xx - 1) >> 8 : ce;
  const int32_t fe = xe & 255, fx = xx - (cx << 8);
  if (cx < w0 || ce > w1) return (cx < w0) != e.left ? (uint32_t)with_sign(ybot - ytop, sgn) << 9 : 0u;
  const int32_t k0 = ce > w0 ? ce : w0, k1 = cx < w1 ? cx : w1;   // the cells inside the tile

  // Crossing y of a column boundary, row-relative.
  auto rel = [&](int32_t q) -> int32_t {
    const int32_t y = e.y0 + q;
    return e.steep ? (y & 255) : y - row_y;
  };
  // Dividend of the crossing of the boundary that cell k0 is left through;
  // each next boundary adds 256 dy.
  double inv_dx = 0.0, num = 0.0, step = 0.0;
  int32_t y_in = ytop;
  if (ce != cx) {
    inv_dx = recip(e.dx);
    step = 256.0 * (double)e.dy;
    num = __builtin_fma((double)(256 * (k0 + 1) - e.x0), (double)e.dy, (double)(e.dx - (e.dx >> 1)));
    // entered through the tile edge: the crossing one boundary earlier
    if (k0 != ce) y_in = rel(div_floor(num - step, inv_dx));
  }
  // Cells left of the tile telescope to the y interval they span: the first
  // ones moving right, the last ones moving left.
  uint32_t backdrop = 0;
  if (!e.left) backdrop = (uint32_t)with_sign(y_in - ytop, sgn) << 9;
  // A cell adds cover * 512 - area to itself and area to the cell on its
  // right, the area measured from its left side; in the direction of travel
  // that is one value per boundary: what the cell before it passes on plus
  // what this cell adds on that side.
  int32_t carry = 0;
  for (int32_t k = k0; k <= k1; k++) {
    const bool last = k == cx;
    const int32_t y_out = last ? ybot : rel(div_floor(num, inv_dx));
    const int32_t cover = with_sign(y_out - y_in, sgn);
    const int32_t area = mul_small(cover, (k == ce ? fe : 0) + (last ? fx : 256));
    const int32_t cell = (e.left ? -k : k) - x_left;
    if ((uint32_t)cell < (uint32_t)width) sink(cell, (uint32_t)(carry + cover * 512 - area));
    carry = area;
    y_in = y_out;
    num += step;
  }
  const int32_t cell = (e.left ? -(k1 + 1) : k1 + 1) - x_left;
  if ((uint32_t)cell < (uint32_t)width) sink(cell, (uint32_t)carry);
  if (e.left && cx > w1) backdrop = (uint32_t)with_sign(ybot - y_in, sgn) << 9;
  return backdrop;
}

}  // namespace ras
}  // namespace b2amd
