// Checks the device edge builder (blend2d_amd/csrc/edge_device.h, compiled
// here for the host) on curves that leave the canvas, up to control points of
// 1e308: every piece taken on the way that place_piece gives it (flattened by
// CurveWalk, one segment, nothing, or the general builder) must end, and give
// the segments that the general builder gives for it; pieces that the general
// builder gives up on must fail both ways.
//
//   edges_check <curves> <seed> <seconds>      exit status 0 when all agree
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <unistd.h>

#include <algorithm>
#include <array>
#include <random>
#include <vector>

#include "../../blend2d_amd/csrc/edge_device.h"

using namespace b2amd;
using namespace b2amd::edge;

namespace {

using Seg = std::array<int32_t, 5>;   // x0, y0, x1, y1, sign

// `walk`: takes the parts inside the box that the builder gives away, as the
// lanes of k_edges_clip do; else it gives none away.
struct Sink {
  bool walk = false;
  double tol_sq = 0.0;
  std::vector<Seg> segs;
  void push(int32_t x0, int32_t y0, int32_t x1, int32_t y1, uint32_t sign) { segs.push_back(Seg{x0, y0, x1, y1, (int32_t)sign}); }
  bool give(const P* p, int n, uint32_t sign);
};
using B = Builder<Sink>;

const long kMaxSteps = 1 << 20;
long steps_over = 0;

void walk_piece(Sink& out, const P p[4], int n, uint32_t sign) {
  CurveWalk<B> w;
  w.start(p, n, sign);
  bool halved = false;
  long steps = 0;
  while (w.step(out.tol_sq, halved, [&](int32_t x0, int32_t y0, int32_t x1, int32_t y1, uint32_t s) { out.push(x0, y0, x1, y1, s); }))
    if (++steps > kMaxSteps) { steps_over++; break; }
}

bool Sink::give(const P* p, int n, uint32_t sign) {
  if (!walk) return false;
  const P q[4] = {p[0], p[1], p[n == 3 ? 2 : 2], p[n - 1]};
  walk_piece(*this, q, n, sign);
  return true;
}

// The pieces of a curve, in order; false: none (its border line, or nothing).
int cut(const P cv[4], int n, P out[8][4]) {
  double ts[8];
  const int cuts = n == 3 ? B::cuts_quad(cv, ts) : B::cuts_cubic(cv, ts);
  if (cuts == 0) {
    for (int i = 0; i < 4; i++) out[0][i] = cv[std::min(i, n - 1)];
    return 1;
  }
  P at = cv[0];
  double t_cut = 0.0;
  int pieces = 0;
  for (int i = 0; i < cuts; i++) {
    if (n == 4 && ts[i] == t_cut) continue;
    P* p = out[pieces++];
    if (n == 3) { B::piece_quad(cv, t_cut, ts[i], i + 1 == cuts, at, p); p[3] = p[2]; }
    else B::piece_cubic(cv, t_cut, ts[i], i + 1 == cuts, at, p);
    at = p[3];
    t_cut = ts[i];
  }
  return pieces;
}

uint32_t build(Sink& out, const Clip& clip, const P p[4], int n) {
  P stack[B::kLimit * 4];
  B b(out, clip, out.tol_sq);
  b.curve_piece(p, n, stack);
  return b.invalid;
}

}  // namespace

int main(int argc, char** argv) {
  const long count = argc > 1 ? atol(argv[1]) : 20000;
  std::mt19937_64 rng(argc > 2 ? strtoull(argv[2], nullptr, 10) : 1);
  alarm(argc > 3 ? atoi(argv[3]) : 60);   // a walk that doesn't end is a failure
  auto uni = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
  const int sizes[5] = {17, 300, 400, 4000, 65535};
  long bad = 0, pieces = 0, odd = 0, failed = 0, ways[4] = {0, 0, 0, 0};
  for (long i = 0; i < count; i++) {
    const int w = sizes[rng() % 5], h = sizes[rng() % 5], n = 3 + (int)(rng() & 1);
    Clip clip;
    clip.x0 = clip.y0 = 0.0;
    clip.x1 = w * 256.0; clip.y1 = h * 256.0;
    clip.ix0 = 0; clip.ix1 = w * 256;
    const bool far = rng() % 4 != 0;
    const double mag = pow(10.0, uni(rng() & 1 ? 300 : 2, 308));
    P cv[4];
    if (i == 0) {   // its first piece starts inside the canvas and ends nowhere
      clip.x1 = 400 * 256.0; clip.y1 = 300 * 256.0; clip.ix1 = 400 * 256;
      cv[0] = P{25600, 25600}; cv[1] = P{4.7e305 * 256, 20 * 256}; cv[2] = cv[3] = P{51200, 30720};
    }
    else
      for (int k = 0; k < 4; k++)
        for (int a = 0; a < 2; a++) {
          const double side = (a ? h : w) * 256.0;
          double& v = a ? cv[k].y : cv[k].x;
          switch (rng() % 4) {
            case 0: v = uni(0, side); break;
            case 1: v = std::array<double, 6>{0.0, side, side + 1, -1.0, side / 2, 1.0}[rng() % 6]; break;
            case 2: v = uni(-side, 2 * side); break;
            default: v = far ? (rng() & 1 ? -mag : mag) * uni(0.1, 5) : uni(-20 * side, 20 * side); break;
          }
        }
    const int points = i == 0 ? 3 : n;
    bool finite = true;
    uint32_t common = 15;
    for (int k = 0; k < points; k++) {
      finite &= isfinite(cv[k].x) && isfinite(cv[k].y);
      common &= fxy(clip, cv[k]);
    }
    if (!finite || common) continue;
    P piece[8][4];
    const int np = cut(cv, points, piece);
    for (int k = 0; k < np; k++) {
      const P* p = piece[k];
      for (int q = 0; q < 4; q++) odd += !(isfinite(p[q].x) && isfinite(p[q].y));
      pieces++;
      Sink want, got;
      want.tol_sq = got.tol_sq = 51.2 * 51.2;
      got.walk = true;
      const uint32_t want_fail = build(want, clip, p, points);
      // as k_edges takes it
      const uint32_t sign = p[0].y > p[3].y ? 1u : 0u;
      const P a = sign ? p[3] : p[0], z = sign ? p[0] : p[3];
      DevSeg line;
      const PieceWay way = place_piece(clip, p, a, z, line);
      uint32_t got_fail = 0;
      ways[way]++;
      if (way == kPieceLine) got.push(line.x0, line.y0, line.x1, line.y1, sign);
      else if (way == kPieceClip) got_fail = build(got, clip, p, points);
      else if (way == kPieceInside) {
        const P c1 = points == 3 ? p[1] : sign ? p[2] : p[1], c2 = points == 3 ? z : sign ? p[1] : p[2];
        const double xl = dmin(a.x, z.x), xr = dmax(a.x, z.x);
        const P top[4] = {a, P{dclamp(c1.x, xl, xr), dclamp(c1.y, a.y, z.y)},
                          points == 3 ? z : P{dclamp(c2.x, xl, xr), dclamp(c2.y, a.y, z.y)}, z};
        walk_piece(got, top, points, sign);
      }
      failed += want_fail != 0;
      if (want_fail || got_fail) {
        if (want_fail == got_fail) continue;
        bad++;
      }
      std::sort(want.segs.begin(), want.segs.end());
      std::sort(got.segs.begin(), got.segs.end());
      if (want.segs != got.segs) {
        if (bad++ < 5)
          fprintf(stderr, "%d points on %d x %d, way %d: (%g,%g) (%g,%g) (%g,%g) (%g,%g): %zu segments for %zu\n", points, w, h, (int)way,
                  p[0].x, p[0].y, p[1].x, p[1].y, p[2].x, p[2].y, p[3].x, p[3].y, got.segs.size(), want.segs.size());
      }
    }
  }
  printf("pieces %ld not finite %ld failed %ld ways %ld %ld %ld %ld endless %ld mismatches %ld\n", pieces, odd, failed, ways[0],
         ways[1], ways[2], ways[3], steps_over, bad + steps_over);
  return bad || steps_over ? 1 : 0;
}
