// walks.hpp -- which pixels the intervening-contour walks cross
// (intervening.cu:44-475), as constants.
//
// The reference walks Bresenham lines from a pixel to every point of the
// boundary of its 11 x 11 window (clipped to the image) and records, for the
// disc points a walk is the best integer approximant of, the affinity of the
// strongest boundary crossed so far; later walks replace earlier ones.
// Which pixels are crossed on the way to a disc point depends only on how
// far the window reaches to the four sides, so the compiler follows the walks
// once per reach.
#pragma once
#include <cstdint>
#include <utility>

namespace dmsc {

constexpr int kWalkArea = 81;   // points of the radius-5 disc, raster order
constexpr int kMaxCross = 13;   // distinct pixels crossed on the way to one

constexpr int walk_half_width(int dy) {
  return dy == 0 ? 5 : (dy >= -3 && dy <= 3) ? 4 : (dy == 4 || dy == -4) ? 3 : 0;
}
constexpr int walk_point(int dy, int dx) {  // raster index of a disc point
  int at = 0;
  for (int y = -5; y < dy; y++) at += 2 * walk_half_width(y) + 1;
  return at + dx + walk_half_width(dy);
}
constexpr int walk_dy(int d) {
  int dy = -5;
  while (d >= 2 * walk_half_width(dy) + 1) d -= 2 * walk_half_width(dy++) + 1;
  return dy;
}
constexpr int walk_dx(int d) {
  int dy = -5;
  while (d >= 2 * walk_half_width(dy) + 1) d -= 2 * walk_half_width(dy++) + 1;
  return d - walk_half_width(dy);
}

struct Walks {
  signed char n[kWalkArea] = {};  // pixels crossed; -1: no walk speaks for the point
  signed char ex[kWalkArea][kMaxCross] = {};
  signed char ey[kWalkArea][kMaxCross] = {};
};

// intervening.cu:44-283: the walk from (0, 0) to (x2, y2) between its
// neighbours (x1, y1) and (x3, y3) on the window's boundary.
constexpr void walk_line(Walks& W, int x1, int y1, int x2, int y2, int x3, int y3) {
  const int dot11 = x1 * x1 + y1 * y1, dot22 = x2 * x2 + y2 * y2, dot33 = x3 * x3 + y3 * y3;
  const int adx = x2 < 0 ? -x2 : x2, ady = y2 < 0 ? -y2 : y2;
  bool xmajor = false;
  if (x2 > 0 && y2 >= 0) xmajor = adx > ady;
  else if (x2 <= 0 && y2 > 0) xmajor = adx >= ady;
  else if (y2 <= 0 && x2 < 0) xmajor = adx > ady;
  else xmajor = adx >= ady;
  const int sx = x2 > 0 ? 1 : -1, sy = y2 > 0 ? 1 : -1;  // a step of a zero component is never taken
  int t = xmajor ? -adx : -ady, xi = 0, yi = 0, n = 0;
  signed char ex[kMaxCross + 4] = {}, ey[kMaxCross + 4] = {};
  auto cross = [&](int x, int y) {
    for (int k = 0; k < n; k++)
      if (ex[k] == x && ey[k] == y) return;
    ex[n] = (signed char)x;
    ey[n] = (signed char)y;
    n++;
  };
  while (xi != x2 || yi != y2) {
    const int ox = xi, oy = yi;
    if (xmajor) {
      xi += sx;
      t += 2 * ady;
      if (t > 0) { yi += sy; t -= 2 * adx; }
    } else {
      yi += sy;
      t += 2 * adx;
      if (t > 0) { xi += sx; t -= 2 * ady; }
    }
    const int hy = (yi > oy ? yi : oy) - 1, vx = (xi > ox ? xi : ox) - 1;
    if (ox == xi) {
      cross(xi, hy);
    } else if (oy == yi) {
      cross(vx, yi);
    } else {  // a diagonal step crosses two horizontal and two vertical edges
      cross(ox, hy);
      cross(xi, hy);
      cross(vx, oy);
      cross(vx, yi);
    }
    const int dotii = xi * xi + yi * yi, d1 = xi * x1 + yi * y1, d2 = xi * x2 + yi * y2, d3 = xi * x3 + yi * y3;
    const bool good = d2 * d2 == dotii * dot22 || (dot11 * d2 * d2 > dot22 * d1 * d1 && dot33 * d2 * d2 >= dot22 * d3 * d3);
    if (!good || dotii > 25) continue;
    const int d = walk_point(yi, xi);
    W.n[d] = (signed char)n;
    for (int k = 0; k < n; k++) {
      W.ex[d][k] = ex[k];
      W.ey[d][k] = ey[k];
    }
  }
}

// intervening.cu:298-475 for a window that reaches l, r, t, b pixels.
constexpr Walks window_walks(int l, int r, int t, int b) {
  Walks W;
  for (int d = 0; d < kWalkArea; d++) W.n[d] = -1;
  if (l > 0) {
    if (t > 0 && b > 0) walk_line(W, -l, -1, -l, 0, -l, 1);
    for (int y = -1; y > -t; y--) walk_line(W, -l, y - 1, -l, y, -l, y + 1);
  }
  if (l > 1 || t > 1 || (l > 0 && t > 0)) walk_line(W, -l, 1 - t, -l, -t, 1 - l, -t);
  if (t > 0)
    for (int x = 1 - l; x < r; x++) walk_line(W, x - 1, -t, x, -t, x + 1, -t);
  if (t > 1 || r > 1 || (t > 0 && r > 0)) walk_line(W, r - 1, -t, r, -t, r, 1 - t);
  if (r > 0)
    for (int y = 1 - t; y < 0; y++) walk_line(W, r, y - 1, r, y, r, y + 1);
  if (l > 0)
    for (int y = 1; y < b; y++) walk_line(W, -l, y - 1, -l, y, -l, y + 1);
  if (l > 1 || b > 1 || (l > 0 && b > 0)) walk_line(W, -l, b - 1, -l, b, 1 - l, b);
  if (b > 0)
    for (int x = 1 - l; x < r; x++) walk_line(W, x - 1, b, x, b, x + 1, b);
  if (b > 1 || r > 1 || (b > 0 && r > 0)) walk_line(W, r - 1, b, r, b, r, b - 1);
  if (r > 0) {
    for (int y = b - 1; y > 0; y--) walk_line(W, r, y - 1, r, y, r, y + 1);
    if (t > 0 && b > 0) walk_line(W, r, -1, r, 0, r, 1);
  }
  // intervening.cu:459-471 corner fixes: an affinity with nothing crossed
  if (t == 1 && (l == 0 || r == 0)) W.n[walk_point(-1, 0)] = 0;
  if (l == 1 && (t == 0 || b == 0)) W.n[walk_point(0, -1)] = 0;
  if (r == 1 && (t == 0 || b == 0)) W.n[walk_point(0, 1)] = 0;
  if (b == 1 && (l == 0 || r == 0)) W.n[walk_point(1, 0)] = 0;
  return W;
}

constexpr Walks kFullWalks = window_walks(5, 5, 5, 5);

constexpr bool same_walk(const Walks& a, const Walks& b, int d) {  // as sets
  if (a.n[d] != b.n[d]) return false;
  for (int i = 0; i < a.n[d]; i++) {
    bool found = false;
    for (int k = 0; k < b.n[d]; k++) found = found || (a.ex[d][i] == b.ex[d][k] && a.ey[d][i] == b.ey[d][k]);
    if (!found) return false;
  }
  return true;
}

// The second set of the points that have one: where a window is clipped,
// some points are spoken for by another walk (the windows clipped on one side
// show all of them), and a corner fix crosses nothing.  n = -1: no second set.
constexpr Walks second_walks() {
  Walks S;
  for (int d = 0; d < kWalkArea; d++) S.n[d] = -1;
  for (int side = 0; side < 4; side++)
    for (int a = 1; a < 5; a++) {
      const Walks W = window_walks(side == 0 ? a : 5, side == 1 ? a : 5, side == 2 ? a : 5, side == 3 ? a : 5);
      for (int d = 0; d < kWalkArea; d++) {
        if (S.n[d] >= 0 || W.n[d] < 0 || same_walk(W, kFullWalks, d)) continue;
        S.n[d] = W.n[d];
        for (int k = 0; k < W.n[d]; k++) {
          S.ex[d][k] = W.ex[d][k];
          S.ey[d][k] = W.ey[d][k];
        }
      }
    }
  S.n[walk_point(-1, 0)] = S.n[walk_point(0, -1)] = S.n[walk_point(0, 1)] = S.n[walk_point(1, 0)] = 0;
  return S;
}
constexpr Walks kSecondWalks = second_walks();

// A walk speaks for exactly the points inside the window, and which set a point
// d takes depends only on how far the window reaches towards it: in x and y
// each the reach to the point's side, or where that component is 0 the smaller
// of both reaches.  Bit walk_bit(d, reach in y, reach in x) of second[d] is set
// where d takes the second set.
struct WalkRules {
  uint32_t second[kWalkArea] = {};
  bool as_described = true;  // of every window, and no window had a third set
};
// In 0..29 where the point is inside the window.
constexpr int walk_bit(int d, int ry, int rx) { return walk_dy(d) ? 6 * (ry - 1) + rx : 6 * (rx - 1) + ry; }

// The rules of the points on one side in x and y (a component of 0 counts as
// negative), for windows that reach ry towards it in y.
template <int SX, int SY, int RY>
constexpr WalkRules quarter_rules() {
  WalkRules R;
  for (int rx = 0; rx < 6; rx++) {
    const Walks W = window_walks(SX < 0 ? rx : 5, SX < 0 ? 5 : rx, SY < 0 ? RY : 5, SY < 0 ? 5 : RY);
    for (int d = 0; d < kWalkArea; d++) {
      const int dx = walk_dx(d), dy = walk_dy(d);
      if ((dx > 0) != (SX > 0) || (dy > 0) != (SY > 0) || d == kWalkArea / 2) continue;
      const bool inside = rx >= (dx < 0 ? -dx : dx) && RY >= (dy < 0 ? -dy : dy);
      R.as_described = R.as_described && (W.n[d] >= 0) == inside;
      if (!inside || same_walk(W, kFullWalks, d)) continue;
      R.as_described = R.as_described && same_walk(W, kSecondWalks, d);
      R.second[d] |= 1u << walk_bit(d, RY, rx);
    }
  }
  return R;
}
template <int SX, int SY, int RY>
constexpr WalkRules kQuarterRules = quarter_rules<SX, SY, RY>();  // each within a compiler's step limit

constexpr void add_rules(WalkRules& R, const WalkRules& Q) {
  for (int d = 0; d < kWalkArea; d++) R.second[d] |= Q.second[d];
  R.as_described = R.as_described && Q.as_described;
}
template <int SX, int SY, int... RY>
constexpr void add_quarter(WalkRules& R, std::integer_sequence<int, RY...>) {
  (add_rules(R, kQuarterRules<SX, SY, RY>), ...);
}
constexpr WalkRules walk_rules() {
  WalkRules R;
  add_quarter<-1, -1>(R, std::make_integer_sequence<int, 6>());
  add_quarter<1, -1>(R, std::make_integer_sequence<int, 6>());
  add_quarter<-1, 1>(R, std::make_integer_sequence<int, 6>());
  add_quarter<1, 1>(R, std::make_integer_sequence<int, 6>());
  return R;
}
constexpr WalkRules kWalkRules = walk_rules();
static_assert(kWalkRules.as_described, "a clipped window's walks");

// The window's reach towards side `d` (a point's component) of position i of n.
constexpr int walk_reach(int d, int i, int n) {
  const int lo = i < 5 ? i : 5, hi = n - 1 - i < 5 ? n - 1 - i : 5;
  return d < 0 ? lo : d > 0 ? hi : lo < hi ? lo : hi;
}

}  // namespace dmsc
