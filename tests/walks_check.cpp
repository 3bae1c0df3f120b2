// The compiled walk rules against the walks of every clipped window: prints the
// number of windows and exits with 1 at the first disc point that differs.
#include <cstdio>

#include "../damascene_amd/csrc/walks.hpp"

using namespace dmsc;

int main() {
  int windows = 0;
  for (int l = 0; l < 6; l++)
    for (int r = 0; r < 6; r++)
      for (int t = 0; t < 6; t++)
        for (int b = 0; b < 6; b++, windows++) {
          const Walks W = window_walks(l, r, t, b);
          // a pixel with these reaches: (l, t) in an image that ends r and b past it
          for (int d = 0; d < kWalkArea; d++) {
            if (d == kWalkArea / 2) continue;  // the pixel itself
            const int dx = walk_dx(d), dy = walk_dy(d);
            const bool inside = dx >= -l && dx <= r && dy >= -t && dy <= b;
            const int at = walk_bit(d, walk_reach(dy, t, t + b + 1), walk_reach(dx, l, l + r + 1));
            const bool second = inside && (kWalkRules.second[d] >> at & 1);
            if (inside != (W.n[d] >= 0) || (inside && (at < 0 || at > 29)) ||
                (inside && !same_walk(W, second ? kSecondWalks : kFullWalks, d))) {
              std::printf("window %d %d %d %d, point %d\n", l, r, t, b, d);
              return 1;
            }
          }
        }
  std::printf("%d windows\n", windows);
  return 0;
}
