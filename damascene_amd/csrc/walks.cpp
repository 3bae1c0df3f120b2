// walks.cpp -- which of a disc point's two crossed sets each clipped window
// takes (walks.hpp).
#include "walks.hpp"

#include <mutex>

namespace dmsc {

static std::vector<uint8_t> build(bool narrow) {
  std::vector<uint8_t> code((size_t)kReaches * kReaches * kWalkArea, 0);
  for (int l = 0; l < 6; l++)
    for (int r = 0; r < 6; r++)
      for (int t = 0; t < 6; t++)
        for (int b = 0; b < 6; b++) {
          if (!narrow && !((l == 5 || r == 5) && (t == 5 || b == 5))) continue;
          const Walks W = window_walks(l, r, t, b);
          for (int d = 0; d < kWalkArea; d++) {
            if (W.n[d] < 0) continue;
            const int c = same_walk(W, kFullWalks, d) ? 1 : same_walk(W, kSecondWalks, d) ? 2 : 0;
            if (c == 0) return {};
            code[((size_t)(t * 6 + b) * kReaches + (l * 6 + r)) * kWalkArea + d] = (uint8_t)c;
          }
        }
  return code;
}

const std::vector<uint8_t>& walk_codes(bool narrow) {
  static std::vector<uint8_t> codes[2];
  static std::once_flag once[2];
  std::call_once(once[narrow], [narrow] { codes[narrow] = build(narrow); });
  return codes[narrow];
}

}  // namespace dmsc
