// The host's rules for launches whose blocks wait for each other: exits with
// the number of the first rule that does not hold, 0 if all do.
#include <memory>

#include "../damascene_amd/csrc/resident_gate.hpp"

using namespace dmsc;

int main() {
  {  // one grid at a time per device, free again after it
    auto first = std::make_unique<ResidentGrid>(0);
    if (!first->held()) return 1;
    {
      ResidentGrid second(0), other(1);
      if (second.held() || !other.held()) return 2;
    }
    ResidentGrid third(0);  // the refused one has not freed it
    if (third.held()) return 3;
    first.reset();
    ResidentGrid again(0), device1(1);
    if (!again.held() || !device1.held()) return 4;
  }
  {  // solves left out after a launch has given up: 1, 2, 4, ... 64, 64
    ResidentBackoff b;
    if (!b.due(100) || !b.due(100)) return 5;
    for (int want = 1, i = 0; i < 9; i++, want = want < 64 ? 2 * want : 64) {
      b.stalled(100);
      for (int k = 0; k < want; k++)
        if (b.due(100)) return 6;
      if (!b.due(100)) return 7;
    }
    b.stalled(100);
    if (b.due(50) || !b.due(101)) return 8;  // a larger bound is tried at once
    b.completed();
    if (!b.due(100)) return 9;
    b.stalled(100);  // from one again
    if (b.due(100) || !b.due(100)) return 10;
  }
  return 0;
}
