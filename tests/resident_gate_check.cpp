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
  return 0;
}
