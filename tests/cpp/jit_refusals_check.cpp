// Host check of clexmc::JitRefusals: the order in which a supercell's launches
// fall back after refusals of the runtime.  Prints one line per step.
#include <cstdio>

#include "../../casmcode_clexmonte_amd/csrc/clexmc_jit.h"

int main() {
  clexmc::JitRefusals r;
  auto show = [&](const char *what) {
    std::printf("%s spread0 %d spread1 %d lds30000 %d lds40000 %d lds50000 %d\n", what, r.allows_spread(0), r.allows_spread(1),
                r.allows(30000), r.allows(40000), r.allows(50000));
  };
  show("start");
  r.refused(1, 45000, 10000);  // the spread kernel, 35,000 bytes without its rows
  show("spread");
  r.refused(1, 40000, 0);
  show("ordinary");
  r.refused(0, 50000, 0);  // (larger than one refused before)
  show("larger");
  return 0;
}
