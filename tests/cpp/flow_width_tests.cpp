// The launch width of the sweeps without barriers (scx_tune.h): the whole grid, 8 workgroups for
// each one per XCD, fits one workgroup per CU.
#include <cstdio>

#include "scx_tune.h"

int main() {
  for (int cus : {1, 7, 8, 31, 32, 64, 100, 128, 256, 304})
    for (int per_cu = 1; per_cu <= 4; ++per_cu)
      for (int xcds = 1; xcds <= 8; ++xcds) {
        const int most = scx::flow_width_limit(per_cu * cus, cus, 256, xcds);
        const int grid = (most + xcds - 1) / xcds * 8;
        if (grid > cus || most > 256 || (cus >= 8) != (most > 0)) {
          std::fprintf(stderr, "%d CUs, %d per CU, %d XCDs: %d\n", cus, per_cu, xcds, most);
          return 1;
        }
      }
  // the whole card: 32 workgroups an XCD; held back by a narrower persistent launch
  if (scx::flow_width_limit(256, 256, 256, 8) != 256 || scx::flow_width_limit(256, 256, 256, 1) != 32 ||
      scx::flow_width_limit(16, 256, 256, 1) != 2)
    return 1;
  std::printf("flow width tests passed\n");
  return 0;
}
