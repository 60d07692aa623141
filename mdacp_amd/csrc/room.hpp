// room.hpp -- room for a first construction, before anything is counted (host
// arithmetic; later constructions have the last one's counts).
#pragma once
#include <algorithm>

namespace mdgpu {

// List slots of `rows` rows of `mean` entries each on average, in `bricks`
// bricks.  A slice takes 64 times its longest row, and every brick with rows
// ends with a slice that is partly empty: with one-cell bricks of 16 rows that
// is three quarters of the list (2,048 particles at rho = 0.5 in 125 such
// bricks: 512,000 slots, where the rows' own lengths ask for 177,000).  Too
// little room costs a construction a second wait, two allocations and its emit
// again.
inline double expected_slots(double rows, double mean, double bricks) {
  const double slices = rows / 64.0 + std::min(bricks, rows);
  return 64.0 * slices * (1.25 * mean + 16.0);
}

}  // namespace mdgpu
