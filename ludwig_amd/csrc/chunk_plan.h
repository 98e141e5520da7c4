// chunk_plan.h -- into how many chunks of x planes a launch of tiled blocks
// cuts a lattice.  Host arithmetic only, so that tests can ask it.

#ifndef LDW_CHUNK_PLAN_H
#define LDW_CHUNK_PLAN_H

#include <stdint.h>

namespace ldw {

// A block that marches over xc planes first loads 4 phi planes and forms 2 Q
// planes, about 3 planes of work, and `slots` blocks run at once: a launch of
// n chunks of ncol columns lasts about this many plane-times.
inline int64_t chunk_cost(int nx, int64_t ncol, int slots, int n) {
  const int xc = (nx + n - 1)/n;
  return ((ncol*n + slots - 1)/slots)*(xc + 3);
}

// The number of chunks of the least cost, the fewest of equal ones: for r rounds
// of blocks the most chunks that fit them, until r rounds of one plane each
// cost as much.
inline int chunk_count(int nx, int64_t ncol, int slots) {
  int best = 1;
  int64_t cost = chunk_cost(nx, ncol, slots, 1);
  for (int64_t r = (ncol + slots - 1)/slots; 4*r < cost; r++) {
    const int64_t fit = r*slots/ncol;
    const int xc = (fit < nx) ? (int) ((nx + fit - 1)/fit) : 1;
    if (r*(xc + 3) < cost) { best = (nx + xc - 1)/xc; cost = r*(xc + 3); }
  }
  return best;
}

}  // namespace ldw

#endif
