// How many workgroups a (batch, head) of the resident-key kernel gets.  Plain C++.
#pragma once

#include <cstdint>

namespace pa {

// Rounds of workgroups times what one takes, in passes of its 8 wavefronts over the keys.  Copying K and V in is priced at 3/4 of one, a
// pass that leaves every SIMD at most one wavefront at 0.6.
inline double resident_cost(int64_t heads, int n_units, int cus, int parts) {
  const double rounds = (double)((heads * parts + cus - 1) / cus);
  const int units = (n_units + parts - 1) / parts, rest = units % 8;
  return rounds * (0.75 + units / 8 + (rest == 0 ? 0. : rest <= 4 ? 0.6 : 1.));
}

// The cheapest number of workgroups per (batch, head), each with four blocks of 32 query rows or more; a larger one must be cheaper by 0.1 %.
// Only numbers at which a workgroup's blocks become fewer are priced (of several with the same blocks the smallest is the cheapest), and
// none beyond the point where copying the keys in so often costs more than the best so far: 24 heads x 32760 rows 24 prices instead of
// 256, 24 x 131072 32 instead of 1024 (a call issued in 17.1 -> 12.2 us).
inline int resident_parts(int64_t heads, int n_units, int cus, int* priced = nullptr) {
  int best = 1, count = 0;
  double best_cost = 1e30;
  const int by_units = (n_units + 3) / 4, most = by_units < 4 * cus ? by_units : 4 * cus;
  for (int parts = 1; parts <= most;) {
    const double cost = resident_cost(heads, n_units, cus, parts);
    ++count;
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = parts;
    }
    const int units = (n_units + parts - 1) / parts;
    if (units <= 1) break;
    parts = (n_units + units - 2) / (units - 1);
    // every block takes an eighth of a pass at least, every workgroup its copies
    if ((double)heads / cus * (0.75 * parts + n_units / 8.) >= best_cost) break;
  }
  if (priced) *priced = count;
  return best;
}

}  // namespace pa
