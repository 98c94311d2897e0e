// Runs of equal cost that the waves of a walk take (hip/vjoin.hip): how a
// launch's pieces are cut into them.  Plain arithmetic, tested on the CPU.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace gemh {

// A wave of a persistent grid takes about CLAIMS runs; a run of whole units has
// at most MAX_RUN of them.
constexpr uint32_t CLAIMS = 4, MAX_RUN = 32;
// Cost of a 64-row unit besides the entries it walks, in entries: its rows'
// setup.  A run of a write walk has at most RUN_COST of it.
constexpr uint32_t UNIT_COST = 256, RUN_COST = UNIT_COST * MAX_RUN;
// The kernels number runs, and what their counters hand out past the last one,
// in 32 bits.
constexpr uint64_t RUN_LIMIT = 1ull << 31;

// A row range of a level: the output bound of its units, and the weight of an
// entry (a level with other lists costs its searches too).
struct WalkPiece {
  uint64_t bound, units, weight;
  uint64_t cost() const { return bound + UNIT_COST * units; }
  uint64_t runs(uint32_t run_cost) const { return (cost() - 1) / run_cost + 1; }
};

// The cost of a run of each piece of a launch of `waves` waves.  False when there
// would be RUN_LIMIT runs or more: final walks under a cap whose entries seldom
// survive take whole levels, which at 3.5e13 entries are 2^32 runs (with the
// last runs' numbers wrapped, they were left out and the count was too small).
// The caller then gives out whole units, of which the rows in memory make fewer.
inline bool plan_runs(const std::vector<WalkPiece> &pieces, uint64_t waves, std::vector<uint32_t> *run_cost) {
  run_cost->clear();
  double total = 0;
  for (const WalkPiece &p : pieces) total += (double)p.cost() * (double)p.weight;
  const double each = total / ((double)waves * CLAIMS) + 1;
  uint64_t runs = 0;
  for (const WalkPiece &p : pieces) {
    const double c = each / (double)p.weight;
    run_cost->push_back((uint32_t)std::min<double>(std::max<double>(c, 4 * UNIT_COST), RUN_COST));
    const uint64_t n = p.runs(run_cost->back());
    if (n >= RUN_LIMIT || (runs += n) >= RUN_LIMIT) {
      run_cost->clear();
      return false;
    }
  }
  return true;
}

}  // namespace gemh
