// Runs of equal cost (host/walk_runs.h): every piece's runs cover its cost, a
// run's cost stays in its bounds, and a launch whose runs could not be numbered
// in 32 bits is refused.
#include <cstdio>
#include <vector>

#include "walk_runs.h"

using namespace gemh;

namespace {

int bad = 0;
void check(bool ok, const char *what, uint64_t a, uint64_t b) {
  if (ok) return;
  std::printf("%s: bound %llu x %llu\n", what, (unsigned long long)a, (unsigned long long)b);
  ++bad;
}

}  // namespace

int main() {
  const uint64_t waves = 5120;
  for (uint64_t n : {1ull, 3ull, 64ull})
    for (int e = 0; e < 62; ++e)
      for (int64_t d : {-1, 0, 1}) {
        const uint64_t bound = (1ull << e) + d, units = 1 + bound % 1000003;
        std::vector<WalkPiece> pieces;
        for (uint64_t i = 0; i < n; ++i) pieces.push_back(WalkPiece{bound, units, 1 + 4 * (i % 8)});
        std::vector<uint32_t> cost;
        const bool fits = plan_runs(pieces, waves, &cost);
        uint64_t runs = 0;
        bool few = true;  // the runs at their longest are few enough
        for (const WalkPiece &p : pieces) few = few && p.runs(RUN_COST) < RUN_LIMIT && (runs += p.runs(RUN_COST)) < RUN_LIMIT;
        if (!few) check(!fits, "taken", bound, n);
        if (few && runs < RUN_LIMIT / 8) check(fits, "refused", bound, n);  // (shorter runs are eight times as many at most)
        check(fits == (cost.size() == n), "sizes", bound, n);
        if (!fits) continue;
        uint64_t sum = 0;
        for (uint64_t i = 0; i < n; ++i) {
          check(cost[i] >= 4 * UNIT_COST && cost[i] <= RUN_COST, "run cost", bound, n);
          const uint64_t r = pieces[i].runs(cost[i]);
          check(r && (r - 1) * cost[i] < pieces[i].cost() && r * cost[i] >= pieces[i].cost(), "cover", bound, n);
          sum += r;
        }
        check(sum < RUN_LIMIT && (uint32_t)sum == sum, "number", bound, n);
      }
  // 64 capped queries that each take a level of 2^45 entries
  std::vector<uint32_t> cost;
  check(!plan_runs(std::vector<WalkPiece>(64, WalkPiece{1ull << 45, 1 << 20, 5}), waves, &cost), "taken", 1ull << 45, 64);
  return bad > 255 ? 255 : bad;
}
