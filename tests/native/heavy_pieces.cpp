// Numbering of set-aside rows and their pieces (host/heavy_pieces.h) far past
// both tables' ends: every entry of the piece table is written once, and those
// of a row that was taken hold that row.  `control`: the same numbers kept in 32
// bits, which the check has to find wrong.
#include <cstdio>
#include <cstring>
#include <type_traits>
#include <vector>

#include "heavy_pieces.h"

using namespace gemh;

namespace {

struct Row {
  uint64_t h, c;
  uint32_t n;
};

// Waves of 64 rows of `len` entries number them as the walk does, until more
// than `pieces` are numbered.  False: an entry was written twice, or left out.
template <class T>
bool numbered_once(uint32_t first_len, uint32_t len, uint32_t piece, uint64_t pieces) {
  constexpr uint32_t FREE = 0xFFFFFFFEu, REFUSED = 0xFFFFFFFFu;
  std::vector<uint32_t> owner(PIECE_CAP, FREE);
  std::vector<Row> rows;
  T nrows = 0, npieces = 0;
  uint64_t asked = 0;
  for (uint64_t wave = 0; asked <= pieces; ++wave) {
    // short rows until the row table is full, then long ones
    const uint32_t l = wave < HEAVY_CAP / 64 + 3 ? first_len : len, n = heavy_pieces(l, piece);
    const uint64_t h0 = nrows, c0 = npieces;
    nrows += 64;
    npieces += (T)(64ull * n);
    asked += 64ull * n;
    for (uint32_t i = 0; i < 64; ++i) {
      const uint64_t h = h0 + i, c = c0 + (uint64_t)i * n;
      const bool taken = heavy_taken(h, c, n);
      if (taken) rows.push_back(Row{h, c, n});
      for (uint32_t x = 0, e = heavy_entries(c, n); x < e; ++x) {
        if (owner[c + x] != FREE) return false;
        owner[c + x] = taken ? (uint32_t)h : REFUSED;
      }
    }
  }
  const uint64_t total = (uint64_t)npieces < PIECE_CAP ? (uint64_t)npieces : PIECE_CAP;
  for (uint64_t x = 0; x < total; ++x)
    if (owner[x] == FREE) return false;
  for (const Row &r : rows)
    for (uint32_t x = 0; x < r.n; ++x)
      if (owner[r.c + x] != r.h) return false;
  return rows.size() <= HEAVY_CAP;
}

}  // namespace

int main(int argc, char **argv) {
  using Counter = decltype(HeavyCounters::pieces);
  static_assert(std::is_same<Counter, decltype(HeavyCounters::rows)>::value, "one type");
  const uint64_t far = (1ull << 32) + (1ull << 30);
  const bool control = argc > 1 && !std::strcmp(argv[1], "control");
  int bad = 0;
  // pieces a row at first and later: the row table ends first, the piece table
  // does, a row does not fit the table at all, rows of the longest list
  const uint32_t lens[][2] = {{1, 1u << 26}, {640, 1u << 26}, {64, 65}, {1u << 28, ~0u}, {65, ~0u}};
  for (auto &l : lens) {
    const uint64_t pieces = l[1] == 65 ? 1ull << 27 : far;
    const bool ok = control ? numbered_once<uint32_t>(l[0], l[1], 64, pieces) : numbered_once<Counter>(l[0], l[1], 64, pieces);
    std::printf("%u then %u entries: %s\n", l[0], l[1], ok ? "each once" : "twice or never");
    bad += !ok;
  }
  // the wave's own sum of 64 rows stays in 32 bits
  if (64ull * heavy_pieces(~0u, 1) > 0xFFFFFFFFull) bad += 100;
  return bad;
}
