// Numbering of the rows that a walk sets aside for k_vext_heavy, and of their
// pieces (hip/vjoin.hip).  Plain arithmetic, shared with a CPU test.
#pragma once

#include <cstdint>

#ifdef __HIP__
#define GEM_HOST_DEVICE __host__ __device__
#else
#define GEM_HOST_DEVICE
#endif

namespace gemh {

// At most this many rows and pieces per launch (a row that finds no room is
// walked by its own wave).
constexpr uint32_t HEAVY_CAP = 1u << 20, PIECE_CAP = 1u << 22;

// Rows and pieces numbered so far, refused ones among them: a launch over whole
// levels can ask for more than 2^32 pieces (2.7e11 entries in pieces of 64), and
// a number handed out twice would lose the row that had it.
struct HeavyCounters {
  unsigned long long rows, pieces;
};

// Pieces of a row of len > 0 entries, as they are numbered (a row of more than
// the table holds is refused whatever its number, and 64 rows' stay below 2^32).
GEM_HOST_DEVICE inline uint32_t heavy_pieces(uint32_t len, uint32_t piece) {
  const uint32_t n = (len - 1) / piece + 1;
  return n <= PIECE_CAP ? n : PIECE_CAP + 1;
}

// Row number h, whose n pieces are numbered from c: is there room for it?
GEM_HOST_DEVICE inline bool heavy_taken(uint64_t h, uint64_t c, uint32_t n) {
  return h < HEAVY_CAP && c + n <= PIECE_CAP;
}

// How many of its pieces have an entry in the piece table: the row's number, or
// a mark that it was refused.
GEM_HOST_DEVICE inline uint32_t heavy_entries(uint64_t c, uint32_t n) {
  return c + n <= PIECE_CAP ? n : c < PIECE_CAP ? PIECE_CAP - (uint32_t)c : 0;
}

}  // namespace gemh
