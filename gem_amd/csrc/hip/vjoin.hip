// Vertex-at-a-time join over many queries at once (the batched path).
//
// Same counts as the edge-at-a-time join (the reference's join(),
// in-core/lib/join/src/join_trie.cu:1087-1277), which is order-invariant, but
// each level adds one query vertex and applies ALL its edges to earlier
// vertices at once: the candidates of the new vertex are the intersection of
// the backward tables' rows (sorted position lists in its candidate set), so a
// closing edge prunes rows before they are ever written instead of after a
// whole level has been materialised.
//
//   k_vlen    per 64-row unit: sum over rows of the shortest list length
//             (an upper bound on the level's output, used to size and split)
//   k_vext    waves walk the shortest ("driver") list of each of their 64
//             rows, 256 items per step (four per lane); each item is
//             binary-searched in the row's other lists and compared with the
//             equal-label columns; survivors are counted (last level) or
//             appended to the output (row order is free); rows with long
//             driving lists are left to k_vext_heavy
//   k_vext_heavy  walks those rows in fixed-size pieces spread over waves
//   k_vcount1 last level with a single backward list: |list| minus the
//             equal-label columns found in it (no walk)
//
// Work distribution: each launch covers many (query, level, row range) items;
// the waves of a persistent grid take runs of their 64-row units, so queries
// of very different sizes share one launch.  The host scheduler
// (host/vsched.h) keeps, per query, a depth-first stack of pending levels and
// cuts them into 64-row-unit ranges whose output bounds fit a memory budget
// shared by all queries; a query stops as soon as its count exceeds the cap.
//
// What bounds the walks is the output: rows written, and the atomics that hand
// out their places (one address serves one per 9-11 ns).  Hence rows hold only
// the columns that are read again (VLevel::src; 2.1x fewer bytes written on 16
// queries of up to 24 vertices, 2^20 R-MAT), and places are reserved once per
// run of a one-list level and once per full stage of the others.  With runs of
// equal cost, units cut between rows and the searches below, k_vext<write> of
// one pass went from 190 to 63 ms on those queries, from 13.3 to 2.1 ms on 24
// exact queries of 4-9 vertices on 2^18.  While it runs now (63 ms pass), the L1
// serves an access in three of four cycles, the vector units issue in two of
// five, and rows go to HBM at 1.8 TB/s.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>

#include "ctx.h"
#include "tcache.h"
#include "vjoin.h"
#include "wave.h"

namespace gemd {

constexpr uint32_t VB = 256;  // rows per task block
constexpr uint32_t VW = VB / 64;
// survivors a wave stages in LDS before it reserves output rows for them (a
// step of k_vext adds at most 256, one of k_vext_heavy 128)
constexpr uint32_t VSTAGE = 384;

__device__ __forceinline__ uint32_t vposition_in(const uint64_t *bm, const uint32_t *rank, uint32_t v) {
  const uint64_t word = ldg(bm + (v >> 6));
  const uint32_t b = v & 63;
  if (!((word >> b) & 1ull)) return NOT_FOUND;
  return ldg(rank + (v >> 6)) + (uint32_t)__popcll(word & ((1ull << b) - 1));
}

// Level descriptors and launch tables do not change while a kernel runs: read
// through the constant address space, uniform indexes become scalar loads.
#define GEM_CONST const __attribute__((address_space(4)))
using CLevel = GEM_CONST VLevel;
using CItem = GEM_CONST VItem;
using CWord = GEM_CONST uint64_t;

__device__ __forceinline__ uint32_t find_item(const uint64_t *blk_prefix, uint32_t nitems, uint64_t g) {
  uint32_t lo = 0, hi = nitems;  // largest t with blk_prefix[t] <= g
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (blk_prefix[mid] <= g)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// ------------------------------------------------------------ length pass
// Per 64-row unit (wave w of 256-row block g -> unit_u[4g + w]): the sum over
// its rows of the shortest backward list, an upper bound on its output rows.
// Rows cost nearly the same (one offset pair per list), so blocks take the
// 256-row tasks in turn: a work queue is one device-wide atomic per task, about
// 11.5 ns each on one address, which bounded this kernel (4.5 ms for the
// 400,000 tasks of a 10^8-row level, whose reads take a tenth of that).
__global__ void __launch_bounds__(VB) k_vlen(const VItem *__restrict__ items, uint32_t nitems,
                                            const uint64_t *__restrict__ blk_prefix, uint64_t *__restrict__ unit_u) {
  const uint64_t total = blk_prefix[nitems];
  uint32_t t = 0;
  for (uint64_t g = blockIdx.x; g < total; g += gridDim.x) {
    while (blk_prefix[t + 1] <= g) ++t;
    const VItem &it = items[t];
    CLevel &L = *(CLevel *)it.lv;
    const uint64_t r = it.row_begin + (g - blk_prefix[t]) * VB + threadIdx.x;
    uint64_t u = 0;
    if (r < it.row_end) {
      const uint32_t *row = it.rows + r * it.k;
      u = ~0ull;
      for (uint32_t j = 0; j < L.nb; ++j) {
        const uint32_t p = ldg(row + L.key_col[j]);
        const uint64_t *off = L.toff[j];
        const uint64_t len = ldg(off + p + 1) - ldg(off + p);
        u = len < u ? len : u;
      }
    }
    u = wave_sum_u64(u);
    if (threadIdx.x % 64 == 0) unit_u[g * VW + threadIdx.x / 64] = u;
  }
}

// Runs of consecutive tasks handed to the waves of a persistent grid.  Wave
// w starts on run w without asking; later runs come from nq = min(WQ, waves)
// counters (wave w asks counter w % nq, which hands out the runs that are w
// modulo nq, so every counter has a wave that empties it).  One
// counter is an atomic on one address, which the device serves one per 11.5
// ns whatever asks: 8,192 waves finding an empty queue took 95 us, and a queue
// of 64-row tasks bounded every large launch.  Runs are as long as leaves a
// wave about CLAIMS of them, so uneven tasks still even out.
using gemh::CLAIMS;
using gemh::MAX_RUN;
struct Runs {
  uint32_t ntask, nrun, run;
  uint32_t per, nq, sub, given;
  unsigned int *q;
  // n tasks, below gemh::RUN_LIMIT: 64-row units of the rows in memory, or runs
  // that gemh::plan_runs made; w, nw: this wave and the waves of the grid
  __device__ __forceinline__ Runs(uint64_t n, uint32_t w, uint32_t nw, uint32_t max_run, unsigned int *queue)
      : ntask((uint32_t)n), run(w) {
    const uint32_t p = ntask / (nw * CLAIMS);
    per = p < 1 ? 1 : p > max_run ? max_run : p;
    nrun = (ntask - 1) / per + 1;
    nq = nw < WQ ? nw : WQ;
    sub = w % nq;
    given = (nw - sub + nq - 1) / nq;
    q = queue + sub * WQ_STRIDE;
  }
  __device__ __forceinline__ bool valid() const { return run < nrun; }
  __device__ __forceinline__ uint32_t begin() const { return run * per; }
  __device__ __forceinline__ uint32_t end() const { return ntask - run * per < per ? ntask : run * per + per; }
  __device__ __forceinline__ void next() {
    if (given * nq + sub >= nrun) {  // every run was given at the start
      run = nrun;
      return;
    }
    uint32_t c = 0;
    if (lane_id() == 0) c = atomicAdd(q, 1u);
    run = (given + readlane_u32(c, 0)) * nq + sub;
  }
};

// Device address of the list of key p in backward table j (b = its first
// offset): in HBM, or through the streamed tables' block map.
template <bool OOC>
__device__ __forceinline__ uint64_t list_addr(CLevel &L, uint32_t j, uint32_t p, uint64_t b) {
  if (OOC) return ldg(L.vmap[j] + (p >> L.kshift[j])) + 4 * b;
  return (uint64_t)(uintptr_t)(L.tval[j] + b);
}

// ------------------------------------------------------ extend (walk) pass
using gemh::RUN_COST;
using gemh::UNIT_COST;

// A unit that costs more than this part of a run is cut between its rows: row
// i starts at the unit's cost plus UNIT_COST / 64 a row and the entries of the
// rows before it, and belongs to the run that holds its start.  (With units
// whole, one unit of 64 rows of up to 1024 entries kept a wave for 1.0 to 2.8 ms
// of launches of 1.5 to 3 ms, whose waves were busy 58% of the time.)
__device__ __forceinline__ bool unit_is_cut(uint64_t cost, uint32_t run) { return cost > run / 2; }

// The units [*j0, *j1) of an item of n units that a run looks at: those whose
// cost starts in [at, at + run) and the one before when it is cut and reaches
// into the run: cost(j) = units[j] - units[0] + UNIT_COST * j, at < cost(n),
// run <= RUN_COST (so they are at most MAX_RUN + 1).  The first is searched 64
// places at a time, the end looked up in one step.
__device__ __forceinline__ void unit_range(const uint64_t *units, uint32_t n, uint64_t at, uint32_t run, uint32_t *j0,
                                           uint32_t *j1) {
  const uint64_t first = ldg(units);
  uint32_t b = 0;
  if (at) {
    uint32_t a = 0;  // cost(a) < at <= cost(b)
    b = n;
    while (b - a > 1) {
      const uint32_t step = (b - a - 1) / 64 + 1;
      const uint64_t x = (uint64_t)a + (uint64_t)(lane_id() + 1) * step;
      bool reached = x >= b;
      if (!reached) reached = ldg(units + x) - first + (uint64_t)UNIT_COST * x >= at;
      const uint32_t f = (uint32_t)__builtin_ctzll(__ballot(reached));
      const uint64_t hi = (uint64_t)a + (uint64_t)(f + 1) * step;
      a += f * step;
      b = hi < b ? (uint32_t)hi : b;
    }
  }
  const uint64_t x = (uint64_t)b + lane_id();
  bool past = x >= n;
  if (!past) past = ldg(units + x) - first + (uint64_t)UNIT_COST * x >= at + run;
  *j1 = b + (uint32_t)__builtin_ctzll(__ballot(past));
  if (b) {
    const u64x2 c = ld_pair(units + b - 1);
    if (unit_is_cut(c.y - c.x + UNIT_COST, run) && c.y - first + (uint64_t)UNIT_COST * b > at) --b;
  }
  *j0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
}

// Loads of N lists (N equal-label columns) of one row at a time, so that a
// row's setup is a few rounds of independent loads and not a chain of them.
template <int N, class F>
__device__ __forceinline__ void row_lists(CLevel &L, const uint32_t *row, uint32_t j, F &&f) {
  uint32_t p[N];
  u64x2 o[N];
#pragma unroll
  for (int i = 0; i < N; ++i) p[i] = ldg(row + L.key_col[j + i]);
#pragma unroll
  for (int i = 0; i < N; ++i) o[i] = ld_pair(L.toff[j + i] + p[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) f(j + i, p[i], o[i].x, (uint32_t)(o[i].y - o[i].x));
}
template <int N, class F>
__device__ __forceinline__ void row_dups(CLevel &L, const uint32_t *row, uint32_t c, F &&f) {
  uint32_t p[N];
#pragma unroll
  for (int i = 0; i < N; ++i) p[i] = ldg(row + L.dup_col[c + i]);
#pragma unroll
  for (int i = 0; i < N; ++i) p[i] = ldg(L.dup_can[c + i] + p[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) f(c + i, p[i]);
}

// Other lists and equal-label columns of a row that k_vext keeps in LDS; what
// a level has beyond them is read again for the items that are still wanted
// by then.  Sized for the levels that occur (most have one or two lists): with
// room for every list of the widest level of a batch, a launch had 11 of a
// CU's 32 waves.
constexpr uint32_t LDS_LISTS = 2, LDS_DUPS = 8;

// Sets aside the rows of the lanes that ask (want; list of len entries, row r
// of item t) for k_vext_heavy; returns the lanes whose row was taken.  Rows and
// pieces are numbered by two atomics per wave; pieces of refused rows are marked.
__device__ __forceinline__ uint64_t set_aside(const HeavyOut &H, bool want, uint32_t t, uint32_t len, uint64_t r) {
  const uint64_t m = __ballot(want);
  if (!m) return 0;
  const uint32_t n = want ? gemh::heavy_pieces(len, H.piece) : 0, incl = wave_incl_scan_u32(n);
  uint64_t h = 0, c = 0;
  if (lane_id() == 0) h = atomicAdd(&H.ctr->rows, (unsigned long long)__popcll(m));
  if (lane_id() == 63) c = atomicAdd(&H.ctr->pieces, (unsigned long long)incl);
  h = readlane_u64(h, 0) + rank_below(m);
  c = readlane_u64(c, 63) + incl - n;
  const bool taken = want && gemh::heavy_taken(h, c, n);
  if (taken) H.rows[h] = HeavyRow{t, len, r, (uint32_t)c, 0};
  const uint32_t entries = gemh::heavy_entries(c, n);
  for (uint32_t x = 0; x < entries; ++x) H.piece_row[c + x] = taken ? (uint32_t)h : NOT_FOUND;
  return __ballot(taken);
}

// Each wave takes runs of 64-row units on its own (no block barrier): of equal
// cost by the length pass's unit prefix, so that a run's rows are reserved
// together however many units that takes, and no wave is left with a run of
// long lists (runs of a fixed number of units: the longest launch took 18 ms
// instead of 5; final walks under a cap with their heavy rows: 0.47 ms a launch,
// by cost 0.40).  Uncapped final walks and streamed ones are not measured, or are
// cut into task groups, and take runs of whole units.  For each of its rows the
// shortest backward list drives; a row whose driving list is longer than the
// threshold is not walked here but appended to the heavy-row list (when it has
// room), which k_vext_heavy then walks in fixed-size chunks spread over all
// waves: a hub row no longer holds one wave for the whole launch.
// Dynamic LDS per wave: lists (lcap x 64 x (u64 address + u32 length)) and
// vertices of equal-label columns (dcap x 64 u32).
// An item (row, value) survives when its value is in the row's other lists and
// its vertex differs from those of the row's equal-label columns.  Survivors
// are written as whole rows: their (parent row, new value) pairs are
// staged in LDS, over all tasks of the item that the wave has in hand, then
// the wave reserves output rows for all of them at once (one atomic on the
// item's counter) and writes them as one run of consecutive words.
// The item count is read from device memory so that one captured graph can
// replay the launch for any number of items.  Tasks [g_begin, g_end) of the
// launch (256-row units) are processed (streamed tables run a launch in task
// groups).
template <bool FINAL, bool OOC>
__global__ void __launch_bounds__(VB) __attribute__((amdgpu_waves_per_eu(6)))
k_vext(const VItem *__restrict__ items, const uint32_t *__restrict__ nitems_p, const uint64_t *__restrict__ blk_prefix,
       unsigned int *__restrict__ queue, uint32_t lcap, uint32_t dcap,
       unsigned long long *__restrict__ prof_items, unsigned long long *__restrict__ prof_out, uint64_t g_begin,
       uint64_t g_end, const HeavyOut heavy_in) {
  const uint32_t nitems = *nitems_p;
  const uint64_t total = blk_prefix[nitems] < g_end ? blk_prefix[nitems] : g_end;
  if (g_begin >= total) return;
  // final walks of measured pieces take runs of equal cost too (all of a launch)
  const bool by_cost = !OOC && (!FINAL || ((CItem *)items)[0].run_cost);
  HeavyOut heavy = heavy_in;
  if (by_cost) heavy.threshold *= 2;  // see ExtSlot::heavy_out
  __shared__ uint32_t st[VW][64];          // first item of each row
  __shared__ uint64_t drv[VW][64];         // address of each row's driving list
  __shared__ uint8_t drv_j[VW][64];        // which of the row's lists drives
  __shared__ uint8_t full_row[VW][64];     // the unit's rows that have entries
  __shared__ uint32_t marks[VW][8];        // bit i: a row's entries start at item i of the step
  __shared__ uint64_t aside[VW][MAX_RUN + 1];  // counted runs: rows of each task set aside as heavy
  __shared__ uint32_t sv_row[VW][VSTAGE];  // staged survivors: row in the item's range
  __shared__ uint32_t sv_val[VW][VSTAGE];  // and new value
  extern __shared__ unsigned char vlds[];
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64;
  unsigned char *mine = vlds + (size_t)w * 64 * (lcap * 12 + dcap * 4);
  uint64_t *obase = reinterpret_cast<uint64_t *>(mine);                            // [lcap][64]
  uint32_t *olen = reinterpret_cast<uint32_t *>(mine + (size_t)64 * 8 * lcap);     // [lcap][64]
  uint32_t *dvert = reinterpret_cast<uint32_t *>(mine + (size_t)64 * 12 * lcap);   // [dcap][64]
  uint64_t walked = 0, written = 0;
  // item in hand: index, its task range [ta, tb), and its fields
  uint32_t t = NOT_FOUND;
  uint64_t ta = 0, tb = 0;
  const VLevel *lv = nullptr;
  const uint32_t *in = nullptr;  // first row of the item's range
  uint64_t nrow = 0;
  uint32_t k = 1, ko = 1;  // columns read and written
  uint64_t survivors = 0;  // final level: survivors of the item in hand
  uint32_t pend = 0;       // survivors staged in LDS, not yet written
  bool counted = false;    // output rows already reserved, from `cursor` on
  uint64_t cursor = 0;
  // Write the staged survivors: one reservation for all of them, then a lane
  // per survivor copies its columns, up to four at a time and two survivors in
  // flight.  (A lane per output word, whose column and survivor it looked up,
  // spent 18 vector instructions a word.)
  auto flush = [&]() {
    CItem &I = ((CItem *)items)[t];
    if (FINAL) {
      if (l == 0 && survivors) atomicAdd(I.counter, (unsigned long long)survivors);
      survivors = 0;
      return;
    }
    if (!pend) return;
    uint64_t base = cursor;
    cursor += pend;
    if (!counted) {
      if (l == 0) base = atomicAdd(I.counter, (unsigned long long)pend);
      base = readlane_u64(base, 0);
    }
    const uint64_t room = I.out_cap > base ? I.out_cap - base : 0;
    const uint32_t n = pend < room ? pend : (uint32_t)room;
    CLevel &L = *(CLevel *)lv;
    uint32_t *dst = I.out + base * ko;
    written += (uint64_t)n * 4 * ko;
    for (uint32_t b = 0; b < n; b += 128) {
      uint32_t v[2];
      const uint32_t *row[2];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const uint32_t i = b + 64 * g + l < n ? b + 64 * g + l : n - 1;
        v[g] = sv_val[w][i];
        row[g] = in + (uint64_t)sv_row[w][i] * k;
      }
      for (uint32_t c = 0; c < ko; c += 4) {
        const uint32_t m = ko - c < 4 ? ko - c : 4;
        u32x4 x[2];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < m) {
            const uint32_t from = L.src[c + e];
#pragma unroll
            for (int g = 0; g < 2; ++g) x[g][e] = from == COL_NEW ? v[g] : ldg(row[g] + from);
          }
#pragma unroll
        for (int g = 0; g < 2; ++g)
          if (b + 64 * g + l < n) st_words(dst + (size_t)(b + 64 * g + l) * ko + c, x[g], m);
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    pend = 0;
  };
  // the item in hand becomes item x
  auto open = [&](uint32_t x) {
    if (t != NOT_FOUND) flush();
    t = x;
    counted = false;
    CItem &I = ((CItem *)items)[t];
    lv = I.lv;
    k = I.k;
    if (!FINAL) ko = ((CLevel *)lv)->kout;
    in = I.rows + I.row_begin * k;
    nrow = I.row_end - I.row_begin;
  };
  // is the lane's row, of len entries, of unit j the run's that starts at `at`?
  auto owned = [&](uint64_t j, uint32_t len, uint64_t at) {
    CItem &I = ((CItem *)items)[t];
    CWord *u = (CWord *)I.units;
    const uint64_t a = u[j], b = u[j + 1];
    if (!unit_is_cut(b - a + UNIT_COST, I.run_cost)) return true;
    const uint32_t n = len < (1u << 25) ? len : 1u << 25;
    const uint64_t c = a - u[0] + UNIT_COST * j + wave_incl_scan_u32(n) - n + UNIT_COST / 64 * l;
    return c >= at && c - at < I.run_cost;
  };
  // walk units [j0, j1) of the item in hand (at most MAX_RUN of them; a write
  // walk's run that starts at cost `at`: MAX_RUN + 1)
  auto walk = [&](uint64_t j0, uint64_t j1, uint64_t at = 0) {
    CLevel &L = *(CLevel *)lv;
    const uint32_t nb = L.nb, ndup = L.ndup;
    if (!FINAL && nb == 1) {
      // One list: every entry survives but those of the equal-label columns,
      // so the run's rows are counted first (the vertices' positions searched
      // in the list) and reserved by one atomic.
      flush();
      counted = true;
      uint64_t cnt = 0;
      for (uint64_t j = j0; j < j1; ++j) {
        const uint64_t r = j * 64 + l;
        const uint32_t *row = in + r * k;
        uint32_t len = 0;
        uint64_t addr = 0;
        if (r < nrow) {
          const uint32_t p = ldg(row + L.key_col[0]);
          const u64x2 o = ld_pair(L.toff[0] + p);
          len = (uint32_t)(o.y - o.x);
          addr = list_addr<OOC>(L, 0, p, o.x);
        }
        if (!OOC && !owned(j, len, at)) len = 0;
        const uint64_t taken = set_aside(heavy, len > heavy.threshold, t, len, ((CItem *)items)[t].row_begin + r);
        if ((taken >> l) & 1ull) len = 0;  // walked by k_vext_heavy
        if (l == 0) aside[w][j - j0] = taken;
        cnt += len;
        if (len)
          for (uint32_t d = 0; d < ndup; ++d) {
            const uint32_t pos = vposition_in(L.bm_new, L.rank_new, ldg(L.dup_can[d] + ldg(row + L.dup_col[d])));
            if (pos != NOT_FOUND && sorted_contains(reinterpret_cast<const uint32_t *>(addr), (uint64_t)len, pos))
              --cnt;
          }
      }
      cnt = wave_sum_u64(cnt);
      cursor = 0;
      if (l == 0 && cnt) cursor = atomicAdd(((CItem *)items)[t].counter, (unsigned long long)cnt);
      cursor = readlane_u64(cursor, 0);
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
  for (uint64_t j = j0; j < j1; ++j) {
    const uint64_t rbase = j * 64;  // in the item's range
    if (rbase >= nrow) break;
    const bool valid = rbase + l < nrow;
    const uint32_t *row = in + (rbase + l) * k;
    // per-row lists: the shortest one drives, the others are probed
    uint32_t dlen = 0, dj = 0;
    uint64_t daddr = 0;
    if (valid) {
      dlen = 0xFFFFFFFFu;
      auto take = [&](uint32_t j, uint32_t p, uint64_t b, uint32_t len) {
        const bool less = len < dlen;
        const uint64_t a = list_addr<OOC>(L, j, p, b);
        if (less) {
          dlen = len;
          dj = j;
          daddr = a;
        }
        if (nb > 1 && j < lcap) {
          obase[j * 64 + l] = a;
          olen[j * 64 + l] = len;
        }
      };
      uint32_t i = 0;
      for (; i + 4 <= nb; i += 4) row_lists<4>(L, row, i, take);
      if (i + 2 <= nb) {
        row_lists<2>(L, row, i, take);
        i += 2;
      }
      if (i < nb) row_lists<1>(L, row, i, take);
    }
    if (by_cost && !owned(j, dlen, at)) dlen = 0;
    const uint64_t taken =
        !FINAL && counted
            ? aside[w][j - j0]
            : set_aside(heavy, dlen > heavy.threshold, t, dlen, ((CItem *)items)[t].row_begin + rbase + l);
    if ((taken >> l) & 1ull) dlen = 0;  // walked by k_vext_heavy
    // a row with nothing to walk here (empty driving list, or set aside as a
    // heavy row) owns no item of the steps below, so its equal-label columns
    // are never read: skip their loads
    if (dlen) {
      auto take = [&](uint32_t c, uint32_t v) { dvert[c * 64 + l] = v; };
      const uint32_t nd = ndup < dcap ? ndup : dcap;
      uint32_t c = 0;
      for (; c + 4 <= nd; c += 4) row_dups<4>(L, row, c, take);
      if (c + 2 <= nd) {
        row_dups<2>(L, row, c, take);
        c += 2;
      }
      if (c < nd) row_dups<1>(L, row, c, take);
    }
    const uint32_t incl = wave_incl_scan_u32(dlen);
    const uint32_t wtotal = readlane_u32(incl, 63);
    const uint32_t start = incl - dlen;
    st[w][l] = start;
    drv[w][l] = daddr;
    {
      const uint64_t full = __ballot(dlen);
      if (dlen) full_row[w][rank_below(full)] = (uint8_t)l;
    }
    if (nb > 1) drv_j[w][l] = (uint8_t)dj;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    walked += wtotal;
    // 256 items per step, four per lane (items s + 64 g + l), so that each
    // lane has four loads in flight at every stage of the probes.  An item's
    // row is the last one to start at or before it: the rows that start in the
    // step mark their items, and the marks up to an item are counted (searched
    // in the starts, the rows took a fifth of the vector instructions).
    uint32_t rows_before = 0;  // rows with entries that start before the step
    for (uint32_t s = 0; s < wtotal; s += 256) {
      uint32_t val[4], rw[4];
      bool keep[4];
      if (l < 8) marks[w][l] = 0;
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (dlen && start - s < 256) atomicOr(&marks[w][(start - s) / 32], 1u << ((start - s) % 32));
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t item = s + 64u * g + l;
        keep[g] = item < wtotal;
        const uint32_t mlo = __builtin_amdgcn_readfirstlane(marks[w][2 * g]);
        const uint32_t mhi = __builtin_amdgcn_readfirstlane(marks[w][2 * g + 1]);
        const uint64_t m = (uint64_t)mhi << 32 | mlo;
        rw[g] = full_row[w][rows_before + rank_below(m) + ((m >> l) & 1) - 1];
        rows_before += (uint32_t)__popcll(m);
        val[g] = keep[g] ? ldg(reinterpret_cast<const uint32_t *>(drv[w][rw[g]]) + (item - st[w][rw[g]])) : 0;
      }
      for (uint32_t j = 0; nb > 1 && j < nb; ++j) {
        const uint32_t *lists[4];
        uint32_t lens[4];
        bool probe[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          probe[g] = keep[g] && drv_j[w][rw[g]] != j;
          lists[g] = nullptr;
          lens[g] = 0;
          if (j < lcap) {
            lists[g] = reinterpret_cast<const uint32_t *>(obase[j * 64 + rw[g]]);
            lens[g] = olen[j * 64 + rw[g]];
          } else if (probe[g]) {
            const uint32_t p = ldg(in + (rbase + rw[g]) * k + L.key_col[j]);
            const u64x2 o = ld_pair(L.toff[j] + p);
            lists[g] = reinterpret_cast<const uint32_t *>(list_addr<OOC>(L, j, p, o.x));
            lens[g] = (uint32_t)(o.y - o.x);
          }
        }
        bool hit[4] = {probe[0], probe[1], probe[2], probe[3]};
        contains_quad(lists, lens, val, hit, in);
#pragma unroll
        for (int g = 0; g < 4; ++g) keep[g] = keep[g] && (hit[g] || !probe[g]);
      }
      if (ndup) {
        uint32_t vert[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) vert[g] = keep[g] ? ldg(L.can_new + val[g]) : 0;
        for (uint32_t c = 0; c < ndup; ++c) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            if (c < dcap)
              keep[g] = keep[g] && dvert[c * 64 + rw[g]] != vert[g];
            else if (keep[g])
              keep[g] = ldg(L.dup_can[c] + ldg(in + (rbase + rw[g]) * k + L.dup_col[c])) != vert[g];
          }
        }
      }
      uint64_t m[4];
      uint32_t nk = 0, before[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        m[g] = __ballot(keep[g]);
        before[g] = nk;
        nk += (uint32_t)__popcll(m[g]);
      }
      if (FINAL) {
        survivors += nk;
      } else if (nk) {
        // stage this step's survivors after the pending ones; the staging
        // area is written out when the next step might not fit
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (keep[g]) {
            const uint32_t i = pend + before[g] + rank_below(m[g]);
            sv_row[w][i] = (uint32_t)rbase + rw[g];
            sv_val[w][i] = val[g];
          }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        pend += nk;
        if (pend > VSTAGE - 256) flush();
      }
    }
    // st / drv / LDS lists of this wave are rewritten by its next task
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  };
  const uint32_t bw = blockDim.x / 64;
  if (!by_cost) {
    // tasks are 64-row units, numbered through the launch
    Runs runs((total - g_begin) * VW, blockIdx.x * bw + w, gridDim.x * bw, FINAL ? 4 : 8, queue);
    for (; runs.valid(); runs.next())
      for (uint64_t q = g_begin * VW + runs.begin(), qe = g_begin * VW + runs.end(); q < qe;) {
        const uint64_t g = q / VW;
        if (t == NOT_FOUND || g < ta || g >= tb) {
          open(find_item(blk_prefix, nitems, g));
          ta = blk_prefix[t];
          tb = blk_prefix[t + 1];
        }
        const uint64_t qn = tb * VW < qe ? tb * VW : qe;
        walk(q - ta * VW, qn - ta * VW);
        q = qn;
      }
  } else {
    // tasks are runs of units of about equal cost: run i of an item holds what
    // starts in [i, i + 1) * run_cost (the item's)
    Runs runs(total - g_begin, blockIdx.x * bw + w, gridDim.x * bw, 1, queue);
    for (; runs.valid(); runs.next()) {
      const uint64_t g = g_begin + runs.begin();
      const uint32_t x = find_item(blk_prefix, nitems, g);
      if (x != t) open(x);
      CItem &I = ((CItem *)items)[t];
      uint32_t j0, j1;
      const uint64_t at = (g - blk_prefix[t]) * I.run_cost;
      unit_range(I.units, I.nunits, at, I.run_cost, &j0, &j1);
      if (j0 < j1) walk(j0, j1, at);
    }
  }
  if (t != NOT_FOUND) flush();
  if (prof_items && l == 0 && walked) atomicAdd(prof_items, (unsigned long long)walked);
  if (prof_out && l == 0 && written) atomicAdd(prof_out, (unsigned long long)written);
}

// Entries of a staged window of the first other list (k_vext_heavy).
constexpr uint32_t HWIN = 512;

// Heavy rows: each wave task walks `chunk` entries of one row's driving list
// (the same list the main pass picked: shortest, first on ties), probing the
// row's other lists and equal-label columns; survivors are counted or appended
// to the row's item output like the main pass's.
template <bool FINAL, bool OOC>
__global__ void __launch_bounds__(VB) __attribute__((amdgpu_waves_per_eu(8)))
k_vext_heavy(const VItem *__restrict__ items, const HeavyOut heavy, unsigned int *__restrict__ queue,
             unsigned long long *__restrict__ prof_items, unsigned long long *__restrict__ prof_out) {
  __shared__ uint64_t oaddr[VW][GEM_MAX_QV];
  __shared__ uint32_t olen[VW][GEM_MAX_QV], dpos[VW][GEM_MAX_QV];
  __shared__ uint32_t wend[VW][64];   // window ends in the first other list
  __shared__ uint32_t win[VW][HWIN];  // staged window
  __shared__ uint32_t prow[VW][GEM_MAX_QV], hsv[VW][VSTAGE];  // parent row, staged surviving values
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64;
  const uint64_t asked = heavy.ctr->pieces;
  const uint32_t total = asked < gemh::PIECE_CAP ? (uint32_t)asked : gemh::PIECE_CAP, chunk = heavy.piece;
  if (!total) return;
  uint64_t walked = 0, written = 0;
  const uint32_t bw = blockDim.x / 64;
  Runs runs(total, blockIdx.x * bw + w, gridDim.x * bw, 1, queue);  // a piece is long enough to ask for one at a time
  for (; runs.valid(); runs.next()) {
    const uint32_t wt = runs.begin();
    const uint32_t h = __builtin_amdgcn_readfirstlane(heavy.piece_row[wt]);
    if (h == NOT_FOUND) continue;
    const HeavyRow e = heavy.rows[h];
    const VItem it = items[e.t];
    CLevel &L = *(CLevel *)it.lv;
    const uint32_t nb = L.nb, ndup = L.ndup;
    const uint32_t *row = it.rows + e.r * it.k;
    // the row's lists (every lane computes the same; lane j keeps list j)
    uint32_t dlen = 0xFFFFFFFFu, dj = 0, dp = 0;
    uint64_t dbase = 0;
    for (uint32_t j = 0; j < nb; ++j) {
      const uint32_t p = ldg(row + L.key_col[j]);
      const uint64_t *off = L.toff[j];
      const uint64_t b = ldg(off + p);
      const uint32_t len = (uint32_t)(ldg(off + p + 1) - b);
      if (len < dlen) {
        dlen = len;
        dj = j;
        dbase = b;
        dp = p;
      }
    }
    const uint32_t *dlist = reinterpret_cast<const uint32_t *>(list_addr<OOC>(L, dj, dp, dbase));
    if (l < nb) {
      const uint32_t j = l;
      const uint32_t p = ldg(row + L.key_col[j]);
      const uint64_t b = ldg(L.toff[j] + p);
      const uint32_t o = j < dj ? j : j - 1;  // other lists, in order, without the driver
      if (j != dj) {
        oaddr[w][o] = list_addr<OOC>(L, j, p, b);
        olen[w][o] = (uint32_t)(ldg(L.toff[j] + p + 1) - b);
      }
    }
    if (l < ndup) dpos[w][l] = vposition_in(L.bm_new, L.rank_new, ldg(L.dup_can[l] + ldg(row + L.dup_col[l])));
    const uint32_t ko = FINAL ? 1 : L.kout;
    uint32_t newc = ko;  // the output column that takes the value (ko: none does)
    if (!FINAL) {
      const uint32_t c = l < ko ? L.src[l] : 0;
      const uint64_t isnew = __ballot(l < ko && c == COL_NEW);
      if (isnew) newc = (uint32_t)__builtin_ctzll(isnew);
      if (l < ko && c != COL_NEW) prow[w][l] = ldg(row + c);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const uint64_t s0 = (uint64_t)(wt - e.piece0) * chunk;
    const uint64_t s1 = s0 + chunk < dlen ? s0 + chunk : dlen;
    walked += s1 - s0;
    uint64_t survivors = 0;
    uint32_t pend = 0;  // surviving values staged, not yet written
    // With no other list the piece's rows are known before it is walked, all
    // entries but the equal-label columns' (as in k_vext): one reservation.
    uint64_t cursor = 0;
    const bool counted = !FINAL && nb == 1;
    if (counted) {
      const bool gone = l < ndup && dpos[w][l] != NOT_FOUND && sorted_contains(dlist + s0, s1 - s0, dpos[w][l]);
      const uint64_t n = s1 - s0 - __popcll(__ballot(gone));
      if (l == 0) cursor = atomicAdd(it.counter, (unsigned long long)n);
      cursor = readlane_u64(cursor, 0);
    }
    // the staged rows share the parent row: pend * ko consecutive words
    // of the output, reserved by one atomic, written by consecutive lanes
    auto flush = [&]() {
      uint64_t base = cursor;
      cursor += pend;
      if (!counted) {
        if (l == 0) base = atomicAdd(it.counter, (unsigned long long)pend);
        base = readlane_u64(base, 0);
      }
      const uint32_t inv = 0xFFFFFFFFu / ko + 1;
      written += (uint64_t)pend * 4 * ko;
      for (uint32_t q = l; q < pend * ko; q += 64) {
        const uint32_t i = ko > 1 ? __umulhi(q, inv) : q, c = q - i * ko;
        if (base + i < it.out_cap) stg(it.out + (base + i) * ko + c, c != newc ? prow[w][c] : hsv[w][i]);
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      pend = 0;
    };
    // Two items per lane per step, as in k_vext.  The first other list is
    // probed through windows: for each 128-entry step of the chunk, the range
    // of that list that can hold the step's values (both lists are sorted and
    // duplicate-free) is found for up to 63 steps at once (lane j: the end of
    // step j, lane 63: the start of the first step), and a window of at most
    // HWIN entries is staged in LDS with coalesced loads and searched there.
    const uint32_t *l0p = nb > 1 ? reinterpret_cast<const uint32_t *>(oaddr[w][0]) : nullptr;
    const uint32_t l0n = nb > 1 ? olen[w][0] : 0;
    for (uint64_t S = s0; S < s1; S += 63 * 128) {
      const uint64_t S1 = S + 63 * 128 < s1 ? S + 63 * 128 : s1;
      const uint32_t nsub = (uint32_t)((S1 - S + 127) / 128);
      if (nb > 1) {
        uint32_t pos = 0;
        if (l < nsub) {
          const uint64_t last = (S + 128ull * (l + 1) < S1 ? S + 128ull * (l + 1) : S1) - 1;
          pos = upper_bound_u32(l0p, l0n, ldg(dlist + last));
        } else if (l == 63) {
          pos = lower_bound_u32(l0p, l0n, ldg(dlist + S));
        }
        wend[w][l] = pos;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      }
      for (uint32_t j = 0; j < nsub; ++j) {
        const uint64_t s = S + 128ull * j;
        bool keep0 = s + l < S1, keep1 = s + 64 + l < S1;
        uint32_t val0 = 0, val1 = 0;
        if (keep0) val0 = ldg(dlist + s + l);
        if (keep1) val1 = ldg(dlist + s + 64 + l);
        for (uint32_t c = 0; c < ndup; ++c) {
          if (dpos[w][c] == val0) keep0 = false;
          if (dpos[w][c] == val1) keep1 = false;
        }
        if (nb > 1) {
          const uint32_t a = __builtin_amdgcn_readfirstlane(j ? wend[w][j - 1] : wend[w][63]);
          const uint32_t wn = __builtin_amdgcn_readfirstlane(wend[w][j]) - a;
          if (wn <= HWIN) {
            for (uint32_t i = l; i < wn; i += 64) win[w][i] = ldg(l0p + a + i);
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            contains_pair<false>(win[w], wn, val0, keep0, val1, keep1);
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
          } else {
            contains_pair(l0p + a, wn, val0, keep0, val1, keep1);
          }
        }
        for (uint32_t o = 1; o + 1 < nb; ++o) {
          const uint32_t *a = reinterpret_cast<const uint32_t *>(oaddr[w][o]);
          contains_pair(a, __builtin_amdgcn_readfirstlane(olen[w][o]), val0, keep0, val1, keep1);
        }
        const uint64_t m0 = __ballot(keep0), m1 = __ballot(keep1);
        const uint32_t nk0 = (uint32_t)__popcll(m0), nk = nk0 + (uint32_t)__popcll(m1);
        if (FINAL) {
          survivors += nk;
        } else if (nk) {
          if (keep0) hsv[w][pend + rank_below(m0)] = val0;
          if (keep1) hsv[w][pend + nk0 + rank_below(m1)] = val1;
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
          pend += nk;
          if (pend > VSTAGE - 128) flush();
        }
      }
      // wend of this wave is rewritten by the next group of steps
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    if (!FINAL && pend) flush();
    if (FINAL && l == 0 && survivors) atomicAdd(it.counter, (unsigned long long)survivors);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (prof_items && l == 0 && walked) atomicAdd(prof_items, (unsigned long long)walked);
  if (prof_out && l == 0 && written) atomicAdd(prof_out, (unsigned long long)written);
}

// Last level, one backward list: |list| - equal-label columns present.  A
// block takes runs of 256-row tasks and keeps its count while they belong to
// one item, so an item's counter sees one atomic per block and item change
// (with one per 256 rows, and one for the work queue, two atomics bounded the
// kernel: 6.4 ms for the 280,000 tasks of a 7 * 10^7-row level).
template <bool OOC>
__global__ void __launch_bounds__(VB) k_vcount1(const VItem *__restrict__ items, const uint32_t *__restrict__ nitems_p,
                                               const uint64_t *__restrict__ blk_prefix,
                                               unsigned int *__restrict__ queue, uint64_t g_begin, uint64_t g_end) {
  const uint32_t nitems = *nitems_p;
  const uint64_t total = blk_prefix[nitems] < g_end ? blk_prefix[nitems] : g_end;
  if (g_begin >= total) return;
  __shared__ uint64_t sm[VW], next_run;
  uint32_t t = NOT_FOUND;  // item in hand
  VItem it{};
  uint64_t cnt = 0;  // this thread's part of the item's count
  auto flush = [&]() {
    const uint64_t c = wave_sum_u64(cnt);
    cnt = 0;
    if (threadIdx.x % 64 == 0) sm[threadIdx.x / 64] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint64_t s = sm[0] + sm[1] + sm[2] + sm[3];
      if (s) atomicAdd(it.counter, (unsigned long long)s);
    }
    __syncthreads();
  };
  Runs runs(total - g_begin, blockIdx.x, gridDim.x, MAX_RUN, queue);
  while (runs.valid()) {
    for (uint64_t g = g_begin + runs.begin(), ge = g_begin + runs.end(); g < ge; ++g) {
      if (t == NOT_FOUND || g < blk_prefix[t] || g >= blk_prefix[t + 1]) {
        if (t != NOT_FOUND) flush();
        t = find_item(blk_prefix, nitems, g);
        it = items[t];
      }
      CLevel &L = *(CLevel *)it.lv;
      const uint64_t r = it.row_begin + (g - blk_prefix[t]) * VB + threadIdx.x;
      if (r >= it.row_end) continue;
      const uint32_t *row = it.rows + r * it.k;
      const uint32_t p = ldg(row + L.key_col[0]);
      const uint64_t b = ldg(L.toff[0] + p), e = ldg(L.toff[0] + p + 1);
      cnt += e - b;
      const uint32_t *lst = nullptr;
      if (L.ndup) lst = reinterpret_cast<const uint32_t *>(list_addr<OOC>(L, 0, p, b));
      for (uint32_t c = 0; c < L.ndup; ++c) {
        const uint32_t pos = vposition_in(L.bm_new, L.rank_new, ldg(L.dup_can[c] + ldg(row + L.dup_col[c])));
        if (pos != NOT_FOUND && sorted_contains(lst, e - b, pos)) --cnt;
      }
    }
    // the block's first wave asks for the next run
    if (threadIdx.x < 64) {
      runs.next();
      if (threadIdx.x == 0) next_run = runs.run;
    }
    __syncthreads();
    runs.run = next_run;
    __syncthreads();
  }
  if (t != NOT_FOUND) flush();
}

// Streamed tables: for every table block a row of the launch will read, the
// first and last task (launch task + base) that reads it.  Blocks (256-row
// tasks) are strided over the grid.
// Only the launch's tasks g with base + g in [wa, wb) are marked, as
// base + g - wa (the iteration is planned one window of tasks at a time).
__global__ void __launch_bounds__(VB) k_vmark(const VItem *__restrict__ items, uint32_t nitems,
                                             const uint64_t *__restrict__ blk_prefix, uint64_t base, uint64_t wa,
                                             uint64_t wb, bool count_only, uint32_t *__restrict__ first,
                                             uint32_t *__restrict__ last) {
  const uint64_t total = blk_prefix[nitems];
  const uint64_t g0 = wa > base ? wa - base : 0;
  const uint64_t g1 = wb - base < total ? wb - base : total;
  for (uint64_t g = g0 + blockIdx.x; g < g1; g += gridDim.x) {
    const uint32_t t = find_item(blk_prefix, nitems, g);
    const VItem it = items[t];
    CLevel &L = *(CLevel *)it.lv;
    const uint64_t r = it.row_begin + (g - blk_prefix[t]) * VB + threadIdx.x;
    // k_vcount1 reads list values only to remove equal-label columns
    if (count_only && L.ndup == 0) continue;
    const bool valid = r < it.row_end;
    const uint32_t *row = it.rows + r * it.k;
    const uint32_t gt = (uint32_t)(base + g - wa);
    for (uint32_t j = 0; j < L.nb; ++j) {
      const uint32_t b = valid ? L.gblk[j] + (ldg(row + L.key_col[j]) >> L.kshift[j]) : 0;
      // one lane per distinct block of the wave's rows marks it (rows of one
      // parent mostly share theirs), and only where the mark moves
      uint64_t rest = __ballot(valid);
      bool lead = false;
      while (rest) {
        const uint32_t x = (uint32_t)__builtin_ctzll(rest);
        const uint64_t same = __ballot(valid && b == readlane_u32(b, x));
        if (threadIdx.x % 64 == x) lead = true;
        rest &= ~same;
      }
      if (lead) {
        if (__hip_atomic_load(&first[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > gt) atomicMin(&first[b], gt);
        if (__hip_atomic_load(&last[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < gt) atomicMax(&last[b], gt);
      }
    }
  }
}

__global__ void k_viota(uint32_t *p, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = (uint32_t)i;
}

// ================================================================== host

void build_vlevels(VQueryState &S) {
  const QueryDev &Qd = *S.qd;
  const gemh::VertexPlan &P = S.plan;
  const uint32_t nv = Qd.Q.nv;
  std::vector<VLevel> lv(nv);
  std::vector<std::vector<uint32_t>> live;
  gemh::live_columns(P, &live);
  S.cols_in.assign(nv, 1);
  for (uint32_t i = 1; i < nv; ++i) S.cols_in[i] = (uint32_t)live[i].size();
  for (uint32_t i = 1; i < nv; ++i) {
    const gemh::VLevelPlan &lp = P.levels[i];
    VLevel &L = lv[i];
    L.nb = lp.nb;
    L.ndup = lp.ndup;
    const std::vector<uint32_t> &in = live[i];
    auto at = [&](uint32_t col) { return (uint32_t)(std::lower_bound(in.begin(), in.end(), col) - in.begin()); };
    for (uint32_t j = 0; j < lp.nb; ++j) {
      const TableDev &T = Qd.tab[lp.directed[j]];
      if (!T.present) throw Error{GEM_E_STATE, "vertex plan uses a table that was not built"};
      L.key_col[j] = at(lp.key_col[j]);
      L.toff[j] = T.off.as<uint64_t>();
      L.tval[j] = T.val.as<uint32_t>();
    }
    const uint32_t u = P.vorder[i];
    for (uint32_t d = 0; d < lp.ndup; ++d) {
      L.dup_col[d] = at(lp.dup_col[d]);
      L.dup_can[d] = Qd.can.as<uint32_t>() + Qd.can_off[P.vorder[lp.dup_col[d]]];
    }
    if (i + 1 < nv) {
      L.kout = (uint32_t)live[i + 1].size();
      for (uint32_t x = 0; x < L.kout; ++x) L.src[x] = live[i + 1][x] == i ? COL_NEW : at(live[i + 1][x]);
    }
    L.can_new = Qd.can.as<uint32_t>() + Qd.can_off[u];
    L.bm_new = Qd.bitmap.as<uint64_t>() + (uint64_t)u * Qd.W;
    L.rank_new = Qd.rank.as<uint32_t>() + (uint64_t)u * (Qd.W + 1);
  }
  S.max_nb.assign(nv, 0);
  S.max_ndup.assign(nv, 0);
  for (uint32_t i = 1; i < nv; ++i) {
    S.max_nb[i] = lv[i].nb;
    S.max_ndup[i] = lv[i].ndup;
  }
  S.hlv = std::move(lv);
  S.dlev = nullptr;
}

void put_levels(gem_ctx *c, VQueryState &S) {
  if (S.dlev) return;
  S.levels.alloc(sizeof(VLevel) * S.hlv.size(), c->stream);
  GEM_HIP_CHECK(
      hipMemcpyAsync(S.levels.p, S.hlv.data(), sizeof(VLevel) * S.hlv.size(), hipMemcpyHostToDevice, c->stream));
  S.dlev = S.levels.as<VLevel>();
}

// The level tables of the states that a run starts with, in one buffer and one
// copy (a copy takes 8 us of the stream whatever its size: 20 queries' took
// a twelfth of their batch).
struct RunLevels {
  std::vector<VQueryState *> in;
  std::vector<VLevel> host;
  DevBuf dev;
  RunLevels(gem_ctx *c, const std::vector<VQueryState *> &qs) {
    for (VQueryState *S : qs)
      if (!S->pending && !S->dlev && !S->hlv.empty()) {
        in.push_back(S);
        host.insert(host.end(), S->hlv.begin(), S->hlv.end());
      }
    if (in.empty()) return;
    dev.alloc(sizeof(VLevel) * host.size(), c->stream);
    GEM_HIP_CHECK(hipMemcpyAsync(dev.p, host.data(), sizeof(VLevel) * host.size(), hipMemcpyHostToDevice, c->stream));
    const VLevel *at = dev.as<VLevel>();
    for (VQueryState *S : in) {
      S->dlev = at;
      at += S->hlv.size();
    }
  }
  ~RunLevels() {
    for (VQueryState *S : in)
      if (S->dlev >= dev.as<VLevel>() && S->dlev < dev.as<VLevel>() + host.size()) S->dlev = nullptr;
  }
};

void replan(VQueryState &S, const std::vector<uint32_t> &vorder) {
  if (gemh::make_vertex_plan(S.Qp ? *S.Qp : S.qd->Q, vorder, &S.plan))
    throw Error{GEM_E_INVALID, "invalid vertex order (leaf first, or a vertex without an earlier neighbour)"};
  if (S.edge_map)
    for (size_t l = 1; l < S.plan.levels.size(); ++l) {
      gemh::VLevelPlan &lp = S.plan.levels[l];
      for (uint32_t j = 0; j < lp.nb; ++j)
        lp.directed[j] = 2 * (*S.edge_map)[lp.directed[j] >> 1] + (lp.directed[j] & 1);
    }
  build_vlevels(S);
  S.mnb_all = std::max(S.mnb_all, *std::max_element(S.max_nb.begin(), S.max_nb.end()));
  S.mnd_all = std::max(S.mnd_all, *std::max_element(S.max_ndup.begin(), S.max_ndup.end()));
}

uint64_t attempt_limit(const VQueryState &S, uint32_t a) {
  if (!S.first_attempt || S.ranked.size() < 2) return 0;
  if (S.max_attempts && a + 1 >= S.max_attempts) return 0;
  const uint32_t rounds = a / std::max<uint32_t>(S.width, 1);
  const double lim = (double)S.first_attempt * std::pow((double)std::max<uint32_t>(S.growth, 2), (double)rounds);
  if (lim >= 9.0e18) return 0;  // beyond 2^63: no limit
  return (uint64_t)lim;
}

// (Re)start a query's attempt: the identity level of its first vertex's
// candidates, no count yet.  Its rows are the first of `identity`, which grows
// to the longest such level.
static void seed_query(gem_ctx *c, VQueryState &V, std::shared_ptr<DevBuf> &identity) {
  hipStream_t s = c->stream;
  put_levels(c, V);
  gemh::SQuery<LevelBuf> &Q = V.s;
  Q.nb = V.max_nb;
  Q.width = V.cols_in;
  Q.count = 0;
  Q.fin_bound = Q.fin_got = 0;
  Q.stack.clear();
  Q.level_rows.assign(Q.nv, 0);
  const uint64_t n0 = V.qd->ncan[V.plan.vorder[0]];
  Q.level_rows[0] = n0;
  if (n0 == 0) {
    Q.done = true;
    return;
  }
  if (!identity || identity->bytes < n0 * 4) {
    const uint64_t n = std::max<uint64_t>({n0, identity ? identity->bytes / 2 : 0, 1 << 16});
    identity = std::make_shared<DevBuf>();
    identity->alloc(n * 4, s);
    k_viota<<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(identity->as<uint32_t>(), n);
    GEM_LAUNCH_CHECK("k_viota");
  }
  auto buf = std::make_shared<LevelBuf>();
  buf->shared = identity;
  buf->p = identity->p;
  buf->bytes = n0 * 4;
  gemh::SLevel<LevelBuf> L;
  L.level = 1;
  L.rows = std::move(buf);
  L.nrows = n0;
  L.k = 1;
  Q.stack.push_back(std::move(L));
}

namespace {

struct Launch {
  std::vector<VItem> items;
  std::vector<uint64_t> blk;  // prefix, items.size() + 1
  uint32_t max_nb = 1, max_ndup = 0;
  // tasks: 256-row blocks unless given
  void add(const VItem &it, uint32_t nb, uint32_t ndup, uint64_t tasks = 0) {
    if (blk.empty()) blk.push_back(0);
    items.push_back(it);
    blk.push_back(blk.back() + (tasks ? tasks : (it.row_end - it.row_begin + VB - 1) / VB));
    max_nb = std::max(max_nb, nb);
    max_ndup = std::max(max_ndup, ndup);
  }
  bool empty() const { return items.empty(); }
};

// Units of a level that a capped run measures at first (see SchedConfig): of
// the levels of 16 queries of up to 24 vertices under a cap of 1e9 (2^20 R-MAT),
// 27 times as many units were measured as walked, half the pass.
constexpr uint64_t MEASURE_UNITS = 4096;

// persistent grid: enough blocks to fill the chip (tunable cap), never more
// than the tasks
uint32_t g_persistent_blocks = 2048;
uint32_t grid_for(uint64_t blocks) {
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(blocks, g_persistent_blocks));
}

// Blocks of VB threads of a kernel that the device runs at once: a persistent
// grid has no use for more (the later ones would start when the work is done,
// and make the runs of the others shorter).
uint32_t resident_blocks(const void *kernel, size_t lds) {
  int per_cu = 0, dev = 0, cus = 0;
  GEM_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, VB, lds));
  GEM_HIP_CHECK(hipGetDevice(&dev));
  GEM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return (uint32_t)std::max(1, per_cu * cus);
}

// Fixed buffers for the extend step of every iteration of one run: item
// tables and block prefixes of the three launches (write, final walk, final
// single-list count), the heavy-row lists of the two walking launches, and a
// header with the item counts, work queues, heavy-row counts, walked-entry
// counts and per-task result counters.  Host side: pinned mirrors.  Because
// every pointer, grid and LDS size is fixed for the run, the step
//   H2D header, prefixes, items -> 3 kernels -> 2 heavy walks
//   -> D2H header
// is captured once as a hipGraph and replayed each iteration (no memset node:
// the zeroed counters travel in the header copy).
struct ExtSlot {
  static constexpr size_t KEEP_LAUNCH = 1 << 20;
  // header: item counts [3], heavy rows and pieces [2], profile counters [6] (u64:
  // entries walked by the write / final / heavy write / heavy final kernels,
  // bytes written by the write / heavy write kernels), queues [3 main + 2
  // heavy] of WQ_WORDS words, result counters [cap] (u64, a cache line each:
  // the waves of one launch add to several of them at once)
  static constexpr size_t HDR_NITEMS = 0, HDR_HEAVYN = 16, HDR_PITEMS = 64, HDR_QUEUE = 128,
                          HDR_CTR = HDR_QUEUE + 5 * 4 * WQ_WORDS, CTR_STRIDE = 8;
  uint32_t cap = 0;  // items per launch = counters
  // one block, on both sides: header, block prefixes [3][cap + 1] and items
  // [3][cap] of a step, copied at once (in seven copies they took the stream 60
  // us), then those of a length pass
  DevBuf block;
  unsigned char *host = nullptr;
  size_t step_bytes = 0, len_bytes = 0;
  bool own_host = false, in_flight = false;
  hipStream_t stream = nullptr;
  const VItem *items[4] = {};
  const uint64_t *blk[4] = {};
  DevBuf heavy[2], pieces[2];  // heavy rows and the rows of their pieces, per walking launch
  VItem *h_items[4] = {};
  uint64_t *h_blk[4] = {};
  unsigned char *h_hdr = nullptr;
  size_t hdr_bytes = 0;
  uint32_t max_nb = 1, max_ndup = 0;
  uint32_t lcap = 0, dcap = 0;  // lists and equal-label columns k_vext keeps in LDS
  size_t lds = 0;
  uint32_t grid[5] = {};  // write walk, final walk, final count, heavy write, heavy final
  uint32_t heavy_t = 1024, heavy_chunk = 1024;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;

  void init(gem_ctx *c, uint32_t capacity, uint32_t mnb, uint32_t mnd) {
    hipStream_t s = c->stream;
    cap = std::max<uint32_t>(capacity, 1);
    max_nb = std::max<uint32_t>(mnb, 1);
    max_ndup = mnd;
    lcap = max_nb > 1 ? std::min(max_nb, LDS_LISTS) : 0;
    dcap = std::min(max_ndup, LDS_DUPS);
    lds = (size_t)VW * 64 * (lcap * 12 + dcap * 4);
    const void *kernels[5] = {(const void *)&k_vext<false, false>, (const void *)&k_vext<true, false>,
                              (const void *)&k_vcount1<false>, (const void *)&k_vext_heavy<false, false>,
                              (const void *)&k_vext_heavy<true, false>};
    for (int i = 0; i < 5; ++i)
      grid[i] = std::min(g_persistent_blocks, resident_blocks(kernels[i], i < 2 ? lds : 0));
    heavy_t = c->heavy_t;
    heavy_chunk = c->heavy_chunk;
    hdr_bytes = HDR_CTR + 8ull * CTR_STRIDE * cap;
    for (int i = 0; i < 2; ++i) {
      heavy[i].alloc(sizeof(HeavyRow) * gemh::HEAVY_CAP, s);
      pieces[i].alloc(4ull * gemh::PIECE_CAP, s);
    }
    const size_t blk_bytes = 8ull * (cap + 1), item_bytes = sizeof(VItem) * cap;
    len_bytes = blk_bytes + item_bytes;
    step_bytes = hdr_bytes + 3 * len_bytes;
    const size_t bytes = step_bytes + len_bytes;
    block.alloc(bytes, s);
    stream = s;
    if (bytes > c->launch_host_bytes) {
      void *p = nullptr;
      const size_t n = std::max<size_t>(bytes, KEEP_LAUNCH / 4);
      GEM_HIP_CHECK(hipHostMalloc(&p, n, hipHostMallocDefault));
      if (bytes > KEEP_LAUNCH) {
        own_host = true;
      } else {
        if (c->launch_host) (void)hipHostFree(c->launch_host);
        c->launch_host = p;
        c->launch_host_bytes = n;
      }
      host = static_cast<unsigned char *>(p);
    } else {
      host = static_cast<unsigned char *>(c->launch_host);
    }
    std::memset(host, 0, bytes);
    h_hdr = host;
    for (int i = 0; i < 4; ++i) {
      const size_t at = i < 3 ? hdr_bytes + i * blk_bytes : step_bytes;
      const size_t it = i < 3 ? hdr_bytes + 3 * blk_bytes + i * item_bytes : step_bytes + blk_bytes;
      h_blk[i] = reinterpret_cast<uint64_t *>(host + at);
      blk[i] = reinterpret_cast<const uint64_t *>(block.as<unsigned char>() + at);
      h_items[i] = reinterpret_cast<VItem *>(host + it);
      items[i] = reinterpret_cast<const VItem *>(block.as<unsigned char>() + it);
    }
  }
  // A launch's items and block prefix to the host side of the block.
  void fill(int i, const Launch &L) {
    if (L.items.size() > cap) throw Error{GEM_E_STATE, "more vjoin items than launch slots"};
    std::copy(L.items.begin(), L.items.end(), h_items[i]);
    std::copy(L.blk.begin(), L.blk.end(), h_blk[i]);
    if (L.blk.empty()) h_blk[i][0] = 0;
  }
  void copy_length_launch() {
    GEM_HIP_CHECK(hipMemcpyAsync(block.as<unsigned char>() + step_bytes, host + step_bytes, len_bytes,
                                 hipMemcpyHostToDevice, stream));
    in_flight = true;
  }
  // Waits for everything enqueued so far; the host side may then be filled anew.
  void wait() {
    GEM_HIP_CHECK(hipStreamSynchronize(stream));
    in_flight = false;
  }
  ~ExtSlot() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (in_flight) (void)hipStreamSynchronize(stream);  // an error cut the run short
    if (own_host) (void)hipHostFree(host);
  }
  uint32_t *nitems(int i) { return reinterpret_cast<uint32_t *>(h_hdr + HDR_NITEMS) + i; }
  uint64_t counter(size_t i) { return reinterpret_cast<uint64_t *>(h_hdr + HDR_CTR)[i * CTR_STRIDE]; }
  uint64_t *pitems() { return reinterpret_cast<uint64_t *>(h_hdr + HDR_PITEMS); }
  unsigned long long *dev_counter(size_t i) {
    return reinterpret_cast<unsigned long long *>(block.as<unsigned char>() + HDR_CTR) + i * CTR_STRIDE;
  }

  // The step's work, enqueued on the stream (eagerly or under capture).
  void enqueue(gem_ctx *c, bool captured, bool prof_kernels, bool count_items) {
    hipStream_t s = c->stream;
    unsigned char *d = block.as<unsigned char>();
    GEM_HIP_CHECK(hipMemcpyAsync(d, host, step_bytes, hipMemcpyHostToDevice, s));
    const uint32_t *dn = reinterpret_cast<const uint32_t *>(d + HDR_NITEMS);
    unsigned int *dq = reinterpret_cast<unsigned int *>(d + HDR_QUEUE);
    auto *hn = reinterpret_cast<gemh::HeavyCounters *>(d + HDR_HEAVYN);
    // a captured step holds every kernel (one without items ends at once);
    // an eager one launches those that have items
    uint64_t e[3];
    for (int i = 0; i < 3; ++i) e[i] = captured || *nitems(i) ? ~0ull : 0;
    launch_kernels<false>(c, ~0u, dn, dq, dq + 3 * WQ_WORDS, hn, prof_kernels, count_items, 0, e[0], 0, e[1], 0, e[2]);
    GEM_HIP_CHECK(hipMemcpyAsync(h_hdr, d, hdr_bytes, hipMemcpyDeviceToHost, s));
  }

  // A walk in runs of equal cost cuts its units between rows, so a row is long
  // for it from twice the threshold on (write walks and their heavy rows in a
  // capped batch, at 1024, 2048 and 4096: 70, 66 and 75 ms on 2^20 vertices, 82, 79
  // and 76 on 2^22).  Streamed walks take whole units: 2048 cost a streamed batch
  // 20%.
  HeavyOut heavy_out(int i, gemh::HeavyCounters *hn) const {
    return HeavyOut{heavy[i].as<HeavyRow>(), pieces[i].as<uint32_t>(), hn + i, heavy_t, heavy_chunk};
  }

  // The three kernels over task ranges [b_i, e_i) of launch i (queues dq,
  // WQ_WORDS words each), then the heavy rows the two walking launches set
  // aside (queues hq, rows and pieces hn[0..1]; everything starts at zero), in
  // at most `most` blocks each.
  template <bool OOC>
  void launch_kernels(gem_ctx *c, uint32_t most, const uint32_t *dn, unsigned int *dq, unsigned int *hq,
                      gemh::HeavyCounters *hn, bool prof_kernels, bool count_items, uint64_t b0, uint64_t e0, uint64_t b1,
                      uint64_t e1, uint64_t b2, uint64_t e2) {
    hipStream_t s = c->stream;
    unsigned long long *dp = reinterpret_cast<unsigned long long *>(block.as<unsigned char>() + HDR_PITEMS);
    if (b0 < e0) {
      ProfLaunch pl(c, prof_kernels ? K_VEXT_WRITE : -1);
      k_vext<false, OOC><<<std::min(most, grid[0]), VB, lds, s>>>(items[0], dn + 0, blk[0], dq + 0, lcap, dcap,
                                               count_items ? dp : nullptr, count_items ? dp + 4 : nullptr,
                                               b0, e0, heavy_out(0, hn));
      GEM_LAUNCH_CHECK("k_vext<write>");
    }
    if (b1 < e1) {
      ProfLaunch pl(c, prof_kernels ? K_VEXT_FINAL : -1);
      k_vext<true, OOC><<<std::min(most, grid[1]), VB, lds, s>>>(items[1], dn + 1, blk[1], dq + WQ_WORDS, lcap, dcap,
                                              count_items ? dp + 1 : nullptr, nullptr, b1, e1,
                                              heavy_out(1, hn));
      GEM_LAUNCH_CHECK("k_vext<final>");
    }
    if (b2 < e2) {
      ProfLaunch pl(c, prof_kernels ? K_VCOUNT1 : -1);
      k_vcount1<OOC><<<std::min(most, grid[2]), VB, 0, s>>>(items[2], dn + 2, blk[2], dq + 2 * WQ_WORDS, b2, e2);
      GEM_LAUNCH_CHECK("k_vcount1");
    }
    if (b0 < e0) {
      ProfLaunch pl(c, prof_kernels ? K_VEXT_HEAVY_WRITE : -1);
      k_vext_heavy<false, OOC><<<std::min(most, grid[3]), VB, 0, s>>>(items[0], heavy_out(0, hn), hq + 0,
                                                                      count_items ? dp + 2 : nullptr,
                                                                      count_items ? dp + 5 : nullptr);
      GEM_LAUNCH_CHECK("k_vext_heavy<write>");
    }
    if (b1 < e1) {
      ProfLaunch pl(c, prof_kernels ? K_VEXT_HEAVY_FINAL : -1);
      k_vext_heavy<true, OOC><<<std::min(most, grid[4]), VB, 0, s>>>(items[1], heavy_out(1, hn),
                                                                     hq + WQ_WORDS, count_items ? dp + 3 : nullptr,
                                                                     nullptr);
      GEM_LAUNCH_CHECK("k_vext_heavy<final>");
    }
  }

  // Streamed tables: the same step, its tasks cut into groups whose table
  // blocks are copied in while the previous group runs (eager launches only).
  void launch_streamed(gem_ctx *c, TableCache &tc) {
    hipStream_t s = c->stream;
    in_flight = true;
    unsigned char *d = block.as<unsigned char>();
    GEM_HIP_CHECK(hipMemcpyAsync(d, host, step_bytes, hipMemcpyHostToDevice, s));
    uint64_t T[3], base[3];
    uint64_t total = 0;
    for (int i = 0; i < 3; ++i) {
      T[i] = *nitems(i) ? h_blk[i][*nitems(i)] : 0;
      base[i] = total;
      total += T[i];
    }
    if (total >= 0xFFFFFFFFull) throw Error{GEM_E_LIMIT, "too many tasks in one streamed iteration"};
    // The iteration is planned in windows of tasks: a block's marks span its
    // first to last use inside the window, so a window whose blocks cannot
    // all be placed is halved (down to one task) and planned again.
    const uint32_t *dn = reinterpret_cast<const uint32_t *>(d + HDR_NITEMS);
    const bool prof = c->prof.on;
    uint64_t wa = 0, W = total;
    while (wa < total) {
      const uint64_t wb = std::min(total, wa + W);
      tc.reset_marks();
      for (int i = 0; i < 3; ++i) {
        if (!T[i] || base[i] + T[i] <= wa || base[i] >= wb) continue;
        const uint64_t lo = std::max(wa, base[i]), hi = std::min(wb, base[i] + T[i]);
        k_vmark<<<(uint32_t)std::min<uint64_t>(hi - lo, 4096), VB, 0, s>>>(
            items[i], *nitems(i), blk[i], base[i], wa, wb, i == 2, tc.d_first(),
            tc.d_last());
        GEM_LAUNCH_CHECK("k_vmark");
      }
      if (!tc.plan(wb - wa)) {
        if (W == 1)
          throw Error{GEM_E_LIMIT, "the table blocks read by one 256-row task do not fit the device cache"};
        W = std::max<uint64_t>(1, W / 2);
        continue;
      }
      const auto &G = tc.groups();
      unsigned int *q = tc.queues();
      for (size_t g = 0; g < G.size(); ++g) {
        tc.issue(g);
        uint64_t lo[3], hi[3];
        for (int i = 0; i < 3; ++i) {
          lo[i] = std::max(wa + G[g].a, base[i]);
          hi[i] = std::min(wa + G[g].b, base[i] + T[i]);
          if (lo[i] < hi[i]) {
            lo[i] -= base[i];
            hi[i] -= base[i];
          } else {
            lo[i] = hi[i] = 0;
          }
        }
        const uint64_t most = std::max(hi[0] - lo[0], std::max(hi[1] - lo[1], hi[2] - lo[2]));
        const uint32_t grd = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(~0u, most));
        // per group: 3 main queues, 2 heavy queues, heavy rows and pieces
        unsigned int *gq = q + (size_t)GROUP_WORDS * g;
        auto *hn = reinterpret_cast<gemh::HeavyCounters *>(gq + 5 * WQ_WORDS);
        launch_kernels<true>(c, grd, dn, gq, gq + 3 * WQ_WORDS, hn, prof, prof, lo[0], hi[0], lo[1], hi[1], lo[2],
                             hi[2]);
        tc.done(g);
      }
      wa = wb;
      W = std::min(total, 2 * W);
    }
    GEM_HIP_CHECK(hipMemcpyAsync(h_hdr, d, hdr_bytes, hipMemcpyDeviceToHost, s));
  }

  void launch(gem_ctx *c, bool use_graph) {
    in_flight = true;
    if (!use_graph) {
      enqueue(c, false, c->prof.on, c->prof.on);
      return;
    }
    if (!exec) {
      hipStream_t s = c->stream;
      GEM_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      try {
        enqueue(c, true, false, false);
      } catch (...) {
        hipGraph_t g = nullptr;
        (void)hipStreamEndCapture(s, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
      }
      GEM_HIP_CHECK(hipStreamEndCapture(s, &graph));
      GEM_HIP_CHECK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    }
    GEM_HIP_CHECK(hipGraphLaunch(exec, c->stream));
  }
};

}  // namespace

namespace {

// Device side of the scheduler (host/vsched.h): level buffers from the
// caching allocator, length passes, extend steps through the fixed launch
// buffers of the run (eager, captured as a hipGraph, or with streamed tables).
struct HipSchedBackend {
  using Buf = LevelBuf;
  using Item = gemh::SItem<LevelBuf>;
  gem_ctx *c;
  std::vector<VQueryState *> &qs;
  ExtSlot &slot;
  TableCache *tc;
  bool verbose;
  uint64_t cap_;
  LazyStates *lazy = nullptr;
  using clk = std::chrono::steady_clock;
  clk::time_point last_print = clk::now();
  double t_len = 0, t_ext = 0;
  uint64_t ext_tasks = 0;
  std::shared_ptr<DevBuf> identity;  // 0, 1, 2, ... (see seed_query)

  static uint64_t buf_bytes(const LevelBuf &b) { return b.bytes; }

  std::shared_ptr<LevelBuf> alloc(uint64_t bytes) {
    auto b = std::make_shared<LevelBuf>();
    b->alloc(bytes, c->stream);
    return b;
  }

  std::shared_ptr<LevelBuf> shrink(const std::shared_ptr<LevelBuf> &from, uint64_t bytes) {
    from->shrink(bytes);
    return from;
  }

  VItem vitem(const Item &x) const {
    VItem it{};
    it.lv = qs[x.q]->dlev + x.level;
    it.rows = x.rows->as<uint32_t>();
    it.row_begin = x.row_begin;
    it.row_end = x.row_end;
    it.k = x.k;
    return it;
  }

  void length_pass(const std::vector<Item> &items, std::vector<std::vector<uint64_t>> *prefix) {
    const auto t0 = clk::now();
    hipStream_t s = c->stream;
    Launch L;
    for (const Item &x : items) L.add(vitem(x), qs[x.q]->max_nb[x.level], qs[x.q]->max_ndup[x.level]);
    slot.fill(3, L);
    slot.copy_length_launch();
    const uint64_t nblk = L.blk.back(), nunit = nblk * VW;
    DevBuf bu;
    auto kept = std::make_shared<DevBuf>();  // the unit prefix, which the levels keep for their write walks
    DevBuf &bp = *kept;
    bu.alloc(nunit * 8, s);
    bp.alloc((nunit + 1) * 8, s);
    {
      ProfLaunch pl(c, K_VLEN);
      k_vlen<<<grid_for(nblk), VB, 0, s>>>(slot.items[3], (uint32_t)L.items.size(), slot.blk[3], bu.as<uint64_t>());
      GEM_LAUNCH_CHECK("k_vlen");
    }
    scan_u64(c, bu.as<uint64_t>(), bp.as<uint64_t>(), nunit);
    for (size_t t = 0; t < items.size(); ++t) {
      const uint64_t lo = items[t].row_begin / gemh::SCHED_UNIT;
      items[t].rows->units = LevelBuf::Units{kept, L.blk[t] * VW - lo, lo, lo + units_of(items[t])};
    }
    if (!prefix) return;
    uint64_t *pref = pinned<uint64_t>(c, nunit + 1);
    GEM_HIP_CHECK(hipMemcpyAsync(pref, bp.p, (nunit + 1) * 8, hipMemcpyDeviceToHost, s));
    slot.wait();
    prefix->resize(items.size());
    for (size_t t = 0; t < items.size(); ++t) {
      const Item &x = items[t];
      const uint64_t u0 = L.blk[t] * VW;
      const uint64_t nu = (x.row_end - x.row_begin + gemh::SCHED_UNIT - 1) / gemh::SCHED_UNIT;
      std::vector<uint64_t> &P = (*prefix)[t];
      P.resize(nu + 1);
      for (uint64_t i = 0; i <= nu; ++i) P[i] = pref[u0 + i] - pref[u0];
      // rows + one offset pair per backward list
      prof_bytes(c, K_VLEN, (double)(x.row_end - x.row_begin) * (4.0 * x.k + 16.0 * qs[x.q]->max_nb[x.level]));
    }
    t_len += std::chrono::duration<double>(clk::now() - t0).count();
  }

  static uint64_t units_of(const Item &x) {
    return (x.row_end - x.row_begin + gemh::SCHED_UNIT - 1) / gemh::SCHED_UNIT;
  }

  // Unit prefixes of chunks that the last measurement of their level does not
  // hold (the level came back from host memory without them).  Returns what
  // they replace, which extend puts back.
  std::vector<std::pair<const LevelBuf *, LevelBuf::Units>> remeasure(const std::vector<Item> &wr_items) {
    std::vector<Item> need;
    std::vector<std::pair<const LevelBuf *, LevelBuf::Units>> old;
    for (const Item &x : wr_items) {
      const uint64_t lo = x.row_begin / gemh::SCHED_UNIT;
      const LevelBuf::Units &u = x.rows->units;
      if (u.prefix && lo >= u.lo && lo + units_of(x) <= u.hi) continue;
      need.push_back(x);
      old.push_back({x.rows, u});
    }
    if (!need.empty()) length_pass(need, nullptr);
    return old;
  }

  // Runs of the walks over these items, CLAIMS per wave of the grid by cost (an
  // entry of a level with other lists costs its searches too); false: too many
  bool plan_runs(const std::vector<Item> &items, uint32_t grid, std::vector<uint32_t> *cost) const {
    std::vector<gemh::WalkPiece> pieces;
    for (const Item &x : items) pieces.push_back({x.out_rows, units_of(x), 4ull * qs[x.q]->max_nb[x.level] - 3});
    return gemh::plan_runs(pieces, (uint64_t)grid * VW, cost);
  }

  // Item x to a launch whose waves take runs of `run_cost` of it.
  void add_by_cost(Launch &L, VItem it, const Item &x, uint32_t run_cost) {
    it.units = x.rows->units.prefix->as<uint64_t>() + x.rows->units.unit0 + x.row_begin / gemh::SCHED_UNIT;
    it.nunits = (uint32_t)units_of(x);
    it.run_cost = run_cost;
    L.add(it, qs[x.q]->max_nb[x.level], qs[x.q]->max_ndup[x.level],
          gemh::WalkPiece{x.out_rows, units_of(x), 1}.runs(run_cost));
  }

  void extend(const std::vector<Item> &wr_items, const std::vector<Item> &fin_items, std::vector<uint64_t> *got_wr,
              std::vector<uint64_t> *got_fin) {
    const auto t0 = clk::now();
    // launch tables: write walks, final walks, final single-list counts; one
    // u64 result counter per item, in the device header
    Launch wr, fin, fin1;
    std::vector<std::pair<int, size_t>> fin_at(fin_items.size());
    size_t nctr = 0;
    // counters / work queues / walked-entry counts travel zeroed in the copy
    std::memset(slot.h_hdr + ExtSlot::HDR_HEAVYN, 0, slot.hdr_bytes - ExtSlot::HDR_HEAVYN);
    // runs of the write walks (see unit_range), and of the final ones when all
    // their pieces are measured (they are under a cap) and the runs few enough
    std::vector<uint32_t> wr_cost, fin_cost;
    std::vector<std::pair<const LevelBuf *, LevelBuf::Units>> replaced;
    if (!tc) {
      std::vector<Item> walked;
      bool measured = true;
      for (const Item &x : fin_items)
        if (qs[x.q]->max_nb[x.level] > 1) {
          walked.push_back(x);
          measured = measured && x.out_rows;
        }
      if (!measured || !plan_runs(walked, slot.grid[1], &fin_cost)) walked.clear();
      if (!plan_runs(wr_items, slot.grid[0], &wr_cost))
        throw Error{GEM_E_LIMIT, "too many runs in one write walk"};
      walked.insert(walked.end(), wr_items.begin(), wr_items.end());
      replaced = remeasure(walked);
    }
    size_t nwr = 0, nfin = 0;
    for (const Item &x : wr_items) {
      VItem it = vitem(x);
      it.out = x.out->as<uint32_t>();
      it.out_cap = x.out_rows;
      it.counter = slot.dev_counter(nctr++);
      if (!tc)
        add_by_cost(wr, it, x, wr_cost[nwr++]);
      else
        wr.add(it, qs[x.q]->max_nb[x.level], qs[x.q]->max_ndup[x.level]);
    }
    std::vector<size_t> fin_ctr(fin_items.size());
    for (size_t t = 0; t < fin_items.size(); ++t) {
      const Item &x = fin_items[t];
      VItem it = vitem(x);
      fin_ctr[t] = nctr;
      it.counter = slot.dev_counter(nctr++);
      if (qs[x.q]->max_nb[x.level] == 1)
        fin1.add(it, 1, qs[x.q]->max_ndup[x.level]);
      else if (!fin_cost.empty())
        add_by_cost(fin, it, x, fin_cost[nfin++]);
      else
        fin.add(it, qs[x.q]->max_nb[x.level], qs[x.q]->max_ndup[x.level]);
    }
    if (nctr > slot.cap) throw Error{GEM_E_STATE, "more vjoin tasks than launch slots"};
    Launch *L3[3] = {&wr, &fin, &fin1};
    for (int i = 0; i < 3; ++i) {
      Launch &L = *L3[i];
      slot.fill(i, L);
      *slot.nitems(i) = (uint32_t)L.items.size();
      ext_tasks += L.blk.empty() ? 0 : L.blk.back();
    }
    const bool prof = c->prof.on;
    if (tc)
      slot.launch_streamed(c, *tc);
    else
      slot.launch(c, c->use_graph && !prof);
    slot.wait();
    if (tc) tc->finish();
    for (auto &r : replaced) r.first->units = r.second;
    got_wr->resize(wr_items.size());
    got_fin->resize(fin_items.size());
    for (size_t t = 0; t < wr_items.size(); ++t) {
      (*got_wr)[t] = slot.counter(t);
      if ((*got_wr)[t] > wr_items[t].out_rows) throw Error{GEM_E_STATE, "vjoin output exceeded its bound"};
    }
    for (size_t t = 0; t < fin_items.size(); ++t) (*got_fin)[t] = slot.counter(fin_ctr[t]);
    if (prof) {
      const uint64_t *pc = slot.pitems();
      // algorithmic bytes: rows read (4 B per column + an offset pair per
      // backward list), 4 B per list entry walked, output rows written
      auto rows_bytes = [&](const Launch &L) {
        double b = 0;
        for (const auto &it : L.items)
          b += (double)(it.row_end - it.row_begin) * (4.0 * it.k + 16.0 * (double)L.max_nb);
        return b;
      };
      // (the heavy-row kernels: the entries they walk and the rows they write)
      prof_bytes(c, K_VEXT_WRITE, rows_bytes(wr) + 4.0 * (double)pc[0] + (double)pc[4]);
      prof_bytes(c, K_VEXT_FINAL, rows_bytes(fin) + 4.0 * (double)pc[1]);
      prof_bytes(c, K_VCOUNT1, rows_bytes(fin1));
      prof_bytes(c, K_VEXT_HEAVY_WRITE, 4.0 * (double)pc[2] + (double)pc[5]);
      prof_bytes(c, K_VEXT_HEAVY_FINAL, 4.0 * (double)pc[3]);
    }
    prof_flush(c);
    t_ext += std::chrono::duration<double>(clk::now() - t0).count();
  }

  // Swapping: a level's rows to pinned host memory and back, both copies on
  // the context stream (the device buffer goes back to the pool at once: its
  // next user is ordered after the copy).  A host buffer is freed after the
  // stream has drained, so no copy still reads or writes it.
  std::shared_ptr<void> swap_out(const LevelBuf &b, uint64_t bytes) {
    void *h = nullptr;
    GEM_HIP_CHECK(hipHostMalloc(&h, std::max<uint64_t>(bytes, 1), hipHostMallocDefault));
    hipStream_t s = c->stream;
    std::shared_ptr<void> hp(h, [s](void *p) {
      (void)hipStreamSynchronize(s);
      (void)hipHostFree(p);
    });
    GEM_HIP_CHECK(hipMemcpyAsync(h, b.p, bytes, hipMemcpyDeviceToHost, s));
    return hp;
  }
  std::shared_ptr<LevelBuf> swap_in(const std::shared_ptr<void> &h, uint64_t bytes) {
    auto b = std::make_shared<LevelBuf>();
    b->alloc(bytes, c->stream);
    GEM_HIP_CHECK(hipMemcpyAsync(b->p, h.get(), bytes, hipMemcpyHostToDevice, c->stream));
    return b;
  }

  bool ready(uint32_t qi) {
    const VQueryState &V = *qs[qi];
    return !V.pending || V.twin || !lazy || lazy->ready(qi);
  }
  void wait_ready(uint32_t qi) {
    const VQueryState &V = *qs[qi];
    if (V.pending && !V.twin && lazy) lazy->complete(qi);
  }

  // A pending state is completed when it starts: a primary by its preparer
  // (ranked orders, plan), a twin from its partner (which started before it).
  // Returns false when there is nothing to run (a twin of a query with one
  // candidate order).
  bool complete(uint32_t qi) {
    VQueryState &V = *qs[qi];
    if (!V.pending) return true;
    if (V.twin) {
      const VQueryState &P = *qs[(size_t)V.s.partner];
      if (P.pending || P.ranked.size() < 2) return false;
      V.first_attempt = P.first_attempt;
      V.growth = P.growth;
      V.width = P.width;
      V.max_attempts = P.max_attempts;
      V.ranked = P.ranked;
      V.ranked_idx = P.ranked_idx;
      V.mnb_all = P.mnb_all;
      V.mnd_all = P.mnd_all;
    } else {
      if (!lazy) throw Error{GEM_E_STATE, "a pending query without a preparer"};
      lazy->complete(qi);
    }
    if (V.mnb_all > slot.max_nb || V.mnd_all > slot.max_ndup)
      throw Error{GEM_E_STATE, "a query needs more launch LDS than the run was sized for"};
    V.pending = false;
    return true;
  }

  void admit(uint32_t qi) {
    VQueryState &V = *qs[qi];
    if (!complete(qi)) {
      V.s.done = true;
      V.s.cancelled = true;
      return;
    }
    if (!V.twin) {
      // a primary completed now: its levels' list counts and first limit
      V.s.nb = V.max_nb;
      if (!V.s.attempts) V.s.attempt_limit = attempt_limit(V, 0);
    }
    if (V.twin && V.s.partner >= 0) {
      // a racing twin starts at its partner's current limit, on the order
      // after the one its partner runs
      const VQueryState &P = *qs[(size_t)V.s.partner];
      const uint32_t K = (uint32_t)V.ranked.size();
      const uint32_t a = P.s.attempts;
      V.shift = (P.cur + 1 + K - a % K) % K;
      V.cur = (a + V.shift) % K;
      replan(V, V.ranked[V.cur]);
      V.s.nb = V.max_nb;
      if (V.mnb_all > slot.max_nb || V.mnd_all > slot.max_ndup)
        throw Error{GEM_E_STATE, "racing order needs more launch LDS than the run was sized for"};
      V.s.attempts = a;
      V.s.attempt_start = V.s.work;
      V.s.attempt_limit = attempt_limit(V, a);
      if (verbose) {
        std::fprintf(stderr, "[vjoin] query %u races query %lld: order %u, limit %.3g\n", qi,
                     (long long)V.s.partner, V.ranked_idx[V.cur], (double)V.s.attempt_limit);
        std::fflush(stderr);
      }
    }
    seed_query(c, V, identity);
  }

  // The attempt of query qi went past its limit with its levels still
  // pending.  It goes on when it has counted at least a quarter of the cap and,
  // at the rate it counted so far, needs less work to pass the cap than 4/5 of
  // the next attempt's limit (a new attempt starts from nothing, and an
  // attempt whose cost is near its limit would otherwise end or restart by
  // chance: the order rows come out of a level in varies from run to run).
  // Its limit becomes what it has spent plus 1.5 times that estimate.
  bool prolong(uint32_t qi) {
    VQueryState &V = *qs[qi];
    gemh::SQuery<LevelBuf> &Q = V.s;
    if (!cap_ || Q.count < cap_ / 4 || Q.count == 0) return false;
    const uint64_t spent = Q.work - Q.attempt_start;
    const double need = (double)spent * ((double)(cap_ + 1) / (double)Q.count - 1.0);
    const uint64_t next = attempt_limit(V, Q.attempts + 1);
    if (next && need >= 0.8 * (double)next) return false;
    Q.attempt_limit = spent + (uint64_t)(1.5 * need) + 1;
    if (verbose) {
      std::fprintf(stderr, "[vjoin] query %u: attempt %u goes on (%.0f%% of the cap counted), limit %.3g\n", qi,
                   Q.attempts, 100.0 * (double)Q.count / (double)cap_, (double)Q.attempt_limit);
      std::fflush(stderr);
    }
    return true;
  }

  // The attempt of query qi went past its limit (its levels are dropped):
  // the next ranked order, with the next attempt's limit.
  bool restart(uint32_t qi) {
    VQueryState &V = *qs[qi];
    gemh::SQuery<LevelBuf> &Q = V.s;
    if (!attempt_limit(V, 0)) return false;
    const uint32_t a = Q.attempts + 1;
    if (V.max_attempts && a >= V.max_attempts) return false;
    // the ended attempt's progress: embeddings counted per unit of work
    const uint32_t K = (uint32_t)V.ranked.size();
    if (V.rate.size() != K) V.rate.assign(K, 0.0);
    const uint64_t spent = Q.work - Q.attempt_start;
    if (spent) V.rate[V.cur] = std::max(V.rate[V.cur], (double)Q.count / (double)spent);
    // every ranked order once, then the one that counted fastest (the ranking
    // again while none has counted anything)
    V.cur = (a + V.shift) % K;
    if (a >= K) {
      uint32_t best = 0;
      for (uint32_t j = 1; j < K; ++j)
        if (V.rate[j] > V.rate[best]) best = j;
      if (V.rate[best] > 0) V.cur = best;
    }
    replan(V, V.ranked[V.cur]);
    if (tc) tc->bind(V, qi);
    if (V.mnb_all > slot.max_nb || V.mnd_all > slot.max_ndup)
      throw Error{GEM_E_STATE, "restart order needs more launch LDS than the run was sized for"};
    Q.attempts = a;
    Q.attempt_start = Q.work;
    Q.attempt_limit = attempt_limit(V, a);
    seed_query(c, V, identity);
    if (verbose) {
      std::fprintf(stderr, "[vjoin] query %u: attempt %u with order %u, limit %.3g\n", qi, a, V.ranked_idx[V.cur],
                   (double)Q.attempt_limit);
      std::fflush(stderr);
    }
    return true;
  }

  // wall time and iterations by the number of queries active (tail: at most 4)
  clk::time_point last_iter = clk::now();
  size_t last_active = 0;
  double t_tail = 0, t_body = 0;
  uint64_t it_tail = 0, it_body = 0;

  void on_iteration(uint64_t iter, size_t active, uint64_t live, uint64_t budget) {
    const auto now = clk::now();
    if (last_active) {
      const double dt = std::chrono::duration<double>(now - last_iter).count();
      if (last_active <= 4) {
        t_tail += dt;
        ++it_tail;
      } else {
        t_body += dt;
        ++it_body;
      }
    }
    last_iter = now;
    last_active = active;
    if (!verbose || now - last_print < std::chrono::seconds(2)) return;
    last_print = clk::now();
    std::fprintf(stderr, "[vjoin] iteration %llu: %zu of %zu queries active, pending levels %.2f of %.2f GiB\n",
                 (unsigned long long)iter, active, qs.size(), live / 1073741824.0, budget / 1073741824.0);
    std::fflush(stderr);
  }
};

}  // namespace

void VBatchRunner::run(std::vector<VQueryState *> &qs) {
  g_persistent_blocks = c_->persistent_blocks;
  // the level budget: given, or a quarter of what the device could still
  // give the run's level buffers (free memory plus empty pool segments)
  uint64_t total_budget = budget_bytes_;
  if (!total_budget) {
    size_t free_b = 0, total_b = 0;
    GEM_HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    total_budget = std::max<uint64_t>((free_b + pool_reusable_bytes()) / 4, 1ull << 30);
  }
  total_budget = std::max<uint64_t>(total_budget, 1ull << 20);
  // fixed launch buffers for the run (at most one item per running query)
  ExtSlot slot;
  {
    uint32_t mnb = 1, mnd = 0;
    for (VQueryState *S : qs) {
      for (size_t i = 0; i < S->max_nb.size(); ++i) {
        mnb = std::max(mnb, S->max_nb[i]);
        mnd = std::max(mnd, S->max_ndup[i]);
      }
      // every order a restart may switch to
      if (attempt_limit(*S, 0)) {
        mnb = std::max(mnb, S->mnb_all);
        mnd = std::max(mnd, S->mnd_all);
      }
    }
    const size_t running = c_->max_active ? std::min<size_t>(qs.size(), c_->max_active) : qs.size();
    slot.init(c_, (uint32_t)running, mnb, mnd);
  }
  // streamed tables: a block cache shared by the run's queries
  std::unique_ptr<TableCache> tc;
  if (streamed_) {
    if (!c_->stream_cache_bytes) throw Error{GEM_E_STATE, "streamed join without a table cache size"};
    tc = std::make_unique<TableCache>(c_, c_->stream_cache_bytes, c_->stream_slot_bytes);
    tc->attach(qs);
  }
  // queries are seeded with the identity level of their first vertex when
  // the scheduler starts them (HipSchedBackend::admit)
  std::vector<gemh::SQuery<LevelBuf> *> sq;
  for (VQueryState *S : qs) {
    gemh::SQuery<LevelBuf> &Q = S->s;
    const int64_t partner = Q.partner;
    Q = gemh::SQuery<LevelBuf>{};
    Q.partner = partner;
    // (a pending state's query may still be being prepared: its vertex count
    // was recorded when the state was made)
    Q.nv = S->pending ? S->pending_nv : S->qd->Q.nv;
    Q.nb = S->pending ? std::vector<uint32_t>(Q.nv, S->max_nb.empty() ? 1u : S->max_nb[0]) : S->max_nb;
    Q.level_rows.assign(Q.nv, 0);
    Q.attempt_limit = S->pending ? 0 : attempt_limit(*S, 0);
    sq.push_back(&Q);
  }
  const char *verbose_env = std::getenv("GEM_VERBOSE");
  const bool verbose = verbose_env && verbose_env[0] == '1';
  RunLevels levels(c_, qs);
  HipSchedBackend be{c_, qs, slot, tc.get(), verbose, cap_, lazy_};
  gemh::SchedConfig cfg;
  cfg.cap = cap_;
  cfg.work_limit = work_limit_;
  cfg.budget = total_budget;
  cfg.max_active = c_->max_active;
  cfg.primaries = primaries_;
  cfg.swap_bytes = c_->swap_bytes;
  if (cap_) cfg.measure_units = MEASURE_UNITS;
  const auto t0 = std::chrono::steady_clock::now();
  stats_ = gemh::SchedStats{};
  gemh::run_schedule(be, sq, cfg, &stats_);
  c_->last_sched = stats_;
  c_->last_budget = total_budget;
  if (verbose) {
    std::fprintf(stderr,
                 "[vjoin] run of %zu queries: %llu iterations in %.2f s: %llu length passes %.2f s, extend steps "
                 "%.2f s (%llu 256-row tasks); budget %.2f GiB, peak charged %.2f GiB, %llu forced iterations, "
                 "%llu restarts, %llu queries started (at most %u at once); %llu iterations with more than 4 "
                 "queries active %.2f s, %llu with at most 4 %.2f s\n",
                 qs.size(), (unsigned long long)stats_.iterations,
                 std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count(),
                 (unsigned long long)stats_.length_passes, be.t_len, be.t_ext, (unsigned long long)be.ext_tasks,
                 total_budget / 1073741824.0, stats_.peak_charged / 1073741824.0,
                 (unsigned long long)stats_.forced, (unsigned long long)stats_.restarts,
                 (unsigned long long)stats_.admitted, cfg.max_active, (unsigned long long)be.it_body, be.t_body,
                 (unsigned long long)be.it_tail, be.t_tail);
    std::fflush(stderr);
  }
}

}  // namespace gemd
