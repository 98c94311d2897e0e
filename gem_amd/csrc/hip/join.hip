// Edge-at-a-time join along a connected edge order (the reference's join():
// in-core/lib/join/src/join_trie.cu:1087-1277 with process() 1025-1085,
// host_select 116-395, direct_join 397-718, refer_join 720-1023).
//
// Rows are materialised level by level as row-major tuples of positions (the
// position of the column's vertex in its query vertex's candidate list), so a
// row's key is read directly instead of climbing the reference's parent-pointer
// chain (join_trie_kernel.cu:124-134) and probing a hash table.
//
//   expand (edge x -> y, y new): row r spawns r + [w] for w in T_{x->y}[r[x]]
//     unless w is the vertex of an earlier column with y's label
//     (injectivity, join_trie.cu:450-462);
//   select (both endpoints present): keep r iff r[m] is in T_{q(k)->q(m)}[r[k]]
//     (sorted list: binary search; join_trie_kernel.cu:148);
//   the last step only counts (join_trie.cu:1204 skip_final_materialization);
//     an expansion's count is |list| minus the equal-label columns found in the
//     list by binary search, so final lists are never walked.
//
// Count pass (one thread per row, 256-row blocks) -> block scan -> write pass
// (waves walk their 64 rows' lists 64 items per step, ballot compaction).  A
// level whose output would exceed the level budget is split into block ranges
// and each range is finished depth-first, so memory stays bounded.  When only
// the count is wanted, a level's rows hold only the columns that a later step
// reads, the steps run as one chain of launches with the row counts on the
// device (k_chain) as far as the levels stay below CHAIN_ROWS rows, and after it
// an expansion and the selects that follow it are one walk (k_expand_select).
#include <algorithm>
#include <cstring>
#include <functional>

#include "ctx.h"
#include "wave.h"

namespace gemd {

constexpr uint32_t JB = 256;  // rows per block
constexpr uint32_t JW = JB / 64;

constexpr uint8_t JCOL_NEW = 0xFF;

struct StepArgs {
  const uint32_t *rows;  // null: row r is the single column r
  uint64_t nrows;
  uint32_t k;        // input row width
  uint32_t ko;       // output row width, and the input column each output
  uint8_t src[GEM_MAX_QV];  // column is copied from (JCOL_NEW: the new position)
  uint32_t key_col;  // column whose position keys the table
  uint32_t val_col;  // select: tested column
  const uint64_t *toff;
  const uint32_t *tval;
  // expand: injectivity against equal-label columns
  uint32_t ndup;
  uint32_t dup_col[GEM_MAX_QV];
  const uint32_t *dup_can[GEM_MAX_QV];  // Can(q(col)) lists (vertex ids)
  const uint64_t *bm_new;               // bitmap / rank of the new vertex's candidates
  const uint32_t *rank_new;
  uint32_t W;
};

__device__ __forceinline__ uint32_t position_in(const uint64_t *bm, const uint32_t *rank, uint32_t v) {
  const uint64_t word = bm[v >> 6];
  const uint32_t b = v & 63;
  if (!((word >> b) & 1ull)) return NOT_FOUND;
  return rank[v >> 6] + (uint32_t)__popcll(word & ((1ull << b) - 1));
}

// Bytes charged for one binary search over a list of len entries:
// 4 * ceil(log2(len) + 1).
__device__ __forceinline__ uint64_t search_bytes(uint64_t len) {
  if (len == 0) return 0;
  const uint32_t cl = len == 1 ? 0u : 64u - (uint32_t)__clzll(len - 1);
  return 4ull * (cl + 1);
}

__device__ __forceinline__ uint32_t col_of(const StepArgs &a, uint64_t r, uint32_t c) {
  return a.rows ? a.rows[r * a.k + c] : (uint32_t)r;
}

// Count of row r's expansion: list length minus equal-label columns that occur
// in the list.  Also returns the list start/length, (optionally) the dup
// positions, and the search bytes spent.
__device__ __forceinline__ uint64_t expand_count_row(const StepArgs &a, uint64_t r, uint64_t *o0, uint64_t *len,
                                                     uint32_t *dup_pos, uint64_t *sbytes) {
  const uint32_t p = col_of(a, r, a.key_col);
  const uint64_t b = a.toff[p], e = a.toff[p + 1];
  *o0 = b;
  *len = e - b;
  uint64_t cnt = e - b;
  for (uint32_t c = 0; c < a.ndup; ++c) {
    const uint32_t vid = a.dup_can[c][col_of(a, r, a.dup_col[c])];
    const uint32_t pos = position_in(a.bm_new, a.rank_new, vid);
    if (dup_pos) dup_pos[c] = pos;
    if (pos != NOT_FOUND) {
      *sbytes += search_bytes(e - b);
      if (sorted_contains(a.tval + b, e - b, pos)) --cnt;
    }
  }
  return cnt;
}

__device__ __forceinline__ bool select_row(const StepArgs &a, uint64_t r, uint64_t *len) {
  const uint32_t p = col_of(a, r, a.key_col), v = col_of(a, r, a.val_col);
  const uint64_t b = a.toff[p], e = a.toff[p + 1];
  *len = e - b;
  return sorted_contains(a.tval + b, e - b, v);
}

__device__ __forceinline__ uint64_t block_sum_u64(uint64_t x, uint64_t *sm) {
  x = wave_sum_u64(x);
  const uint32_t w = threadIdx.x / 64;
  if (threadIdx.x % 64 == 0) sm[w] = x;
  __syncthreads();
  uint64_t t = 0;
  for (uint32_t i = 0; i < JW; ++i) t += sm[i];
  __syncthreads();
  return t;
}

// Per-block counts (or, with FINAL, one atomic add of the block sum into
// aux[0]).  With `prof` set, aux[1] += list entries addressed and aux[2] +=
// binary-search bytes (algorithmic-byte bookkeeping).
template <bool SELECT, bool FINAL>
__global__ void __launch_bounds__(JB) k_step_count(const StepArgs a, uint64_t *__restrict__ block_counts,
                                                  unsigned long long *__restrict__ aux, int prof) {
  __shared__ uint64_t sm[JW];
  const uint32_t b = xcd_swizzle(blockIdx.x, gridDim.x);
  const uint64_t r = (uint64_t)b * JB + threadIdx.x;
  uint64_t cnt = 0, len = 0, sb = 0;
  if (r < a.nrows) {
    if (SELECT) {
      cnt = select_row(a, r, &len) ? 1 : 0;
      sb = search_bytes(len);
    } else {
      uint64_t o0;
      cnt = expand_count_row(a, r, &o0, &len, nullptr, &sb);
    }
  }
  const uint64_t s = block_sum_u64(cnt, sm);
  if (threadIdx.x == 0) {
    if (FINAL) {
      if (s) atomicAdd(aux, (unsigned long long)s);
    } else {
      block_counts[b] = s;
    }
  }
  if (prof) {
    const uint64_t ls = block_sum_u64(len, sm), ss = block_sum_u64(sb, sm);
    if (threadIdx.x == 0) {
      atomicAdd(aux + 1, (unsigned long long)ls);
      atomicAdd(aux + 2, (unsigned long long)ss);
    }
  }
}

// Block-level exclusive scan of one u64 per thread.
__device__ __forceinline__ uint64_t block_excl_u64(uint64_t x, uint64_t *sm) {
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint64_t inc = wave_incl_scan_u64(x);
  if (l == 63) sm[w] = inc;
  __syncthreads();
  uint64_t base = 0;
  for (uint32_t i = 0; i < w; ++i) base += sm[i];
  __syncthreads();
  return base + inc - x;
}

// Select write: compact kept rows.  Blocks [b_first, b_first + gridDim.x).
__global__ void __launch_bounds__(JB) k_select_write(const StepArgs a, const uint64_t *__restrict__ block_off,
                                                    uint32_t b_first, uint64_t out_base, uint32_t *__restrict__ out) {
  __shared__ uint64_t sm[JW];
  const uint32_t b = b_first + xcd_swizzle(blockIdx.x, gridDim.x);
  const uint64_t r = (uint64_t)b * JB + threadIdx.x;
  uint64_t len;
  const bool keep = r < a.nrows && select_row(a, r, &len);
  const uint64_t ex = block_excl_u64(keep ? 1 : 0, sm);
  if (keep) {
    const uint64_t o = block_off[b] - out_base + ex;
    uint32_t *dst = out + o * a.ko;
    for (uint32_t c = 0; c < a.ko; ++c) dst[c] = col_of(a, r, a.src[c]);
  }
}

__device__ __forceinline__ uint64_t lanes_between(uint32_t lo, uint32_t hi) {  // bits [lo, hi]
  const uint64_t h = (hi >= 63) ? ~0ull : ((1ull << (hi + 1)) - 1);
  return h & ~((1ull << lo) - 1);
}

// A wave writes the extensions of its 64 rows [row0, row0 + 64): the lists are
// walked 64 items per group; st = starts of the rows' lists in the flattened
// range (st[64] = total), ob = their first entries, ro = their first output
// rows, dups = the equal-label columns' positions (ndup per row).  Row order
// and list order are kept.
__device__ __forceinline__ void write_extensions(const StepArgs &a, uint64_t row0, const uint32_t *st,
                                                 const uint64_t *ob, const uint64_t *ro, const uint32_t *dups,
                                                 uint32_t *out) {
  const uint32_t l = lane_id(), total = st[64];
  uint32_t carry = 0;
  for (uint32_t t = 0; t < total; t += 64) {
    const uint32_t item = t + l;
    const bool iv = item < total;
    const uint32_t row = iv ? seg_of(st, item) : 63;
    const uint32_t rs = st[row], re = st[row + 1];
    const uint32_t last = min(63u, total - 1 - t);
    const uint32_t first = readlane_u32(row, 0);
    bool keep = false;
    uint32_t val = 0;
    if (iv) {
      val = a.tval[ob[row] + (item - rs)];
      keep = true;
      const uint32_t *rdp = dups + (uint64_t)row * a.ndup;
      for (uint32_t c = 0; c < a.ndup; ++c)
        if (rdp[c] == val) keep = false;
    }
    const uint64_t m = __ballot(keep);
    const uint32_t seg_lo = rs > t ? rs - t : 0;
    const uint32_t seg_hi = (re < t + 64 ? re - t : 64) - 1;
    const bool row_done = re <= t + 64;
    const uint32_t before = (row == first) ? carry : 0;
    if (keep) {
      const uint64_t below = lanes_between(seg_lo, l) & ~(1ull << l);
      const uint64_t o = ro[row] + before + (uint64_t)__popcll(m & below);
      uint32_t *dst = out + o * a.ko;
      for (uint32_t c = 0; c < a.ko; ++c) dst[c] = a.src[c] == JCOL_NEW ? val : col_of(a, row0 + row, a.src[c]);
    }
    const uint32_t tot_row = iv ? before + (uint32_t)__popcll(m & lanes_between(seg_lo, seg_hi)) : 0;
    carry = readlane_u32(row_done ? 0u : tot_row, last);
  }
}

// Expand write.  Dynamic LDS: JW * 64 * ndup u32 dup positions.
__global__ void __launch_bounds__(JB) k_expand_write(const StepArgs a, const uint64_t *__restrict__ block_off,
                                                    uint32_t b_first, uint64_t out_base, uint32_t *__restrict__ out,
                                                    unsigned long long *__restrict__ aux, int prof) {
  __shared__ uint64_t sm[JW];
  __shared__ uint32_t st[JW][65];
  __shared__ uint64_t ob[JW][64];
  __shared__ uint64_t ro[JW][64];
  extern __shared__ uint32_t dup_lds[];
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint32_t b = b_first + xcd_swizzle(blockIdx.x, gridDim.x);
  const uint64_t r = (uint64_t)b * JB + threadIdx.x;
  uint32_t *dp = dup_lds + (uint64_t)(w * 64 + l) * a.ndup;
  uint64_t cnt = 0, o0 = 0, len = 0, sb = 0;
  if (r < a.nrows) cnt = expand_count_row(a, r, &o0, &len, dp, &sb);
  const uint64_t ex = block_excl_u64(cnt, sm);
  const uint32_t ilen = (uint32_t)len;
  const uint32_t incl = wave_incl_scan_u32(ilen);
  const uint32_t total = readlane_u32(incl, 63);
  if (prof && l == 0 && total) atomicAdd(aux + 1, (unsigned long long)total);
  st[w][l] = incl - ilen;
  if (l == 63) st[w][64] = total;
  ob[w][l] = o0;
  ro[w][l] = block_off[b] - out_base + ex;
  __syncthreads();
  write_extensions(a, (uint64_t)b * JB + w * 64, st[w], ob[w], ro[w], dup_lds + (uint64_t)w * 64 * a.ndup, out);
}

// One step of the count-only chain: the level's row count comes from the step
// before (*n_in) and goes to the next (*n_out); output places are handed out by
// one atomic per 64 rows (a count does not depend on row order).  A level past
// its room (cap_in, cap_out rows) is counted but not written whole, and the
// steps after it do nothing: the host goes on from it with the count / scan /
// write passes.  A step of those costs three launches, a copy and two waits,
// 40 us however few the rows; a chained one 5 to 8 us.  (A 5-vertex query on
// 10,000 vertices: 246 us, chained 128.)
// FINAL: *n_out += the count.  Dynamic LDS as k_expand_write (expand).
constexpr uint32_t CHAIN_BLOCKS = 1024;
constexpr uint64_t CHAIN_ROWS = 1ull << 18, CHAIN_LEAST = 1ull << 13;
template <bool SELECT, bool FINAL>
__global__ void __launch_bounds__(JB) k_chain(const StepArgs a, const unsigned long long *__restrict__ n_in,
                                             uint64_t cap_in, unsigned long long *__restrict__ n_out,
                                             uint64_t cap_out, uint32_t *__restrict__ out) {
  __shared__ uint32_t st[JW][65];
  __shared__ uint64_t ob[JW][64];
  __shared__ uint64_t ro[JW][64];
  extern __shared__ uint32_t dup_lds[];
  const uint64_t n = *n_in;
  if (n > cap_in) return;
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  uint64_t sum = 0;
  for (uint64_t row0 = ((uint64_t)blockIdx.x * JW + w) * 64; row0 < n; row0 += (uint64_t)gridDim.x * JB) {
    const uint64_t r = row0 + l;
    uint64_t cnt = 0, o0 = 0, len = 0, sb = 0;
    uint32_t *dp = dup_lds + (uint64_t)(w * 64 + l) * a.ndup;
    if (r < n) {
      if (SELECT)
        cnt = select_row(a, r, &len) ? 1 : 0;
      else
        cnt = expand_count_row(a, r, &o0, &len, FINAL ? nullptr : dp, &sb);
    }
    if (FINAL) {
      sum += cnt;
      continue;
    }
    const uint64_t incl = wave_incl_scan_u64(cnt), all = readlane_u64(incl, 63);
    if (!all) continue;
    uint64_t base = 0;
    if (l == 0) base = atomicAdd(n_out, (unsigned long long)all);
    base = readlane_u64(base, 0);
    if (base + all > cap_out) continue;
    if (SELECT) {
      if (cnt) {
        uint32_t *dst = out + (base + incl - 1) * a.ko;
        for (uint32_t c = 0; c < a.ko; ++c) dst[c] = col_of(a, r, a.src[c]);
      }
      continue;
    }
    const uint32_t il = wave_incl_scan_u32((uint32_t)len);
    st[w][l] = il - (uint32_t)len;
    if (l == 63) st[w][64] = il;
    ob[w][l] = o0;
    ro[w][l] = base + incl - cnt;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    write_extensions(a, row0, st[w], ob[w], ro[w], dup_lds + (uint64_t)w * 64 * a.ndup, out);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (FINAL) {
    sum = wave_sum_u64(sum);
    if (l == 0 && sum) atomicAdd(n_out, (unsigned long long)sum);
  }
}

// An expansion and the selects that follow it, in one walk (counts only): the
// expanded rows, of which the selects mostly keep a part, are never written.
// (An 8-vertex query on a 2^18 R-MAT graph: the expansion wrote its rows in 820
// us, the two selects counted and wrote theirs in 428 and 682, 222 and 341 us;
// the whole match 3.30 ms, fused 1.25.)
// A wave takes `group` rows at a time (chosen on the host so that it walks
// about GROUP_ITEMS entries: 64 rows of long lists would leave waves idle at
// the end), 256 entries a step, four per lane, so that a lane has four searches
// in flight; survivors are staged over all groups of the wave, so that an atomic
// on the output counter (10 ns each, device-wide) is paid once per 768 or more.
// ctr[j] += rows that pass select j; the last one's counter hands out the places.
// FINAL: the last select is the query's last step, whose rows are only counted.
constexpr uint32_t MAX_SELECTS = 4, GROUP_ITEMS = 2048, SSTAGE = 1024, SELECT_BLOCKS = 1024;
struct Selects {
  uint32_t n;
  // columns of the row before the expansion, or JCOL_NEW
  uint8_t key_col[MAX_SELECTS], val_col[MAX_SELECTS];
  const uint64_t *toff[MAX_SELECTS];
  const uint32_t *tval[MAX_SELECTS];
};
template <bool FINAL>
__global__ void __launch_bounds__(JB) k_expand_select(const StepArgs a, const Selects q, uint32_t group,
                                                     unsigned long long *__restrict__ ctr, uint64_t cap_out,
                                                     uint32_t *__restrict__ out) {
  constexpr uint32_t STAGE = FINAL ? 1 : SSTAGE;
  __shared__ uint32_t st[JW][64];                          // first item of each row of the group
  __shared__ uint64_t ob[JW][64];                          // its list's first entry
  __shared__ uint8_t full_row[JW][64];                     // the group's rows that have entries
  __shared__ uint32_t marks[JW][8];                        // bit i: a row's entries start at item i of the step
  __shared__ uint32_t sv_row[JW][STAGE], sv_val[JW][STAGE];  // staged survivors
  __shared__ unsigned long long total[MAX_SELECTS];
  extern __shared__ uint32_t dup_lds[];
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64;
  if (threadIdx.x < MAX_SELECTS) total[threadIdx.x] = 0;
  __syncthreads();
  uint32_t *dp = dup_lds + (uint64_t)(w * 64 + l) * a.ndup;
  const uint32_t *any = reinterpret_cast<const uint32_t *>(a.toff);  // a readable word
  uint64_t cnt[MAX_SELECTS] = {};
  uint32_t pend = 0;
  auto settle = [&]() {
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  };
  auto flush = [&]() {
    if (FINAL || !pend) return;
    uint64_t base = 0;
    if (l == 0) base = atomicAdd(&ctr[q.n - 1], (unsigned long long)pend);
    base = readlane_u64(base, 0);
    const uint32_t n = base >= cap_out ? 0 : cap_out - base < pend ? (uint32_t)(cap_out - base) : pend;
    for (uint32_t i = l; i < n; i += 64) {
      const uint64_t r = sv_row[w][i];
      const uint32_t v = sv_val[w][i];
      uint32_t *dst = out + (base + i) * a.ko;
      for (uint32_t c = 0; c < a.ko; c += 4) {
        const uint32_t m = a.ko - c < 4 ? a.ko - c : 4;
        u32x4 x;
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
          if (e < m) x[e] = a.src[c + e] == JCOL_NEW ? v : col_of(a, r, a.src[c + e]);
        st_words(dst + c, x, m);
      }
    }
    settle();
    pend = 0;
  };
  const uint64_t step = (uint64_t)gridDim.x * JW * group;
  for (uint64_t row0 = ((uint64_t)blockIdx.x * JW + w) * group; row0 < a.nrows; row0 += step) {
    uint64_t o0 = 0, len64 = 0;
    const uint64_t r = row0 + l;
    if (l < group && r < a.nrows) {
      const uint32_t p = col_of(a, r, a.key_col);
      const u64x2 o = ld_pair(a.toff + p);
      o0 = o.x;
      len64 = o.y - o.x;
      for (uint32_t c = 0; c < a.ndup; ++c)
        dp[c] = position_in(a.bm_new, a.rank_new, a.dup_can[c][col_of(a, r, a.dup_col[c])]);
    }
    const uint32_t len = (uint32_t)len64, incl = wave_incl_scan_u32(len), start = incl - len;
    const uint32_t items = readlane_u32(incl, 63);
    st[w][l] = start;
    ob[w][l] = o0;
    const uint64_t full = __ballot(len);
    if (len) full_row[w][rank_below(full)] = (uint8_t)l;
    settle();
    uint32_t rows_before = 0;  // rows with entries that start before the step
    for (uint32_t s = 0; s < items; s += 256) {
      if (l < 8) marks[w][l] = 0;
      settle();
      if (len && start - s < 256) atomicOr(&marks[w][(start - s) / 32], 1u << ((start - s) % 32));
      settle();
      uint32_t val[4], rw[4];
      bool keep[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t item = s + 64u * g + l;
        keep[g] = item < items;
        const uint32_t mlo = __builtin_amdgcn_readfirstlane(marks[w][2 * g]);
        const uint32_t mhi = __builtin_amdgcn_readfirstlane(marks[w][2 * g + 1]);
        const uint64_t m = (uint64_t)mhi << 32 | mlo;
        rw[g] = full_row[w][rows_before + rank_below(m) + ((m >> l) & 1) - 1];
        rows_before += (uint32_t)__popcll(m);
        val[g] = keep[g] ? ldg(a.tval + ob[w][rw[g]] + (item - st[w][rw[g]])) : 0;
      }
      for (uint32_t c = 0; c < a.ndup; ++c)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (dup_lds[(uint64_t)(w * 64 + rw[g]) * a.ndup + c] == val[g]) keep[g] = false;
      uint64_t m[4];
      uint32_t nk = 0, before[4];
      for (uint32_t j = 0; j < q.n; ++j) {
        const uint32_t *lists[4];
        uint32_t lens[4], v[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          lists[g] = any;
          lens[g] = v[g] = 0;
          if (keep[g]) {
            const uint64_t row = row0 + rw[g];
            const uint32_t p = q.key_col[j] == JCOL_NEW ? val[g] : col_of(a, row, q.key_col[j]);
            v[g] = q.val_col[j] == JCOL_NEW ? val[g] : col_of(a, row, q.val_col[j]);
            const u64x2 o = ld_pair(q.toff[j] + p);
            lists[g] = q.tval[j] + o.x;
            lens[g] = (uint32_t)(o.y - o.x);
          }
        }
        contains_quad(lists, lens, v, keep, any);
        nk = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          m[g] = __ballot(keep[g]);
          before[g] = nk;
          nk += (uint32_t)__popcll(m[g]);
        }
#pragma unroll
        for (uint32_t x = 0; x < MAX_SELECTS; ++x)
          if (x == j) cnt[x] += nk;
        if (!nk) break;
      }
      if (!FINAL && nk) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (keep[g]) {
            const uint32_t i = pend + before[g] + rank_below(m[g]);
            sv_row[w][i] = (uint32_t)(row0 + rw[g]);
            sv_val[w][i] = val[g];
          }
        settle();
        pend += nk;
        if (pend > STAGE - 256) flush();
      }
    }
    settle();  // the group's lists are rewritten by the next one
  }
  flush();
  if (l == 0)
    for (uint32_t j = 0; j < q.n; ++j) {
      uint64_t c = 0;
#pragma unroll
      for (uint32_t x = 0; x < MAX_SELECTS; ++x) c = x == j ? cnt[x] : c;
      if (c) atomicAdd(&total[j], (unsigned long long)c);
    }
  __syncthreads();
  // (the last select's counter has counted its rows as it gave their places)
  if (threadIdx.x < q.n - (FINAL ? 0 : 1) && total[threadIdx.x]) atomicAdd(&ctr[threadIdx.x], total[threadIdx.x]);
}

// Level counts of a chain: n[0] = first, the rest zero; and to the host.
__global__ void k_chain_init(unsigned long long *n, uint32_t steps, uint64_t first) {
  for (uint32_t i = threadIdx.x; i <= steps; i += blockDim.x) n[i] = i ? 0 : first;
}
__global__ void k_chain_done(const unsigned long long *__restrict__ n, uint32_t steps, uint64_t *__restrict__ host) {
  for (uint32_t i = threadIdx.x; i <= steps; i += blockDim.x) host[i] = n[i];
}

// Final rows (positions) -> vertex ids in query-vertex order.
__global__ void k_rows_to_ids(const uint32_t *__restrict__ rows, uint64_t nrows, uint32_t k,
                              const uint32_t *const *__restrict__ col_can, const uint32_t *__restrict__ col_u,
                              uint32_t nv, uint32_t *__restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrows * k) return;
  const uint64_t r = i / k;
  const uint32_t c = (uint32_t)(i % k);
  out[r * nv + col_u[c]] = col_can[c][rows[i]];
}

struct JStep {
  bool select;
  uint32_t table;  // directed edge
  uint32_t key_col, val_col, new_u;
  uint32_t ndup;
  uint32_t dup_col[GEM_MAX_QV];
  // query columns of the rows the step reads, and of those it writes
  uint32_t ncols;
  std::vector<uint32_t> in, out;
};

class JoinRunner {
 public:
  JoinRunner(gem_ctx *c, const gemh::JoinPlan &plan, uint64_t cap, gem_step_log *log, EmbSink *sink)
      : c_(c), Qd_(c->q), cap_(cap), log_(log), sink_(sink) {
    // step 0: the first table seeds 2-column rows from the 1-column identity
    JStep s0{};
    s0.select = false;
    s0.table = plan.first_directed;
    s0.key_col = 0;
    s0.new_u = plan.col_u[1];
    steps_.push_back(s0);
    for (const auto &ps : plan.steps) {
      JStep s{};
      s.select = ps.select;
      s.table = ps.directed;
      s.key_col = ps.key_col;
      s.val_col = ps.val_col;
      s.new_u = ps.new_u;
      s.ndup = ps.num_dup;
      for (uint32_t i = 0; i < ps.num_dup; ++i) s.dup_col[i] = ps.dup_cols[i];
      steps_.push_back(s);
    }
    // columns each step's rows hold: all of them for a sink, else those that
    // this step or a later one reads
    std::vector<uint32_t> last(plan.col_u.size(), 0);
    for (uint32_t i = 0; i < steps_.size(); ++i) {
      const JStep &st = steps_[i];
      last[st.key_col] = i;
      if (st.select) last[st.val_col] = i;
      for (uint32_t d = 0; d < st.ndup; ++d) last[st.dup_col[d]] = i;
    }
    uint32_t ncols = 1;
    for (uint32_t i = 0; i < steps_.size(); ++i) {
      JStep &st = steps_[i];
      st.ncols = ncols;
      for (uint32_t c = 0; c < ncols; ++c)
        if (sink_ || last[c] >= i) st.in.push_back(c);
      if (!st.select) ++ncols;
      for (uint32_t c = 0; c < ncols; ++c)
        if (sink_ || last[c] > i) st.out.push_back(c);
    }
    col_u_ = plan.col_u;
    rows_.assign(steps_.size(), 0);
    ms_.assign(steps_.size(), 0.0f);
    budget_ = std::max<uint64_t>(c->level_budget_bytes, 1ull << 20);
    work_limit_ = c->work_limit_rows;
  }

  void run(JoinOut *out) {
    hipStream_t s = c_->stream;
    d_aux_.alloc(24, s);
    if (log_) {
      GEM_HIP_CHECK(hipEventCreate(&e0_));
      GEM_HIP_CHECK(hipEventCreate(&e1_));
    }
    const uint32_t a = col_u_[0];
    const uint64_t n0 = Qd_.ncan[a];
    if (n0) {
      if (!log_ && !sink_ && !c_->prof.on) {
        shuffled_ = true;
        chain(n0);
        if (ordered_again_) {
          shuffled_ = stop_ = work_limited_ = false;
          processed_ = 0;
          level(0, nullptr, n0);
        }
      } else {
        level(0, nullptr, n0);
      }
    }
    if (e0_) (void)hipEventDestroy(e0_);
    if (e1_) (void)hipEventDestroy(e1_);
    out->count = saturated_ ? cap_ : final_total_;
    out->saturated = saturated_;
    out->emb_written = emb_rows_;
    out->sink_stopped = sink_stopped_;
    out->rows_processed = processed_;
    out->work_limited = work_limited_;
    if (work_limited_) {
      out->count = 0;
      out->saturated = false;
    }
    if (log_) {
      for (size_t i = 0; i < steps_.size() && i < GEM_MAX_QE; ++i) {
        log_->edge[i] = i == 0 ? first_edge_ : steps_[i].table >> 1;
        log_->is_select[i] = steps_[i].select;
        log_->rows[i] = rows_[i];
        log_->ms[i] = ms_[i];
      }
    }
  }

  uint32_t first_edge_ = 0;

 private:
  gem_ctx *c_;
  QueryDev &Qd_;
  uint64_t cap_;
  gem_step_log *log_;
  EmbSink *sink_;
  std::vector<JStep> steps_;
  std::vector<uint32_t> col_u_;
  std::vector<uint64_t> rows_;
  std::vector<float> ms_;
  uint64_t budget_;
  DevBuf d_aux_;
  uint64_t final_total_ = 0;
  bool saturated_ = false;
  bool stop_ = false;
  uint64_t processed_ = 0;
  uint64_t work_limit_ = 0;
  bool work_limited_ = false;
  uint64_t emb_rows_ = 0;
  bool sink_stopped_ = false;
  // chained or fused steps leave a level's rows in no fixed order.  A level cut
  // into ranges under a cap or a work limit needs one, as the ranges that are
  // reached before the join stops decide the rows it has processed: the first
  // such cut starts the join again without those steps.
  bool shuffled_ = false, ordered_again_ = false;
  std::vector<uint32_t> host_rows_;
  hipEvent_t e0_{}, e1_{};

  StepArgs args(const JStep &st, const uint32_t *rows, uint64_t n) {
    StepArgs a{};
    a.rows = rows;
    a.nrows = n;
    a.k = (uint32_t)st.in.size();
    a.ko = (uint32_t)st.out.size();
    auto at = [&](uint32_t col) { return (uint32_t)(std::lower_bound(st.in.begin(), st.in.end(), col) - st.in.begin()); };
    for (uint32_t c = 0; c < a.ko; ++c) a.src[c] = st.out[c] == st.ncols ? JCOL_NEW : (uint8_t)at(st.out[c]);
    a.key_col = at(st.key_col);
    if (st.select) a.val_col = at(st.val_col);
    const TableDev &T = Qd_.tab[st.table];
    if (!T.present) throw Error{GEM_E_STATE, "join step uses a table that was not built"};
    a.toff = T.off.as<uint64_t>();
    a.tval = T.val.as<uint32_t>();
    a.ndup = st.ndup;
    a.W = Qd_.W;
    if (!st.select) {
      a.bm_new = Qd_.bitmap.as<uint64_t>() + (uint64_t)st.new_u * Qd_.W;
      a.rank_new = Qd_.rank.as<uint32_t>() + (uint64_t)st.new_u * (Qd_.W + 1);
      for (uint32_t i = 0; i < st.ndup; ++i) {
        a.dup_col[i] = at(st.dup_col[i]);
        a.dup_can[i] = Qd_.can.as<uint32_t>() + Qd_.can_off[col_u_[st.dup_col[i]]];
      }
    }
    return a;
  }

  // Step times are taken for a log only (each waits for its step).
  void time_begin() {
    if (log_) GEM_HIP_CHECK(hipEventRecord(e0_, c_->stream));
  }
  void time_end(uint32_t s) {
    if (!log_) return;
    GEM_HIP_CHECK(hipEventRecord(e1_, c_->stream));
    GEM_HIP_CHECK(hipEventSynchronize(e1_));
    float ms = 0;
    GEM_HIP_CHECK(hipEventElapsedTime(&ms, e0_, e1_));
    ms_[s] += ms;
  }

  // aux[0] = final count, aux[1] = list entries addressed, aux[2] = search bytes
  void read_aux(uint64_t *out3) {
    uint64_t *h = pinned<uint64_t>(c_, 3);
    GEM_HIP_CHECK(hipMemcpyAsync(h, d_aux_.p, 24, hipMemcpyDeviceToHost, c_->stream));
    GEM_HIP_CHECK(hipStreamSynchronize(c_->stream));
    out3[0] = h[0];
    out3[1] = h[1];
    out3[2] = h[2];
  }

  // Did the rows read so far, with n more, pass the work limit?
  bool over_limit(uint64_t n) {
    processed_ += n;
    if (!work_limit_ || processed_ <= work_limit_) return false;
    work_limited_ = true;
    stop_ = true;
    return true;
  }

  // The steps as one chain of launches from the identity rows of the first
  // column, with one wait at its end; from the first level without room on
  // (CHAIN_ROWS rows, or the level budget), level() takes over.
  void chain(uint64_t n0) {
    hipStream_t s = c_->stream;
    const uint32_t ns = (uint32_t)steps_.size();
    // rows a level has room for: many times its estimate by the tables' mean
    // list lengths, so that small queries take small buffers
    std::vector<uint64_t> cap(ns + 1, ~0ull);
    size_t words[2] = {0, 0};
    double est = (double)n0;
    for (uint32_t i = 0; i + 1 < ns; ++i) {
      const JStep &st = steps_[i];
      const TableDev &T = Qd_.tab[st.table];
      if (!st.select) est *= (double)T.size / std::max<double>(1, Qd_.ncan[T.key_u]);
      cap[i + 1] = std::min<uint64_t>(CHAIN_ROWS, budget_ / (4ull * (st.select ? st.ncols : st.ncols + 1)));
      cap[i + 1] = std::min<uint64_t>(cap[i + 1], std::max<uint64_t>(CHAIN_LEAST, (uint64_t)std::min(16 * est, 1e9)));
      words[i & 1] = std::max<size_t>(words[i & 1], cap[i + 1] * st.out.size());
    }
    DevBuf buf[2], dn;
    for (int i = 0; i < 2; ++i) buf[i].alloc(words[i] * 4, s);
    dn.alloc((ns + 1) * 8, s);
    auto *n = dn.as<unsigned long long>();
    k_chain_init<<<1, 64, 0, s>>>(n, ns, n0);
    for (uint32_t i = 0; i < ns; ++i) {
      const JStep &st = steps_[i];
      const uint32_t *rows = i ? buf[(i - 1) & 1].as<uint32_t>() : nullptr;
      uint32_t *out = buf[i & 1].as<uint32_t>();
      const StepArgs a = args(st, rows, 0);
      const bool last = i + 1 == ns;
      const size_t lds = last || st.select ? 0 : (size_t)JW * 64 * st.ndup * 4;
      const uint64_t most = i ? cap[i] : n0;
      const uint32_t grid = (uint32_t)std::min<uint64_t>((most + JB - 1) / JB, CHAIN_BLOCKS);
      auto kernel = st.select ? (last ? k_chain<true, true> : k_chain<true, false>)
                              : (last ? k_chain<false, true> : k_chain<false, false>);
      kernel<<<grid, JB, lds, s>>>(a, n + i, cap[i], n + i + 1, cap[i + 1], out);
    }
    uint64_t *h = pinned<uint64_t>(c_, ns + 1);
    k_chain_done<<<1, 64, 0, s>>>(n, ns, pinned_dev(c_, h));
    GEM_LAUNCH_CHECK("k_chain");
    GEM_HIP_CHECK(hipStreamSynchronize(s));
    const std::vector<uint64_t> got(h, h + ns + 1);
    for (uint32_t i = 0; i < ns; ++i) {
      if (!got[i]) return;
      if (got[i + 1] > cap[i + 1]) {  // no room: step i again, the other way
        level(i, i ? buf[(i - 1) & 1].as<uint32_t>() : nullptr, got[i]);
        return;
      }
      if (over_limit(got[i])) return;
    }
    final_total_ = got[ns];
    if (cap_ && final_total_ > cap_) saturated_ = true;
  }

  // Step si, an expansion of n rows to `total`, and the selects after it (up to
  // MAX_SELECTS), then the steps after those.
  void expand_select(uint32_t si, const uint32_t *rows, uint64_t n, uint64_t total) {
    hipStream_t s = c_->stream;
    const uint32_t ns = (uint32_t)steps_.size();
    const JStep &st = steps_[si];
    Selects q{};
    while (q.n < MAX_SELECTS && si + 1 + q.n < ns && steps_[si + 1 + q.n].select) ++q.n;
    const uint32_t se = si + q.n;  // the last select
    const bool last = se + 1 == ns;
    StepArgs a = args(st, rows, n);
    auto at = [&](uint32_t col) {
      return col == st.ncols ? JCOL_NEW
                             : (uint8_t)(std::lower_bound(st.in.begin(), st.in.end(), col) - st.in.begin());
    };
    for (uint32_t j = 0; j < q.n; ++j) {
      const JStep &sel = steps_[si + 1 + j];
      const TableDev &T = Qd_.tab[sel.table];
      if (!T.present) throw Error{GEM_E_STATE, "join step uses a table that was not built"};
      q.key_col[j] = at(sel.key_col);
      q.val_col[j] = at(sel.val_col);
      q.toff[j] = T.off.as<uint64_t>();
      q.tval[j] = T.val.as<uint32_t>();
    }
    const std::vector<uint32_t> &cols = steps_[se].out;
    a.ko = last ? 0 : (uint32_t)cols.size();
    for (uint32_t c = 0; c < a.ko; ++c) a.src[c] = at(cols[c]);
    DevBuf outb, ctr;
    outb.alloc(total * 4ull * a.ko, s);
    ctr.alloc(MAX_SELECTS * 8, s);
    uint32_t group = 64;
    while (group > 4 && (double)total / (double)n * group > GROUP_ITEMS) group /= 2;
    const uint64_t groups = (n + group - 1) / group;
    const uint32_t grid = (uint32_t)std::min<uint64_t>((groups + JW - 1) / JW, SELECT_BLOCKS);
    const size_t lds = (size_t)JW * 64 * st.ndup * 4;
    auto *dc = ctr.as<unsigned long long>();
    k_chain_init<<<1, 64, 0, s>>>(dc, q.n - 1, 0);
    if (last)
      k_expand_select<true><<<grid, JB, lds, s>>>(a, q, group, dc, 0, nullptr);
    else
      k_expand_select<false><<<grid, JB, lds, s>>>(a, q, group, dc, total, outb.as<uint32_t>());
    uint64_t *h = pinned<uint64_t>(c_, MAX_SELECTS);
    k_chain_done<<<1, 64, 0, s>>>(dc, q.n - 1, pinned_dev(c_, h));
    GEM_LAUNCH_CHECK("k_expand_select");
    GEM_HIP_CHECK(hipStreamSynchronize(s));
    uint64_t got[MAX_SELECTS];
    std::copy(h, h + q.n, got);
    uint64_t in = total;  // rows that select j read
    for (uint32_t j = 0; j < q.n; ++j) {
      if (!in || over_limit(in)) return;
      in = got[j];
    }
    if (last) {
      final_total_ += in;
      if (cap_ && final_total_ > cap_) saturated_ = stop_ = true;
      return;
    }
    outb.shrink(in * 4ull * a.ko);
    level(se + 1, outb.as<uint32_t>(), in);
  }

  void final_count(uint32_t si, const uint32_t *rows, uint64_t n) {
    const JStep &st = steps_[si];
    StepArgs a = args(st, rows, n);
    const uint32_t k = a.k;
    const uint32_t nb = (uint32_t)((n + JB - 1) / JB);
    const int prof = c_->prof.on ? 1 : 0;
    time_begin();
    GEM_HIP_CHECK(hipMemsetAsync(d_aux_.p, 0, 24, c_->stream));
    {
      ProfLaunch pl(c_, st.select ? K_SELECT_FINAL : K_EXPAND_FINAL);
      if (st.select)
        k_step_count<true, true><<<nb, JB, 0, c_->stream>>>(a, nullptr, d_aux_.as<unsigned long long>(), prof);
      else
        k_step_count<false, true><<<nb, JB, 0, c_->stream>>>(a, nullptr, d_aux_.as<unsigned long long>(), prof);
      GEM_LAUNCH_CHECK("k_step_count<final>");
    }
    uint64_t aux[3];
    read_aux(aux);
    time_end(si);
    // rows + offset pair per row + searches
    prof_bytes(c_, st.select ? K_SELECT_FINAL : K_EXPAND_FINAL, (4.0 * k + 8.0) * n + (double)aux[2]);
    const uint64_t got = aux[0];
    rows_[si] += got;
    final_total_ += got;
    if (cap_ && final_total_ > cap_) {
      saturated_ = true;
      stop_ = true;
    }
  }

  void emit_rows(const uint32_t *rows, uint64_t n, uint32_t k) {
    // rows are final (k == nv columns): vertex ids, in query-vertex order, to the sink
    const uint32_t nv = Qd_.Q.nv;
    if (!sink_ || n == 0) return;
    hipStream_t s = c_->stream;
    std::vector<const uint32_t *> cc(k);
    for (uint32_t c = 0; c < k; ++c) cc[c] = Qd_.can.as<uint32_t>() + Qd_.can_off[col_u_[c]];
    DevBuf dcc, dcu, dout;
    dcc.alloc(k * 8, s);
    dcu.alloc(k * 4, s);
    dout.alloc(n * nv * 4, s);
    GEM_HIP_CHECK(hipMemcpyAsync(dcc.p, cc.data(), k * 8, hipMemcpyHostToDevice, s));
    GEM_HIP_CHECK(hipMemcpyAsync(dcu.p, col_u_.data(), k * 4, hipMemcpyHostToDevice, s));
    const uint64_t tot = n * k;
    k_rows_to_ids<<<(uint32_t)((tot + 255) / 256), 256, 0, s>>>(rows, n, k, dcc.as<const uint32_t *>(),
                                                                 dcu.as<uint32_t>(), nv, dout.as<uint32_t>());
    GEM_LAUNCH_CHECK("k_rows_to_ids");
    uint32_t *host = sink_->place(n, nv);
    if (!host) {
      host_rows_.resize(n * nv);
      host = host_rows_.data();
    }
    GEM_HIP_CHECK(hipMemcpyAsync(host, dout.p, n * nv * 4, hipMemcpyDeviceToHost, s));
    GEM_HIP_CHECK(hipStreamSynchronize(s));
    emb_rows_ += n;
    if (!sink_->put(host, n, nv)) {
      sink_stopped_ = true;
      stop_ = true;
    }
  }

  // Apply step si to `n` rows.
  void level(uint32_t si, const uint32_t *rows, uint64_t n) {
    if (stop_ || n == 0 || over_limit(n)) return;
    const JStep &st = steps_[si];
    const bool last = si + 1 == steps_.size();
    if (last && !sink_) {
      final_count(si, rows, n);
      return;
    }
    hipStream_t s = c_->stream;
    StepArgs a = args(st, rows, n);
    const uint32_t k = a.k;
    const uint32_t nb = (uint32_t)((n + JB - 1) / JB);
    const int prof = c_->prof.on ? 1 : 0;
    time_begin();
    DevBuf bc, bo;
    bc.alloc((uint64_t)nb * 8, s);
    bo.alloc(((uint64_t)nb + 1) * 8, s);
    if (prof) GEM_HIP_CHECK(hipMemsetAsync(d_aux_.p, 0, 24, s));
    {
      ProfLaunch pl(c_, st.select ? K_SELECT_COUNT : K_EXPAND_COUNT);
      if (st.select)
        k_step_count<true, false><<<nb, JB, 0, s>>>(a, bc.as<uint64_t>(), d_aux_.as<unsigned long long>(), prof);
      else
        k_step_count<false, false><<<nb, JB, 0, s>>>(a, bc.as<uint64_t>(), d_aux_.as<unsigned long long>(), prof);
      GEM_LAUNCH_CHECK("k_step_count");
    }
    uint64_t *htot = pinned<uint64_t>(c_, 1);
    scan_u64(c_, bc.as<uint64_t>(), bo.as<uint64_t>(), nb, pinned_dev(c_, htot));
    GEM_HIP_CHECK(hipStreamSynchronize(s));
    const uint64_t total = *htot;
    bc.reset();
    rows_[si] += total;
    // the budget is charged for every column, held or not (so the chunks do
    // not depend on which are)
    const uint64_t row_bytes = 4ull * (st.select ? st.ncols : st.ncols + 1), out_bytes = 4ull * a.ko;
    double search_per_row = 0;
    if (prof) {
      uint64_t aux[3];
      read_aux(aux);
      // count pass: rows, offset pairs, searches
      prof_bytes(c_, st.select ? K_SELECT_COUNT : K_EXPAND_COUNT, (4.0 * k + 8.0) * n + (double)aux[2]);
      search_per_row = n ? (double)aux[2] / (double)n : 0.0;
    }
    if (total == 0) {
      time_end(si);
      return;
    }
    // block ranges whose output fits the level budget
    std::vector<std::pair<uint32_t, uint32_t>> ranges;
    std::vector<uint64_t> hoff;
    if (total * row_bytes <= budget_) {
      ranges.push_back({0, nb});
    } else if (shuffled_ && (cap_ || work_limit_)) {
      ordered_again_ = stop_ = true;
      return;
    } else {
      hoff.resize((size_t)nb + 1);
      GEM_HIP_CHECK(hipMemcpyAsync(hoff.data(), bo.p, ((uint64_t)nb + 1) * 8, hipMemcpyDeviceToHost, s));
      GEM_HIP_CHECK(hipStreamSynchronize(s));
      const uint64_t lim = std::max<uint64_t>(budget_ / row_bytes, 1);
      uint32_t b0 = 0;
      while (b0 < nb) {
        uint32_t b1 = b0 + 1;
        while (b1 < nb && hoff[b1 + 1] - hoff[b0] <= lim) ++b1;
        ranges.push_back({b0, b1});
        b0 = b1;
      }
    }
    if (shuffled_ && !st.select && steps_[si + 1].select && ranges.size() == 1 && n <= 0xFFFFFFFFull &&
        st.ndup <= 16) {  // (LDS: 36 KB and 1 KB per equal-label column)
      expand_select(si, rows, n, total);
      return;
    }
    bool timed = false;
    for (auto [b0, b1] : ranges) {
      if (stop_) break;
      const uint64_t base = hoff.empty() ? 0 : hoff[b0];
      const uint64_t cnt = hoff.empty() ? total : hoff[b1] - hoff[b0];
      if (cnt == 0) continue;
      if (timed) time_begin();
      DevBuf outb;
      outb.alloc(cnt * out_bytes, s);
      const uint32_t g = b1 - b0;
      if (prof) GEM_HIP_CHECK(hipMemsetAsync(d_aux_.p, 0, 24, s));
      {
        ProfLaunch pl(c_, st.select ? K_SELECT_WRITE : K_EXPAND_WRITE);
        if (st.select) {
          k_select_write<<<g, JB, 0, s>>>(a, bo.as<uint64_t>(), b0, base, outb.as<uint32_t>());
          GEM_LAUNCH_CHECK("k_select_write");
        } else {
          const size_t lds = (size_t)JW * 64 * st.ndup * 4;
          k_expand_write<<<g, JB, lds, s>>>(a, bo.as<uint64_t>(), b0, base, outb.as<uint32_t>(),
                                            d_aux_.as<unsigned long long>(), prof);
          GEM_LAUNCH_CHECK("k_expand_write");
        }
      }
      if (prof) {
        // rows of the range (+ their searches), list entries walked, rows written
        uint64_t aux[3];
        read_aux(aux);
        const double nr = (double)std::min<uint64_t>((uint64_t)(b1 - b0) * JB, n - (uint64_t)b0 * JB);
        prof_bytes(c_, st.select ? K_SELECT_WRITE : K_EXPAND_WRITE,
                   (4.0 * k + 8.0 + search_per_row) * nr + 4.0 * (double)aux[1] + (double)out_bytes * cnt);
      }
      time_end(si);
      timed = true;
      if (last) {
        emit_rows(outb.as<uint32_t>(), cnt, a.ko);
        final_total_ += cnt;
      } else {
        level(si + 1, outb.as<uint32_t>(), cnt);
      }
    }
    if (!timed) time_end(si);
  }
};

// Keeps the first `cap` rows in a host array; later rows are dropped and
// mark the array overflowed (the join goes on and counts them).
struct ArraySink : EmbSink {
  uint32_t *out;
  uint64_t cap, rows = 0;
  bool overflow = false;
  ArraySink(uint32_t *o, uint64_t c) : out(o), cap(c) {}
  // rows that fit are copied from the device to their place in the array
  uint32_t *place(uint64_t n, uint32_t nv) override {
    return overflow || rows + n > cap ? nullptr : out + rows * nv;
  }
  bool put(const uint32_t *r, uint64_t n, uint32_t nv) override {
    if (overflow || rows + n > cap) {
      overflow = true;
      return true;
    }
    if (r != out + rows * nv) std::memcpy(out + rows * nv, r, n * nv * 4);
    rows += n;
    return true;
  }
};

void run_join_sink(gem_ctx *c, const uint32_t *order, uint64_t cap, JoinOut *out, gem_step_log *log,
                   EmbSink *sink) {
  QueryDev &Qd = c->q;
  if (!Qd.tabled) throw Error{GEM_E_STATE, "edge tables have not been built"};
  gemh::JoinPlan plan;
  if (gemh::make_join_plan(Qd.Q, order, &plan)) throw Error{GEM_E_INVALID, "edge order is not a connected order"};
  hipStream_t s = c->stream;
  GEM_HIP_CHECK(hipEventRecord(c->ev[4], s));
  JoinRunner jr(c, plan, sink ? 0 : cap, log, sink);
  jr.first_edge_ = plan.first_edge;
  jr.run(out);
  GEM_HIP_CHECK(hipEventRecord(c->ev[5], s));
  GEM_HIP_CHECK(hipStreamSynchronize(s));
  float ms = 0;
  GEM_HIP_CHECK(hipEventElapsedTime(&ms, c->ev[4], c->ev[5]));
  c->times.join_ms = ms;
  settle_times(c);
  prof_flush(c);
}

void run_join(gem_ctx *c, const uint32_t *order, uint64_t cap, JoinOut *out, gem_step_log *log, uint32_t *emb_out,
              uint64_t emb_capacity) {
  if (!emb_out) {
    run_join_sink(c, order, cap, out, log, nullptr);
    return;
  }
  ArraySink sink(emb_out, emb_capacity);
  run_join_sink(c, order, cap, out, log, &sink);
  out->emb_written = sink.overflow ? 0 : sink.rows;
}

}  // namespace gemd
