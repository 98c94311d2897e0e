// Edge-candidate tables (the reference's construct_edge_candidates,
// in-core/lib/structure/src/unifiedTrie.cu:1020-1391 with kernels
// construct_kernel.cu:1183-1340; CPU form out-of-core/.../unifiedTrie.cu:1224-1427).
//
// For every query vertex u that is not a leaf and every query neighbour u_j of
// u, table T_{u->u_j} has one row per v in Can(u) (row i <-> Can(u)[i]) holding
// the neighbours w of v with w in Can(u_j), in adjacency order.  Values are
// stored as positions of w in Can(u_j) (pos = rank in u_j's candidate bitmap),
// so join rows carry positions and never need a hash probe.
//
// One pass over adjacency serves all of u's tables: a wave takes 64
// consecutive candidates of one u, flattens their adjacency lists into one
// item range (wave scan of degrees) and walks it 64 items per group; item ->
// row by binary lifting over the 64 row starts in LDS; membership of w in each
// Can(u_j) is one bit of u_j's bitmap (L2-resident), looked up only where w's
// label (one byte per adjacency slot, GraphDev::nbr_lab) is u_j's; per-row
// counts and in-row ranks come from ballots restricted to the row's lane
// segment, with one carried count for the row that spans two groups.  Count
// pass -> per-table exclusive scan -> write pass; candidates of degree above
// TABLE_HEAVY_ROW are walked in pieces of TABLE_CHUNK slots by other waves.
// The count pass hands out the pieces itself, so that nothing between the
// parameters' upload and the table sizes waits for the host.  Tables of a
// 16-vertex query on the 2^22-vertex R-MAT graph: 0.43 ms of kernels, against
// 1.42 with a bitmap word per neighbour and table, two numbering atomics a wave
// and one-block scans.
#include "ctx.h"
#include "wave.h"

namespace gemd {

constexpr uint32_t TAB_WAVES = 4;

// Candidates a wave of k_tables takes: a list of 64 rows of up to 256 slots is
// walked in up to 128 dependent steps, so builds of few candidates take fewer
// rows per wave until the chip has waves enough (about 8 per SIMD, twice).  64
// rows per wave: 68 us a pass for queries of a few thousand candidates on 2^18;
// on 2^22 (4 * 10^5 candidates) count / write passes of 119 / 136 us with two groups of 64
// slots a step and 8192 waves enough, 111 / 114 with 16384, 101 / 117 with four.
constexpr uint32_t MIN_ROWS = 8, ENOUGH_WAVES = 16384, STEP = 4;

struct TableJob {
  uint32_t nu;
  uint32_t W;
  uint32_t rows;  // candidates per wave
  uint32_t wave_start[GEM_MAX_QV + 1];
  uint32_t ncan[GEM_MAX_QV];
  uint64_t can_off[GEM_MAX_QV];
  uint32_t nd[GEM_MAX_QV];    // tables keyed on this u
  uint32_t tab0[GEM_MAX_QV];  // first entry in the TableDesc list
};

struct TableDesc {
  uint32_t val_u;
  uint32_t lab;  // dense label of val_u
  uint64_t *off;
  uint32_t *val;
};

// A heavy row: candidate i of the ju-th keyed vertex, its pieces [c0, c0 + n).
struct HeavyTab {
  uint32_t ju, i, c0, n;
};

// Device counters of one build (uploaded as zeros with the descriptors).
struct TableCtr {
  unsigned long long rows_pieces;  // heavy rows (low word) and their pieces
};

// The graph as the table kernels read it.
struct TableGraph {
  const uint64_t *off;
  const uint32_t *nbr;
  const uint8_t *nl;  // labels of the adjacency slots (NL)
};

__device__ __forceinline__ uint64_t lane_range(uint32_t a, uint32_t b) {  // bits [a, b], a <= b < 64
  const uint64_t hi = (b >= 63) ? ~0ull : ((1ull << (b + 1)) - 1);
  return hi & ~((1ull << a) - 1);
}

// Is neighbour wv (label lw, when known) to be looked up in a table whose
// value vertex has label lab?
template <bool NL>
__device__ __forceinline__ bool wanted(bool iv, uint32_t lw, uint32_t lab) {
  return iv && (!NL || lw == lab);
}

template <bool WRITE, bool NL>
__global__ void __launch_bounds__(TAB_WAVES * 64)
k_tables(const TableGraph G, const uint32_t *__restrict__ can, const uint64_t *__restrict__ bitmap,
         const uint32_t *__restrict__ rank, const TableJob job, const TableDesc *__restrict__ desc,
         TableCtr *__restrict__ ctr, HeavyTab *__restrict__ heavy, uint32_t *__restrict__ piece_row) {
  __shared__ uint32_t st[TAB_WAVES][65];
  __shared__ uint64_t ob[TAB_WAVES][64];
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint32_t gw = blockIdx.x * TAB_WAVES + w;
  uint32_t ju = 0;
  while (ju + 1 < job.nu && job.wave_start[ju + 1] <= gw) ++ju;
  const uint32_t row_base = (gw - job.wave_start[ju]) * job.rows;
  const uint32_t ncan = job.ncan[ju];
  const uint32_t i = row_base + l;
  const bool valid = l < job.rows && i < ncan;
  uint64_t o0 = 0;
  uint32_t len = 0, full_len = 0;
  if (valid) {
    const uint32_t v = can[job.can_off[ju] + i];
    o0 = G.off[v];
    full_len = (uint32_t)(G.off[v + 1] - o0);
    len = full_len > TABLE_HEAVY_ROW ? 0u : full_len;
  }
  if (!WRITE) {
    // One atomic a block numbers its heavy rows and their pieces (two a wave
    // were 12,400 on one address, the 240 us of a pass over 4 * 10^5 candidates).
    __shared__ uint32_t wrows[TAB_WAVES], wpieces[TAB_WAVES];
    __shared__ unsigned long long first;
    const uint64_t hv = __ballot(full_len > TABLE_HEAVY_ROW);
    const uint32_t n = full_len > TABLE_HEAVY_ROW ? (full_len + TABLE_CHUNK - 1) / TABLE_CHUNK : 0;
    const uint32_t incl = wave_incl_scan_u32(n);
    if (l == 63) {
      wrows[w] = (uint32_t)__popcll(hv);
      wpieces[w] = incl;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long sum = 0;
      for (uint32_t x = 0; x < TAB_WAVES; ++x) sum += (unsigned long long)wpieces[x] << 32 | wrows[x];
      first = sum ? atomicAdd(&ctr->rows_pieces, sum) : 0;
    }
    __syncthreads();
    if (hv) {
      uint32_t r = (uint32_t)first + rank_below(hv), c = (uint32_t)(first >> 32) + incl - n;
      for (uint32_t x = 0; x < w; ++x) {
        r += wrows[x];
        c += wpieces[x];
      }
      if (n) heavy[r] = HeavyTab{ju, i, c, n};
      for (uint32_t x = 0; x < n; ++x) piece_row[c + x] = r;
    }
  }
  const uint32_t incl = wave_incl_scan_u32(len);
  const uint32_t total = readlane_u32(incl, 63);
  st[w][l] = incl - len;
  ob[w][l] = o0;
  if (l == 63) st[w][64] = total;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const uint32_t nd = job.nd[ju], t0 = job.tab0[ju];
  if (!WRITE && valid && full_len == 0)
    for (uint32_t j = 0; j < nd; ++j) desc[t0 + j].off[i] = 0;
  const uint32_t W = job.W;
  // lane j < nd holds table j: value vertex and its label, row offsets, values
  uint32_t my_vu = 0, my_lab = 0;
  uint64_t my_off = 0, my_val = 0;
  if (l < nd) {
    const TableDesc d = desc[t0 + l];
    my_vu = d.val_u;
    my_lab = d.lab;
    my_off = reinterpret_cast<uint64_t>(d.off);
    my_val = reinterpret_cast<uint64_t>(d.val);
  }
  uint32_t carry_reg = 0;  // lane j: hits of the row carried into the next group, table j
  // One 64-item group of the flattened adjacency: the lane's row, its value
  // and label, and the lane range of its row inside the group.
  struct Grp {
    bool iv, row_done;
    uint32_t row, wv, lw, last, row0, seg_hi;
    uint64_t seg_mask, below_mask;
  };
  auto group = [&](uint32_t t) {
    Grp g;
    const uint32_t item = t + l;
    g.iv = item < total;
    g.row = g.iv ? seg_of(st[w], item) : 63;
    const uint32_t rs = st[w][g.row], re = st[w][g.row + 1];
    const uint64_t at = ob[w][g.row] + (item - rs);
    g.wv = g.iv ? G.nbr[at] : 0;
    g.lw = NL && g.iv ? G.nl[at] : 0;
    g.last = t < total ? min(63u, total - 1 - t) : 0;
    g.row0 = readlane_u32(g.row, 0);
    const uint32_t seg_lo = rs > t ? rs - t : 0;
    g.seg_hi = (re < t + 64 ? re - t : 64) - 1;
    g.row_done = re <= t + 64;
    g.seg_mask = g.iv ? lane_range(seg_lo, g.seg_hi) : 0;
    g.below_mask = g.iv ? (lane_range(seg_lo, l) & ~(1ull << l)) : 0;
    return g;
  };
  // table j over one group, `carry` = the row's hits before the group; returns
  // the hits carried into the next group
  auto apply = [&](const Grp &g, uint32_t j, uint32_t vu, uint64_t word, uint32_t carry) {
    const bool hit = (word >> (g.wv & 63)) & 1ull;
    const uint64_t m = __ballot(hit);
    const uint32_t before = (g.row == g.row0) ? carry : 0;
    const uint32_t tot_row = before + (uint32_t)__popcll(m & g.seg_mask);
    uint64_t *off = reinterpret_cast<uint64_t *>(readlane_u64(my_off, j));
    if (WRITE) {
      if (hit) {
        uint32_t *val = reinterpret_cast<uint32_t *>(readlane_u64(my_val, j));
        const uint32_t r = before + (uint32_t)__popcll(m & g.below_mask);
        const uint32_t p = rank[(uint64_t)vu * (W + 1) + (g.wv >> 6)] +
                           (uint32_t)__popcll(word & ((1ull << (g.wv & 63)) - 1));
        stg(val + ldg(off + row_base + g.row) + r, p);
      }
    } else {
      if (g.iv && l == g.seg_hi && g.row_done) stg(off + row_base + g.row, (uint64_t)tot_row);
    }
    return readlane_u32(g.row_done ? 0u : tot_row, g.last);
  };
  // STEP groups per step: all their loads are in flight before the first
  // group's ballots
  for (uint32_t t = 0; t < total; t += 64 * STEP) {
    Grp g[STEP];
#pragma unroll
    for (uint32_t x = 0; x < STEP; ++x) g[x] = group(t + 64 * x);
    for (uint32_t j = 0; j < nd; ++j) {
      const uint32_t vu = readlane_u32(my_vu, j), lab = readlane_u32(my_lab, j);
      const uint64_t *bm = bitmap + (uint64_t)vu * W;
      uint64_t word[STEP];
#pragma unroll
      for (uint32_t x = 0; x < STEP; ++x) word[x] = wanted<NL>(g[x].iv, g[x].lw, lab) ? bm[g[x].wv >> 6] : 0;
      uint32_t carry = readlane_u32(carry_reg, j);
#pragma unroll
      for (uint32_t x = 0; x < STEP; ++x)
        if (t + 64 * x < total) carry = apply(g[x], j, vu, word[x], carry);
      if (l == j) carry_reg = carry;
    }
  }
}

// Persistent grid over the heavy rows' pieces; lane j carries table j's
// running count.  The count pass stores each piece's hits per table
// (ccnt[piece * ndmax + j]); k_theavy_bases turns those into each piece's
// offset inside its row and writes the rows' totals; the write pass starts
// each piece's hits at that offset, so values stay in adjacency order.  Four
// groups of 64 slots per step: their loads, and then the bitmap words of each
// table for the slots of its label, are in flight together.
template <bool WRITE, bool NL>
__global__ void __launch_bounds__(TAB_WAVES * 64)
k_tables_heavy(const TableGraph G, const uint32_t *__restrict__ can, const uint64_t *__restrict__ bitmap,
               const uint32_t *__restrict__ rank, const TableJob job, const TableDesc *__restrict__ desc,
               TableCtr *__restrict__ ctr, const HeavyTab *__restrict__ heavy, const uint32_t *__restrict__ piece_row,
               uint32_t *__restrict__ ccnt, uint32_t ndmax) {
  constexpr int GR = 4;
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint32_t W = job.W, pieces = (uint32_t)(ctr->rows_pieces >> 32);
  for (uint32_t c = blockIdx.x * TAB_WAVES + w; c < pieces; c += gridDim.x * TAB_WAVES) {
    const HeavyTab e = heavy[piece_row[c]];
    const uint32_t v = can[job.can_off[e.ju] + e.i];
    const uint64_t o0 = G.off[v], len = G.off[v + 1] - o0;
    const uint64_t t0 = (uint64_t)(c - e.c0) * TABLE_CHUNK, t1 = t0 + TABLE_CHUNK < len ? t0 + TABLE_CHUNK : len;
    const uint32_t nd = job.nd[e.ju], tb = job.tab0[e.ju];
    // lane j < nd holds table j: its value vertex and label, (write) the
    // address of the row's first value, and its running count in the row
    uint32_t my_vu = 0, my_lab = 0, run_reg = 0;
    uint64_t my_dst = 0;
    if (l < nd) {
      const TableDesc d = desc[tb + l];
      my_vu = d.val_u;
      my_lab = d.lab;
      if (WRITE) {
        my_dst = reinterpret_cast<uint64_t>(d.val + d.off[e.i]);
        run_reg = ccnt[(uint64_t)c * ndmax + l];
      }
    }
    for (uint64_t t = t0; t < t1; t += 64 * GR) {
      uint32_t wv[GR], lw[GR];
      bool iv[GR];
#pragma unroll
      for (int g = 0; g < GR; ++g) {
        const uint64_t x = t + 64 * g + l;
        iv[g] = x < t1;
        wv[g] = iv[g] ? G.nbr[o0 + x] : 0;
        lw[g] = NL && iv[g] ? G.nl[o0 + x] : 0;
      }
      for (uint32_t j = 0; j < nd; ++j) {
        const uint32_t vu = readlane_u32(my_vu, j), lab = readlane_u32(my_lab, j);
        const uint64_t *bm = bitmap + (uint64_t)vu * W;
        const uint32_t *rk = rank + (uint64_t)vu * (W + 1);
        uint64_t word[GR];
        uint32_t r[GR];
#pragma unroll
        for (int g = 0; g < GR; ++g) {
          const bool want = wanted<NL>(iv[g], lw[g], lab);
          word[g] = want ? bm[wv[g] >> 6] : 0;
          if (WRITE) r[g] = want ? rk[wv[g] >> 6] : 0;
        }
        uint32_t run = readlane_u32(run_reg, j);
        uint32_t *dst = reinterpret_cast<uint32_t *>(readlane_u64(my_dst, j));
#pragma unroll
        for (int g = 0; g < GR; ++g) {
          const bool hit = (word[g] >> (wv[g] & 63)) & 1ull;
          const uint64_t m = __ballot(hit);
          if (WRITE && hit)
            stg(dst + run + rank_below(m), r[g] + (uint32_t)__popcll(word[g] & ((1ull << (wv[g] & 63)) - 1)));
          run += (uint32_t)__popcll(m);
        }
        if (l == j) run_reg = run;
      }
    }
    if (!WRITE && l < nd) ccnt[(uint64_t)c * ndmax + l] = run_reg;
  }
}

// One thread per (heavy row, table slot): piece counts -> piece offsets inside
// the row, and the row's total as its count.
__global__ void __launch_bounds__(256) k_theavy_bases(const TableJob job, const TableDesc *__restrict__ desc,
                                                     const TableCtr *__restrict__ ctr,
                                                     const HeavyTab *__restrict__ heavy, uint32_t *__restrict__ ccnt,
                                                     uint32_t ndmax) {
  const uint64_t n = (uint64_t)(uint32_t)ctr->rows_pieces * ndmax;
  for (uint64_t x = (uint64_t)blockIdx.x * 256 + threadIdx.x; x < n; x += (uint64_t)gridDim.x * 256) {
    const HeavyTab e = heavy[x / ndmax];
    const uint32_t j = (uint32_t)(x % ndmax);
    if (j >= job.nd[e.ju]) continue;
    uint32_t run = 0;
    for (uint32_t c = 0; c < e.n; c += 8) {  // eight loads in flight
      uint32_t h[8];
      uint32_t *at = ccnt + (uint64_t)(e.c0 + c) * ndmax + j;
#pragma unroll
      for (uint32_t x = 0; x < 8; ++x) h[x] = c + x < e.n ? at[x * ndmax] : 0;
#pragma unroll
      for (uint32_t x = 0; x < 8; ++x) {
        if (c + x < e.n) at[x * ndmax] = run;
        run += h[x];
      }
    }
    stg(desc[job.tab0[e.ju] + j].off + e.i, (uint64_t)run);
  }
}

void run_tables(gem_ctx *c) { run_tables(c, c->q, true); }

// The launches over the build's parameters; passes by `write`.
struct TableRun {
  gem_ctx *c;
  const GraphDev &G;
  QueryDev &Qd;
  TableJob job{};
  uint32_t waves = 0, ndmax = 1;
  uint64_t rows_bound = 0, pieces_bound = 0;  // heavy rows and pieces there can be
  DevBuf heavy, piece_row, ccnt;
  TableDesc *desc = nullptr;
  TableCtr *ctr = nullptr;
  std::vector<uint32_t> desc_tab;  // TableDesc index -> directed edge

  template <bool WRITE, bool NL>
  void pass_as() {
    hipStream_t s = c->stream;
    const TableGraph g{G.off.as<uint64_t>(), G.nbr_dev(), G.nbr_lab.as<uint8_t>()};
    if (waves) {
      k_tables<WRITE, NL><<<(waves + TAB_WAVES - 1) / TAB_WAVES, TAB_WAVES * 64, 0, s>>>(
          g, Qd.can.as<uint32_t>(), Qd.bitmap.as<uint64_t>(), Qd.rank.as<uint32_t>(), job, desc, ctr,
          heavy.as<HeavyTab>(), piece_row.as<uint32_t>());
      GEM_LAUNCH_CHECK("k_tables");
    }
    if (waves && rows_bound) {
      const uint32_t hb = (uint32_t)std::min<uint64_t>((pieces_bound + TAB_WAVES - 1) / TAB_WAVES, 2048);
      k_tables_heavy<WRITE, NL><<<hb, TAB_WAVES * 64, 0, s>>>(
          g, Qd.can.as<uint32_t>(), Qd.bitmap.as<uint64_t>(), Qd.rank.as<uint32_t>(), job, desc, ctr,
          heavy.as<HeavyTab>(), piece_row.as<uint32_t>(), ccnt.as<uint32_t>(), ndmax);
      GEM_LAUNCH_CHECK("k_tables_heavy");
      if (!WRITE) {
        k_theavy_bases<<<(uint32_t)std::min<uint64_t>((rows_bound * ndmax + 255) / 256, 1024), 256, 0, s>>>(
            job, desc, ctr, heavy.as<HeavyTab>(), ccnt.as<uint32_t>(), ndmax);
        GEM_LAUNCH_CHECK("k_theavy_bases");
      }
    }
  }
  void pass(bool write) {
    ProfLaunch pl(c, write ? K_TABLES_WRITE : K_TABLES_COUNT);
    if (G.nbr_lab.p)
      write ? pass_as<true, true>() : pass_as<false, true>();
    else
      write ? pass_as<true, false>() : pass_as<false, false>();
  }
};

// Sum of the degrees of n vertices (for the algorithmic bytes, while profiling;
// counted by the build itself it is an atomic a wave and heavy piece, which
// were half of a profiled count pass).
__global__ void __launch_bounds__(256) k_degree_sum(const uint64_t *__restrict__ off, const uint32_t *__restrict__ v,
                                                   uint32_t n, unsigned long long *__restrict__ out) {
  __shared__ uint64_t sm[4];
  uint64_t x = 0;
  for (uint32_t i = threadIdx.x; i < n; i += 256) x += off[v[i] + 1] - off[v[i]];
  x = wave_sum_u64(x);
  if (threadIdx.x % 64 == 0) sm[threadIdx.x / 64] = x;
  __syncthreads();
  if (threadIdx.x == 0) *out = sm[0] + sm[1] + sm[2] + sm[3];
}
static uint64_t degree_sum(gem_ctx *c, const GraphDev &G, const uint32_t *v, uint32_t n) {
  DevBuf d;
  d.alloc(8, c->stream);
  k_degree_sum<<<1, 256, 0, c->stream>>>(G.off.as<uint64_t>(), v, n, d.as<unsigned long long>());
  GEM_LAUNCH_CHECK("k_degree_sum");
  uint64_t h = 0;
  GEM_HIP_CHECK(hipMemcpyAsync(&h, d.p, 8, hipMemcpyDeviceToHost, c->stream));
  GEM_HIP_CHECK(hipStreamSynchronize(c->stream));
  return h;
}

// The tables of Qd's query, without their values, and its launches' sizes.
static void plan_tables(TableRun &R) {
  const gemh::QueryInfo &Q = R.Qd.Q;
  const GraphDev &G = R.G;
  QueryDev &Qd = R.Qd;
  Qd.tab.clear();
  Qd.tab.resize(2 * Q.ne);
  TableJob &job = R.job;
  job.W = Qd.W;
  for (uint32_t u = 0; u < Q.nv; ++u) {
    if (Q.deg[u] == 1) continue;  // leaves key no table (unifiedTrie.cu:1045,1095)
    const uint32_t ju = job.nu++;
    job.ncan[ju] = Qd.ncan[u];
    job.can_off[ju] = Qd.can_off[u];
    job.tab0[ju] = (uint32_t)R.desc_tab.size();
    for (auto [un, e] : Q.adj[u]) {
      const uint32_t d = 2 * e + (Q.edges[e].first == u ? 0 : 1);
      TableDev &T = Qd.tab[d];
      T.present = true;
      T.key_u = u;
      T.val_u = un;
      T.off.alloc(((uint64_t)Qd.ncan[u] + 1) * 8, R.c->stream);
      R.desc_tab.push_back(d);
      job.nd[ju]++;
    }
    R.ndmax = std::max(R.ndmax, job.nd[ju]);
    auto it = G.label_id.find(Q.lab[u]);
    if (it != G.label_id.end()) {
      R.rows_bound += std::min<uint64_t>(G.label_long[it->second], Qd.ncan[u]);
      R.pieces_bound += G.label_chunks[it->second];
    }
  }
  for (job.rows = 64;; job.rows /= 2) {
    R.waves = 0;
    for (uint32_t ju = 0; ju < job.nu; ++ju) {
      job.wave_start[ju] = R.waves;
      R.waves += (job.ncan[ju] + job.rows - 1) / job.rows;
    }
    if (job.rows == MIN_ROWS || R.waves >= ENOUGH_WAVES / 2) break;
  }
  job.wave_start[job.nu] = R.waves;
}

void run_tables(gem_ctx *c, QueryDev &Qd, bool wait) { run_tables(c, &Qd, 1, wait); }

void run_tables(gem_ctx *c, QueryDev *Qds, uint32_t n, bool wait) {
  const GraphDev &G = graph(c);
  hipStream_t s = c->stream;
  for (uint32_t i = 0; i < n; ++i)
    if (!Qds[i].filtered) throw Error{GEM_E_STATE, "filter has not run"};
  GEM_HIP_CHECK(hipEventRecord(c->ev[2], s));
  std::vector<TableRun> runs;
  runs.reserve(n);
  size_t nt = 0;
  for (uint32_t i = 0; i < n; ++i) {
    runs.push_back(TableRun{c, G, Qds[i]});
    plan_tables(runs.back());
    nt += runs.back().desc_tab.size();
  }
  // Parameters of the builds: one staging block, one device block: the tables,
  // the scan segments (and, before them on the host, the sizes that the scan
  // writes), the counters.
  const size_t at_seg = nt * sizeof(TableDesc), at_ctr = at_seg + nt * sizeof(ScanSeg);
  const size_t bytes = at_ctr + n * sizeof(TableCtr);
  uint64_t *sizes = pinned<uint64_t>(c, nt + (bytes + 7) / 8);
  unsigned char *stage = reinterpret_cast<unsigned char *>(sizes + nt);
  TableDesc *hdesc = reinterpret_cast<TableDesc *>(stage);
  ScanSeg *hseg = reinterpret_cast<ScanSeg *>(stage + at_seg);
  DevBuf params;
  params.alloc(bytes, s);
  unsigned char *dev = params.as<unsigned char>();
  uint32_t chunks = 0;
  size_t k = 0;
  for (uint32_t i = 0; i < n; ++i) {
    TableRun &R = runs[i];
    R.desc = reinterpret_cast<TableDesc *>(dev) + k;
    R.ctr = reinterpret_cast<TableCtr *>(dev + at_ctr) + i;
    for (uint32_t d : R.desc_tab) {
      const TableDev &T = R.Qd.tab[d];
      auto it = G.label_id.find(R.Qd.Q.lab[T.val_u]);
      hdesc[k] = TableDesc{T.val_u, it == G.label_id.end() ? ~0u : it->second, T.off.as<uint64_t>(), nullptr};
      hseg[k] = ScanSeg{T.off.as<uint64_t>(), (uint64_t)R.Qd.ncan[T.key_u], chunks};
      chunks += scan_chunks(R.Qd.ncan[T.key_u]);
      ++k;
    }
    reinterpret_cast<TableCtr *>(stage + at_ctr)[i] = TableCtr{};
  }
  GEM_HIP_CHECK(hipMemcpyAsync(dev, stage, bytes, hipMemcpyHostToDevice, s));
  for (TableRun &R : runs) {
    if (R.rows_bound) {
      R.heavy.alloc(R.rows_bound * sizeof(HeavyTab), s);
      R.piece_row.alloc(R.pieces_bound * 4, s);
      R.ccnt.alloc(R.pieces_bound * R.ndmax * 4, s);
    }
    R.pass(false);
  }
  // row counts -> offsets of every table, the sizes straight to the host
  scan_segments_u64(c, reinterpret_cast<ScanSeg *>(dev + at_seg), (uint32_t)nt, chunks, pinned_dev(c, sizes));
  GEM_HIP_CHECK(hipStreamSynchronize(s));
  k = 0;
  for (TableRun &R : runs) {
    const size_t k0 = k;
    for (uint32_t d : R.desc_tab) {
      TableDev &T = R.Qd.tab[d];
      T.size = sizes[k];
      T.val.alloc(std::max<uint64_t>(T.size, 1) * 4, s);
      hdesc[k++].val = T.val.as<uint32_t>();
    }
    if (c->prof.on) {
      // algorithmic bytes: per keyed u, its candidates (4 B), offset pairs (8 B)
      // and adjacency (4 B per slot) once for all its tables; per table the value
      // vertex's bitmap (|V|/8) and the row counts / offsets (8 B per row)
      const TableJob &job = R.job;
      const QueryDev &Qd = R.Qd;
      double shared_bytes = 0, count_bytes = 0, write_bytes = 0;
      for (uint32_t ju = 0; ju < job.nu; ++ju)
        shared_bytes += 12.0 * job.ncan[ju] +
                        4.0 * (double)degree_sum(c, G, Qd.can.as<uint32_t>() + job.can_off[ju], job.ncan[ju]);
      for (size_t x = k0; x < k; ++x) {
        const TableDev &T = Qd.tab[R.desc_tab[x - k0]];
        count_bytes += 8.0 * Qd.W + 8.0 * Qd.ncan[T.key_u];
        write_bytes += 12.0 * Qd.W + 8.0 * Qd.ncan[T.key_u] + 4.0 * (double)T.size;
      }
      prof_bytes(c, K_TABLES_COUNT, shared_bytes + count_bytes);
      prof_bytes(c, K_TABLES_WRITE, shared_bytes + write_bytes);
    }
  }
  GEM_HIP_CHECK(hipMemcpyAsync(dev, stage, nt * sizeof(TableDesc), hipMemcpyHostToDevice, s));
  for (TableRun &R : runs) {
    R.pass(true);
    R.Qd.tabled = true;
  }
  GEM_HIP_CHECK(hipEventRecord(c->ev[3], s));
  c->tables_timed = true;
  if (wait || c->prof.on) {
    GEM_HIP_CHECK(hipStreamSynchronize(s));
    prof_flush(c);
    settle_times(c);
  }
}

}  // namespace gemd
