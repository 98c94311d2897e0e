// Candidate filter and position index.
//
// Predicate (out-of-core/lib/filter/src/filter.cu:160-240; in-core
// filter_kernel.cu:198-265): v is a candidate of query vertex u iff
//   lab(v) == lab(u),  deg(u) <= deg(v) + T,
//   sum over query labels l of max(0, nlc_u[l] - nlc_v[l]) <= T,
// where nlc_x[l] counts neighbours of x with label l, over labels present in
// the query.
//
// Layout: one wave owns a tile of 64 consecutive data vertices (lane = vertex)
// and writes, for every query vertex u, one 64-bit word of u's candidate bitmap
// (ballot of the lanes that pass).  A per-u scan of the words' popcounts gives
// rank[u][tile] = #candidates before the tile, so
//   pos_u(v) = rank[u][v/64] + popcount(bitmap[u][v/64] & below(v % 64))
// equals lower_bound(Can(u), v): the value the reference's cuckoo hash returns
// (unifiedTrie.cuh:84-125, unifiedTrie.cu:54-101), in one cache line, with no
// build retries.  The same pass writes Can(u) in ascending order.
//
// Neighbour labels are read as one byte per adjacency slot (GraphDev::nbr_lab,
// made once per data graph): contiguous bytes in place of a neighbour id and a
// gather of its label.  A lane counts its neighbours into an LDS column of its
// own, four 8-bit counts to a word (label slot s: word s / 4, byte s % 4), with
// LDS adds that return nothing.  Vertices of degree <= 64 take one lane, larger
// ones a wave, those past FILTER_HUB_DEG a block; which is which depends on
// the data graph alone, so the two lists are made with it.
// All kernels of a 16-vertex query on the 2^22-vertex R-MAT graph (65 M slots):
// 215 us, against 1,060 with a gather per neighbour, lists made per query and
// one-block scans; k_filter (103 us) reads 100 MB and is bound by the LDS adds
// of its longest lanes, k_filter_heavy (88) by the block of the largest hub.
#include <mutex>
#include <string>

#include "ctx.h"
#include "wave.h"

namespace gemd {

constexpr uint32_t FILTER_WAVES = 4, HEAVY_WAVES = 8;
constexpr uint32_t HIST_WORDS = GEM_MAX_QV / 4 + 1;  // the last word takes labels outside the query
constexpr uint32_t OUT_SLOT = GEM_MAX_QV;

// The query and, for byte labels, its label -> slot table, as a kernel argument.
struct FilterArgs {
  FilterQuery fq;
  uint8_t slot_of[256];
};

// Query and slot table in LDS.
struct FilterLds {
  FilterQuery fq;
  uint8_t tab[256];
};
__device__ __forceinline__ void load_args(const FilterArgs &a, FilterLds &s) {
  static_assert(sizeof(FilterArgs) % 4 == 0 && sizeof(FilterLds) == sizeof(FilterArgs), "copied by words");
  const uint32_t *src = reinterpret_cast<const uint32_t *>(&a);
  uint32_t *dst = reinterpret_cast<uint32_t *>(&s);
  for (uint32_t i = threadIdx.x; i < sizeof(FilterArgs) / 4; i += blockDim.x) dst[i] = src[i];
  __syncthreads();
}

// The graph as the filter reads it.  nl (NL): labels of the adjacency slots,
// readable to 16 bytes past the last; slot_of (LabT = u32): label -> slot.
template <class LabT>
struct FilterGraph {
  const uint64_t *off;
  const uint32_t *nbr;
  const uint8_t *nl;
  const LabT *lab;
  const uint8_t *slot_of;
  uint32_t n;
};
template <class LabT>
__device__ __forceinline__ uint32_t label_slot(const FilterGraph<LabT> &G, const FilterLds &A, LabT x) {
  const uint32_t s = sizeof(LabT) == 1 ? A.tab[x] : G.slot_of[x];
  return s == NO_SLOT ? OUT_SLOT : s;
}

typedef uint64_t u64u __attribute__((aligned(1)));

// Adds adjacency slots j, j + step, ... < end to the lane's column: 8 slots
// at a time (NL; j and step are then in units of slots but multiples of 8
// from the list's start), or one neighbour's label at a time.
template <class LabT, bool NL>
__device__ __forceinline__ void count_slots(const FilterGraph<LabT> &G, const FilterLds &A, uint64_t o0, uint64_t j,
                                            uint64_t end, uint64_t step, uint32_t *col, uint32_t stride) {
  auto add = [&](uint32_t s) { atomicAdd(&col[(s >> 2) * stride], 1u << ((s & 3) * 8)); };
  for (; j < end; j += step) {
    if (NL) {
      const uint64_t x = *reinterpret_cast<const u64u *>(G.nl + o0 + j);
      const uint32_t m = end - j < 8 ? (uint32_t)(end - j) : 8;
#pragma unroll
      for (uint32_t b = 0; b < 8; ++b) {
        const uint32_t s = A.tab[(x >> (8 * b)) & 0xFF];
        add(b < m && s != NO_SLOT ? s : OUT_SLOT);
      }
    } else {
      add(label_slot(G, A, G.lab[G.nbr[o0 + j]]));
    }
  }
}

// Tiles of 64 vertices, those of degree <= FILTER_LIGHT_DEG counted here.
template <class LabT, bool NL>
__global__ void __launch_bounds__(FILTER_WAVES * 64)
k_filter(const FilterGraph<LabT> G, const FilterArgs args, uint64_t *__restrict__ bitmap) {
  __shared__ FilterLds A;
  __shared__ uint32_t hist[FILTER_WAVES][HIST_WORDS][64];
  load_args(args, A);
  const FilterQuery &fq = A.fq;
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint32_t T = fq.T, W = fq.W, nw = (fq.nslots + 3) / 4;
  uint32_t *col = &hist[w][0][l];
  for (uint32_t tile = blockIdx.x * FILTER_WAVES + w; tile < W; tile += gridDim.x * FILTER_WAVES) {
    const uint64_t v = (uint64_t)tile * 64 + l;
    uint64_t o0 = 0, deg = 0;
    uint32_t cmask = 0, pass = 0;
    if (v < G.n) {
      const uint32_t slot = label_slot(G, A, G.lab[v]);
      if (slot != OUT_SLOT) {
        o0 = G.off[v];
        deg = G.off[v + 1] - o0;
        uint32_t g = deg <= FILTER_LIGHT_DEG ? fq.group[slot] : 0;
        while (g) {
          const uint32_t u = __builtin_ctz(g);
          g &= g - 1;
          if ((uint64_t)fq.qdeg[u] <= deg + T) cmask |= 1u << u;
        }
      }
    }
    if (cmask) {
      for (uint32_t s = 0; s < nw; ++s) col[s * 64] = 0;
      count_slots<LabT, NL>(G, A, o0, 0, deg, NL ? 8 : 1, col, 64);
      uint32_t g = cmask;
      while (g) {
        const uint32_t u = __builtin_ctz(g);
        g &= g - 1;
        uint32_t deficit = 0;
        for (uint32_t r = 0; r < fq.nreq[u]; ++r) {
          const uint32_t need = fq.req_cnt[u][r], s = fq.req_slot[u][r];
          const uint32_t have = (col[(s >> 2) * 64] >> ((s & 3) * 8)) & 0xFF;
          deficit += need > have ? need - have : 0;
        }
        if (deficit <= T) pass |= 1u << u;
      }
    }
    uint64_t mine = 0;  // lane u: u's word
    for (uint32_t u = 0; u < fq.nv; ++u) {
      const uint64_t m = __ballot((pass >> u) & 1u);
      if (l == u) mine = m;
    }
    if (l < fq.nv) bitmap[(uint64_t)l * W + tile] = mine;
  }
}

// Label counts of a wave's columns (each lane's at most 255): cnt[s] += the
// sum over lanes; the columns are cleared.
__device__ __forceinline__ void sum_columns(uint32_t *col, uint32_t nslots, uint32_t l, uint32_t *cnt) {
  for (uint32_t w = 0; w < (nslots + 3) / 4; ++w) {
    uint32_t e = col[w * 64] & 0x00FF00FFu, o = (col[w * 64] >> 8) & 0x00FF00FFu;
    col[w * 64] = 0;
#pragma unroll
    for (uint32_t d = 32; d >= 1; d >>= 1) {
      e += __shfl_xor(e, d, 64);
      o += __shfl_xor(o, d, 64);
    }
    // slots 4 w ...: e low, o low, e high, o high
    const uint32_t x = l & 1 ? o : e, y = l & 2 ? x >> 16 : x & 0xFFFFu;
    if (l < 4 && 4 * w + l < nslots) atomicAdd(&cnt[4 * w + l], y);
  }
}

// Query vertex l's decision for data vertex v of degree deg whose neighbour
// label counts are cnt: lane l sets v's bit.
__device__ __forceinline__ void filter_decide(const FilterQuery &fq, uint32_t l, uint32_t v, uint64_t deg, uint32_t g,
                                              const uint32_t *cnt, unsigned long long *bitmap) {
  if (l < fq.nv && ((g >> l) & 1u) && (uint64_t)fq.qdeg[l] <= deg + fq.T) {
    uint32_t deficit = 0;
    for (uint32_t r = 0; r < fq.nreq[l]; ++r) {
      const uint32_t need = fq.req_cnt[l][r], have = cnt[fq.req_slot[l][r]];
      deficit += need > have ? need - have : 0;
    }
    if (deficit <= fq.T) atomicOr(&bitmap[(uint64_t)l * fq.W + (v >> 6)], 1ull << (v & 63));
  }
}

// The graph's vertices past FILTER_LIGHT_DEG, after k_filter wrote the words:
// blocks [0, n_hub) take one hub each (all waves), the waves of the others the
// list of the rest.
template <class LabT, bool NL>
__global__ void __launch_bounds__(HEAVY_WAVES * 64)
k_filter_heavy(const FilterGraph<LabT> G, const FilterArgs args, const uint32_t *__restrict__ heavy, uint32_t n_heavy,
               const uint32_t *__restrict__ hubs, uint32_t n_hub, unsigned long long *__restrict__ bitmap) {
  __shared__ FilterLds A;
  __shared__ uint32_t hist[HEAVY_WAVES][HIST_WORDS][64];
  __shared__ uint32_t cnt[HEAVY_WAVES][GEM_MAX_QV];
  load_args(args, A);
  const FilterQuery &fq = A.fq;
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64, per = NL ? 8 : 1;
  uint32_t *col = &hist[w][0][l];
  for (uint32_t s = 0; s < (fq.nslots + 3) / 4; ++s) col[s * 64] = 0;
  if (l < GEM_MAX_QV) cnt[w][l] = 0;
  __syncthreads();
  if (blockIdx.x < n_hub) {
    const uint32_t v = hubs[blockIdx.x];
    const uint32_t slot = label_slot(G, A, G.lab[v]);
    if (slot == OUT_SLOT) return;
    const uint64_t o0 = G.off[v], deg = G.off[v + 1] - o0;
    // a lane's 8-bit counts hold 248 slots
    const uint64_t round = (uint64_t)HEAVY_WAVES * 64 * 248;
    for (uint64_t j0 = 0; j0 < deg; j0 += round) {
      const uint64_t end = deg - j0 < round ? deg : j0 + round;
      count_slots<LabT, NL>(G, A, o0, j0 + (uint64_t)threadIdx.x * per, end, (uint64_t)HEAVY_WAVES * 64 * per, col, 64);
      sum_columns(col, fq.nslots, l, cnt[0]);
    }
    __syncthreads();
    if (w == 0) filter_decide(fq, l, v, deg, fq.group[slot], cnt[0], bitmap);
    return;
  }
  for (uint32_t i = (blockIdx.x - n_hub) * HEAVY_WAVES + w; i < n_heavy; i += (gridDim.x - n_hub) * HEAVY_WAVES) {
    const uint32_t v = heavy[i];
    const uint32_t slot = label_slot(G, A, G.lab[v]);
    if (slot == OUT_SLOT) continue;
    const uint64_t o0 = G.off[v], deg = G.off[v + 1] - o0;
    count_slots<LabT, NL>(G, A, o0, (uint64_t)l * per, deg, 64 * per, col, 64);
    sum_columns(col, fq.nslots, l, cnt[w]);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    filter_decide(fq, l, v, deg, fq.group[slot], cnt[w], bitmap);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (l < GEM_MAX_QV) cnt[w][l] = 0;
  }
}

// Ranks and candidate lists in chunks of RANK_CHUNK bitmap words: chunk sums
// (left out when one chunk holds all), then each block adds up the sums before
// its own and scans it.  Wave w of a block holds words [w, w + 1) * 1024 of the
// chunk, lane = word modulo 64.  With one block per query vertex scanning all
// words, and a launch of its own for the lists, the ranks of the 2^22-vertex
// graph took 108 us and its lists 63.
constexpr uint32_t RANK_STEPS = 16, RANK_CHUNK = 4 * 64 * RANK_STEPS;

__global__ void __launch_bounds__(256) k_rank_sums(const uint64_t *__restrict__ bitmap, uint32_t W,
                                                  uint32_t *__restrict__ sums) {
  __shared__ uint32_t sm[4];
  const uint32_t u = blockIdx.y, w0 = blockIdx.x * RANK_CHUNK;
  uint32_t x = 0;
#pragma unroll
  for (uint32_t i = 0; i < RANK_STEPS; ++i) {
    const uint32_t word = w0 + i * 256 + threadIdx.x;
    if (word < W) x += (uint32_t)__popcll(bitmap[(uint64_t)u * W + word]);
  }
  x = (uint32_t)wave_sum_u64(x);
  if (threadIdx.x % 64 == 0) sm[threadIdx.x / 64] = x;
  __syncthreads();
  if (threadIdx.x == 0) sums[u * gridDim.x + blockIdx.x] = sm[0] + sm[1] + sm[2] + sm[3];
}

struct CanOffsets {
  uint64_t at[GEM_MAX_QV + 1];
};
// can == null: counts and ranks only.  ncan[u] = |Can(u)| (device or mapped
// host memory).
__global__ void __launch_bounds__(256) k_rank_lists(const uint64_t *__restrict__ bitmap, uint32_t W,
                                                   const uint32_t *__restrict__ sums, uint32_t *__restrict__ rank,
                                                   const CanOffsets can_off, uint32_t *__restrict__ can,
                                                   uint32_t *__restrict__ ncan) {
  __shared__ uint32_t sm[4], before[4];
  const uint32_t u = blockIdx.y, w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint32_t w0 = blockIdx.x * RANK_CHUNK + w * 64 * RANK_STEPS;
  uint64_t m[RANK_STEPS];
  uint32_t x = 0;
#pragma unroll
  for (uint32_t i = 0; i < RANK_STEPS; ++i) {
    const uint32_t word = w0 + i * 64 + l;
    m[i] = word < W ? bitmap[(uint64_t)u * W + word] : 0;
    x += (uint32_t)__popcll(m[i]);
  }
  uint32_t y = 0;  // candidates of the chunks before
  for (uint32_t c = threadIdx.x; c < blockIdx.x; c += 256) y += sums[u * gridDim.x + c];
  x = (uint32_t)wave_sum_u64(x);
  y = (uint32_t)wave_sum_u64(y);
  if (l == 0) {
    sm[w] = x;
    before[w] = y;
  }
  __syncthreads();
  uint32_t run = before[0] + before[1] + before[2] + before[3];
  for (uint32_t i = 0; i < w; ++i) run += sm[i];
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 192) {  // the last wave's first lane
    ncan[u] = run + sm[3];
    rank[(uint64_t)u * (W + 1) + W] = run + sm[3];
  }
  uint32_t *out = can ? can + can_off.at[u] : nullptr;
#pragma unroll
  for (uint32_t i = 0; i < RANK_STEPS; ++i) {
    if (w0 + i * 64 >= W) break;
    const uint32_t word = w0 + i * 64 + l, c = (uint32_t)__popcll(m[i]);
    const uint32_t incl = wave_incl_scan_u32(c);
    uint32_t r = run + incl - c;
    if (word < W) rank[(uint64_t)u * (W + 1) + word] = r;
    if (out)
      for (uint64_t b = m[i]; b; b &= b - 1) out[r++] = word * 64 + (uint32_t)__builtin_ctzll(b);
    run += readlane_u32(incl, 63);
  }
}

// Labels of the adjacency slots (255, no label, for a neighbour out of range).
__global__ void k_slot_labels(const uint32_t *__restrict__ nbr, uint64_t slots, const uint8_t *__restrict__ lab,
                              uint32_t n, uint8_t *__restrict__ nl) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < slots; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t v = nbr[i];
    nl[i] = v < n ? lab[v] : 255;
  }
}

void make_slot_labels(gem_ctx *c, GraphDev &G) {
  if (!G.lab8 || !G.slots) return;
  // A graph works without them (with gathers), so they are left out rather than
  // failing a load: past the context's limit, by default a quarter of the free
  // memory (asked for past 16 MiB: the answer takes 0.7 ms), or when refused.
  const uint64_t bytes = G.slots + 16;
  uint64_t most = c->slot_label_bytes;
  if (most == ~0ull) {
    most = 16ull << 20;
    if (bytes > most) {
      size_t free_b = 0, total_b = 0;
      GEM_HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
      most = std::max<uint64_t>(most, (free_b + pool_reusable_bytes()) / 4);
    }
  }
  if (bytes > most) return;
  try {
    G.nbr_lab.alloc(bytes, c->stream);
  } catch (const Error &e) {
    if (e.code != GEM_E_NOMEM) throw;
    return;
  }
  k_slot_labels<<<(uint32_t)std::min<uint64_t>((G.slots + 255) / 256, 16384), 256, 0, c->stream>>>(
      G.nbr_dev(), G.slots, G.lab.as<uint8_t>(), G.n, G.nbr_lab.as<uint8_t>());
  GEM_LAUNCH_CHECK("k_slot_labels");
}

__global__ void k_position_lookup(const uint64_t *__restrict__ bitmap, const uint32_t *__restrict__ rank, uint32_t W,
                                  uint32_t n, uint32_t u, const uint32_t *__restrict__ vs, uint64_t cnt,
                                  uint32_t *__restrict__ pos) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  const uint32_t v = vs[i];
  uint32_t p = NOT_FOUND;
  if (v < n) {
    const uint64_t m = bitmap[(uint64_t)u * W + (v >> 6)];
    const uint32_t b = v & 63;
    if (m >> b & 1ull) p = rank[(uint64_t)u * (W + 1) + (v >> 6)] + (uint32_t)__popcll(m & ((1ull << b) - 1));
  }
  pos[i] = p;
}

// Device buffers of one filter run (library-owned, or carved from the
// no-allocation scratch array).
struct FilterBufs {
  const uint8_t *slot_of = nullptr;  // label -> slot, when labels are not bytes
  uint64_t *bitmap = nullptr;        // u64[nv * W]
  uint32_t *sums = nullptr;          // u32[nv * chunks]
  uint32_t *rank = nullptr;          // u32[nv * (W + 1)]
  uint32_t *can = nullptr;           // candidate lists at can_off[u]
  uint32_t *ncan = nullptr;          // u32[nv]
};

// Host side of a filter run: the query's label slots and per-vertex label
// requirements, the dense-label -> slot map, the candidate-list offsets (upper
// bound per list = frequency of the vertex's label) and the adjacency slots of
// label-matching vertices (for the algorithmic bytes).
struct FilterPrep {
  FilterArgs args{};
  std::vector<uint8_t> slot_of;
  std::vector<uint64_t> can_off;
  double adj = 0;
};

static void filter_prepare(const GraphDev &G, const gemh::QueryInfo &Q, uint32_t T, uint32_t W, FilterPrep *P) {
  const uint32_t nv = Q.nv;
  // query label slots in first-seen order (in-core/lib/io/src/io.cu:135-161)
  P->args = FilterArgs{};
  FilterQuery &fq = P->args.fq;
  fq.nv = nv;
  fq.T = T;
  fq.W = W;
  std::vector<uint32_t> slot(nv);
  std::vector<uint32_t> slot_label;
  for (uint32_t u = 0; u < nv; ++u) {
    uint32_t s = 0;
    while (s < slot_label.size() && slot_label[s] != Q.lab[u]) ++s;
    if (s == slot_label.size()) slot_label.push_back(Q.lab[u]);
    slot[u] = s;
    fq.group[s] |= 1u << u;
    fq.qdeg[u] = Q.deg[u];
  }
  fq.nslots = (uint32_t)slot_label.size();
  for (uint32_t u = 0; u < nv; ++u) {
    uint32_t cnt[GEM_MAX_QV] = {};
    for (auto [w, e] : Q.adj[u]) cnt[slot[w]]++;
    for (uint32_t s = 0; s < fq.nslots; ++s)
      if (cnt[s]) {
        fq.req_slot[u][fq.nreq[u]] = (uint8_t)s;
        fq.req_cnt[u][fq.nreq[u]] = (uint8_t)cnt[s];
        fq.nreq[u]++;
      }
  }
  // dense data label -> query slot
  const uint32_t nlab = (uint32_t)G.label_freq.size();
  P->slot_of.assign(std::max<uint32_t>(nlab, 1), (uint8_t)NO_SLOT);
  for (uint32_t s = 0; s < fq.nslots; ++s) {
    auto it = G.label_id.find(slot_label[s]);
    if (it != G.label_id.end()) P->slot_of[it->second] = (uint8_t)s;
  }
  if (G.lab8) {
    std::fill(std::begin(P->args.slot_of), std::end(P->args.slot_of), (uint8_t)NO_SLOT);
    std::copy(P->slot_of.begin(), P->slot_of.end(), P->args.slot_of);
  }
  // candidate storage: upper bound = frequency of u's label
  P->can_off.assign(nv + 1, 0);
  for (uint32_t u = 0; u < nv; ++u) {
    auto it = G.label_id.find(Q.lab[u]);
    uint64_t ub = it == G.label_id.end() ? 0 : G.label_freq[it->second];
    P->can_off[u + 1] = P->can_off[u] + ub;
  }
  P->adj = 0;
  for (uint32_t sl = 0; sl < fq.nslots; ++sl) {
    auto it = G.label_id.find(slot_label[sl]);
    if (it != G.label_id.end()) P->adj += (double)G.label_deg[it->second];
  }
}

// The filter's kernels on the context stream.  No allocation, no copy (a
// caller may capture the stream).
template <class LabT, bool NL>
static void filter_launch_as(gem_ctx *c, uint32_t W, const FilterPrep &P, const FilterBufs &B) {
  const GraphDev &G = graph(c);
  hipStream_t s = c->stream;
  const FilterGraph<LabT> g{G.off.as<uint64_t>(), G.nbr_dev(), G.nbr_lab.as<uint8_t>(), G.lab.as<LabT>(), B.slot_of, G.n};
  {
    ProfLaunch pl(c, K_FILTER);
    k_filter<LabT, NL><<<std::min<uint32_t>((W + FILTER_WAVES - 1) / FILTER_WAVES, 4096), FILTER_WAVES * 64, 0, s>>>(
        g, P.args, B.bitmap);
    GEM_LAUNCH_CHECK("k_filter");
  }
  if (G.n_heavy + G.n_hub) {
    ProfLaunch pl(c, K_FILTER_HEAVY);
    const uint32_t blocks = G.n_hub + std::min<uint32_t>((G.n_heavy + HEAVY_WAVES - 1) / HEAVY_WAVES, 2048);
    k_filter_heavy<LabT, NL><<<blocks, HEAVY_WAVES * 64, 0, s>>>(g, P.args, G.heavy.as<uint32_t>(), G.n_heavy,
                                                                 G.heavy.as<uint32_t>() + G.n_heavy, G.n_hub,
                                                                 reinterpret_cast<unsigned long long *>(B.bitmap));
    GEM_LAUNCH_CHECK("k_filter_heavy");
  }
}

static uint32_t rank_chunks(uint32_t W) { return (W + RANK_CHUNK - 1) / RANK_CHUNK; }

static void filter_launch(gem_ctx *c, uint32_t nv, uint32_t W, const FilterPrep &P, const uint64_t *can_off,
                          const FilterBufs &B) {
  const GraphDev &G = graph(c);
  hipStream_t s = c->stream;
  if (!G.lab8)
    filter_launch_as<uint32_t, false>(c, W, P, B);
  else if (G.nbr_lab.p)
    filter_launch_as<uint8_t, true>(c, W, P, B);
  else
    filter_launch_as<uint8_t, false>(c, W, P, B);
  const dim3 grid(rank_chunks(W), nv);
  CanOffsets co{};
  std::copy(can_off, can_off + nv + 1, co.at);
  ProfLaunch pl(c, K_COMPACT);
  if (grid.x > 1) {
    k_rank_sums<<<grid, 256, 0, s>>>(B.bitmap, W, B.sums);
    GEM_LAUNCH_CHECK("k_rank_sums");
  }
  k_rank_lists<<<grid, 256, 0, s>>>(B.bitmap, W, B.sums, B.rank, co, B.can, B.ncan);
  GEM_LAUNCH_CHECK("k_rank_lists");
}

void run_filter(gem_ctx *c, const gem_query_view *qv, uint32_t T) { run_filter(c, c->q, qv, T); }

void run_filter(gem_ctx *c, QueryDev &Qd, const gem_query_view *qv, uint32_t T) { run_filters(c, &Qd, &qv, 1, T); }

void run_filters(gem_ctx *c, QueryDev *Qds, const gem_query_view *const *qv, uint32_t n, uint32_t T) {
  if (!graph(c).loaded) throw Error{GEM_E_STATE, "no data graph loaded"};
  const GraphDev &G = graph(c);
  const uint32_t W = (G.n + 63) / 64;
  uint32_t nvs = 0;
  for (uint32_t i = 0; i < n; ++i) {
    Qds[i] = QueryDev();
    std::string why;
    int st = gemh::analyse_query(qv[i], &Qds[i].Q, &why);
    if (st) throw Error{st, why};
    nvs += Qds[i].Q.nv;
  }
  struct Run {
    FilterPrep P;
    DevBuf slot_of, sums;
  };
  std::vector<Run> runs(n);
  uint32_t *const h = pinned<uint32_t>(c, nvs);  // |Can(u)|, written by the last kernel of each
  hipStream_t s = c->stream;
  uint32_t *hq = h;
  for (uint32_t i = 0; i < n; ++i) {
    QueryDev &Qd = Qds[i];
    const uint32_t nv = Qd.Q.nv;
    FilterPrep &P = runs[i].P;
    Qd.W = W;
    filter_prepare(G, Qd.Q, T, W, &P);
    Qd.can_off = P.can_off;
    if (!i) GEM_HIP_CHECK(hipEventRecord(c->ev[0], s));
    FilterBufs B;
    DevBuf &slot_of = runs[i].slot_of, &sums = runs[i].sums;
    if (!G.lab8) {
      slot_of.alloc(P.slot_of.size(), s);
      GEM_HIP_CHECK(hipMemcpyAsync(slot_of.p, P.slot_of.data(), P.slot_of.size(), hipMemcpyHostToDevice, s));
    }
    Qd.bitmap.alloc((uint64_t)nv * W * 8, s);
    Qd.rank.alloc((uint64_t)nv * (W + 1) * 4, s);
    Qd.can.alloc(std::max<uint64_t>(Qd.can_off[nv], 1) * 4, s);
    sums.alloc((uint64_t)nv * rank_chunks(W) * 4, s);
    B.slot_of = slot_of.as<uint8_t>();
    B.bitmap = Qd.bitmap.as<uint64_t>();
    B.sums = sums.as<uint32_t>();
    B.rank = Qd.rank.as<uint32_t>();
    B.can = Qd.can.as<uint32_t>();
    B.ncan = pinned_dev(c, hq);
    hq += nv;
    filter_launch(c, nv, W, P, Qd.can_off.data(), B);
    // algorithmic bytes: 16 B per vertex (label, degree, offset pair), 8 B per
    // adjacency slot of a label-matching vertex (neighbour id + its label; 1 B
    // with slot labels), the candidate bitmaps written
    prof_bytes(c, K_FILTER, 16.0 * G.n + (G.nbr_lab.p ? 1.0 : 8.0) * P.adj + nv * (double)W * 8);
  }
  GEM_HIP_CHECK(hipEventRecord(c->ev[1], s));
  GEM_HIP_CHECK(hipStreamSynchronize(s));
  hq = h;
  for (uint32_t i = 0; i < n; ++i) {
    QueryDev &Qd = Qds[i];
    const uint32_t nv = Qd.Q.nv;
    Qd.ncan.assign(hq, hq + nv);
    hq += nv;
    double ncan_sum = 0;
    for (uint32_t u = 0; u < nv; ++u) ncan_sum += Qd.ncan[u];
    prof_bytes(c, K_COMPACT, nv * (double)W * 12 + 4.0 * ncan_sum);
    Qd.filtered = true;
  }
  prof_flush(c);
  if (!n) return;
  float ms = 0;  // of all n
  GEM_HIP_CHECK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
  c->times.filter_ms = ms;
  c->times.index_ms = 0;  // the index (bitmap + rank) is a by-product of the filter
}

// ------------------------------------------------ no-allocation variant
// Scratch of gem_hip_filter_noalloc: the label map, bitmaps, rank chunk sums and
// ranks of one call, carved from one fixed device array (each device holds its
// own copy until the process ends).  Calls that overlap on one device share it
// and race.
constexpr uint64_t FILTER_SCRATCH_BYTES = 64ull << 20;
constexpr int SCRATCH_MAX_DEVICES = 64;
static __device__ __align__(256) unsigned char scratch[FILTER_SCRATCH_BYTES];
static std::mutex g_scratch_mu;
static unsigned char *g_scratch_ptr[SCRATCH_MAX_DEVICES];  // device address of `scratch`, per device

void filter_scratch_init(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (device < 0 || device >= SCRATCH_MAX_DEVICES) throw Error{GEM_E_LIMIT, "device id beyond the scratch table"};
  if (g_scratch_ptr[device]) return;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p)
    throw Error{GEM_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e)};
  g_scratch_ptr[device] = static_cast<unsigned char *>(p);
}

// What a call is accepted by: the documented bound, which does not move with the
// kernels.  They take less than it (its terms: a query description, the label
// map, list offsets, bitmaps, a count per tile, ranks, and vertex lists).
uint64_t filter_scratch_bytes(const GraphDev &G, uint32_t nv) {
  const uint64_t W = (G.n + 63) / 64;
  const uint64_t hub_cap = std::max<uint32_t>(G.n_hub, 1);
  auto up = [](uint64_t x) { return (x + 255) / 256 * 256; };
  return up(sizeof(FilterQuery)) + up(std::max<uint64_t>(G.label_freq.size(), 1)) + up(8ull * (nv + 1)) +
         up(8ull * nv * W) + up(4ull * nv * W) + up(4ull * nv * (W + 1)) + up(4ull * std::max<uint64_t>(G.n, 1)) +
         up(4) + up(4 * hub_cap) + up(4) + up(4ull * hub_cap * GEM_MAX_QV);
}

void run_filter_noalloc(gem_ctx *c, const gem_query_view *qv, uint32_t T, uint32_t *d_num_can, uint32_t *d_can,
                        uint64_t can_pitch) {
  if (!graph(c).loaded) throw Error{GEM_E_STATE, "no data graph loaded"};
  if (!d_num_can) throw Error{GEM_E_INVALID, "d_num_can is null"};
  if (c->device < 0 || c->device >= SCRATCH_MAX_DEVICES || !g_scratch_ptr[c->device])
    throw Error{GEM_E_STATE, "scratch not initialised on this device"};
  gemh::QueryInfo Q;
  std::string why;
  int st = gemh::analyse_query(qv, &Q, &why);
  if (st) throw Error{st, why};
  const GraphDev &G = graph(c);
  const uint32_t nv = Q.nv;
  const uint32_t W = (G.n + 63) / 64;
  const uint64_t need = filter_scratch_bytes(G, nv);
  if (need > FILTER_SCRATCH_BYTES)
    throw Error{GEM_E_LIMIT, "gem_hip_filter_noalloc: this graph and query need " + std::to_string(need) +
                                 " bytes of scratch, more than its " + std::to_string(FILTER_SCRATCH_BYTES)};
  FilterPrep P;
  filter_prepare(G, Q, T, W, &P);
  // candidate lists at u * can_pitch in the caller's array: each list needs
  // room for its label's frequency (the bound the kernels write within)
  std::vector<uint64_t> can_off(nv + 1, 0);
  for (uint32_t u = 0; u < nv; ++u) {
    const uint64_t ub = P.can_off[u + 1] - P.can_off[u];
    if (d_can && ub > can_pitch)
      throw Error{GEM_E_INVALID, "can_pitch is smaller than the frequency of a query vertex's label"};
    can_off[u] = (uint64_t)u * can_pitch;
  }
  can_off[nv] = (uint64_t)nv * can_pitch;
  // carve the scratch array (its layout takes less than the limit above)
  unsigned char *base = g_scratch_ptr[c->device];
  uint64_t at = 0;
  auto take = [&](uint64_t bytes) {
    unsigned char *p = base + at;
    at += (bytes + 255) / 256 * 256;
    return p;
  };
  FilterBufs B;
  uint8_t *d_slot_of = take(P.slot_of.size());
  B.slot_of = d_slot_of;
  B.bitmap = reinterpret_cast<uint64_t *>(take(8ull * nv * W));
  B.sums = reinterpret_cast<uint32_t *>(take(4ull * nv * std::max<uint32_t>(rank_chunks(W), 1)));
  B.rank = reinterpret_cast<uint32_t *>(take(4ull * nv * (W + 1)));
  if (at > FILTER_SCRATCH_BYTES) throw Error{GEM_E_STATE, "scratch layout exceeds its size"};
  B.can = d_can;  // null: counts only
  B.ncan = d_num_can;
  hipStream_t s = c->stream;
  if (!G.lab8)
    GEM_HIP_CHECK(hipMemcpyAsync(d_slot_of, P.slot_of.data(), P.slot_of.size(), hipMemcpyHostToDevice, s));
  filter_launch(c, nv, W, P, can_off.data(), B);
  // the host arrays above are read by the copies: wait before they go
  GEM_HIP_CHECK(hipStreamSynchronize(s));
}

void run_position_lookup(gem_ctx *c, uint32_t u, const uint32_t *h_vertices, uint64_t n, uint32_t *h_pos) {
  QueryDev &Qd = c->q;
  if (!Qd.filtered) throw Error{GEM_E_STATE, "filter has not run"};
  if (u >= Qd.Q.nv) throw Error{GEM_E_INVALID, "query vertex out of range"};
  if (n == 0) return;
  hipStream_t s = c->stream;
  DevBuf dv, dp;
  dv.alloc(n * 4, s);
  dp.alloc(n * 4, s);
  GEM_HIP_CHECK(hipMemcpyAsync(dv.p, h_vertices, n * 4, hipMemcpyHostToDevice, s));
  k_position_lookup<<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(Qd.bitmap.as<uint64_t>(), Qd.rank.as<uint32_t>(), Qd.W,
                                                                c->g.n, u, dv.as<uint32_t>(), n, dp.as<uint32_t>());
  GEM_LAUNCH_CHECK("k_position_lookup");
  GEM_HIP_CHECK(hipMemcpyAsync(h_pos, dp.p, n * 4, hipMemcpyDeviceToHost, s));
  GEM_HIP_CHECK(hipStreamSynchronize(s));
}

}  // namespace gemd
