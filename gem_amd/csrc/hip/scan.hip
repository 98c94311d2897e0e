// Exclusive prefix sums used by the filter (candidate ranks), the edge tables
// (row offsets) and the join (output offsets).  Reduce-then-scan: per-tile sums,
// then a tile-local scan whose blocks add up the sums before theirs.  Integer
// adds only, so results are exact and order-independent.
#include "ctx.h"
#include "wave.h"

namespace gemd {

constexpr uint32_t SCAN_THREADS = 256;
constexpr uint32_t SCAN_ITEMS = 16;
constexpr uint32_t SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__global__ void __launch_bounds__(SCAN_THREADS) k_tile_sums_u64(const uint64_t *in, uint64_t n, uint64_t *sums) {
  __shared__ uint64_t sm[8];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
  uint64_t acc = 0;
  for (uint32_t i = 0; i < SCAN_ITEMS; ++i) {
    uint64_t idx = base + (uint64_t)i * SCAN_THREADS + threadIdx.x;
    if (idx < n) acc += in[idx];
  }
  uint64_t ex;
  uint64_t tot = block_excl_scan_u64(acc, &ex, sm);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Tile-local scan: wave w of a block holds entries [w, w + 1) * 64 * SCAN_ITEMS
// of its tile, lane = entry modulo 64.  SUMS: `before` holds the tiles' sums and
// a block adds up those before its own, else it holds their exclusive scan.
// The last tile's block writes the total to out[n] (and *total, when given).
template <bool SUMS>
__global__ void __launch_bounds__(SCAN_THREADS) k_tile_scan_u64(const uint64_t *in, uint64_t n, const uint64_t *before,
                                                              uint64_t *out, uint64_t *total) {
  __shared__ uint64_t sm[4], pre[4];
  const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + w * 64 * SCAN_ITEMS;
  uint64_t v[SCAN_ITEMS], x = 0, y = 0;
#pragma unroll
  for (uint32_t i = 0; i < SCAN_ITEMS; ++i) {
    const uint64_t at = base + i * 64 + l;
    v[i] = at < n ? in[at] : 0;
    x += v[i];
  }
  if (SUMS)
    for (uint32_t c = threadIdx.x; c < blockIdx.x; c += SCAN_THREADS) y += before[c];
  x = wave_sum_u64(x);
  y = wave_sum_u64(y);
  if (l == 0) {
    sm[w] = x;
    pre[w] = y;
  }
  __syncthreads();
  uint64_t run = SUMS ? pre[0] + pre[1] + pre[2] + pre[3] : before[blockIdx.x];
  for (uint32_t i = 0; i < w; ++i) run += sm[i];
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == SCAN_THREADS - 64) {  // the last wave
    out[n] = run + sm[3];
    if (total) *total = run + sm[3];
  }
#pragma unroll
  for (uint32_t i = 0; i < SCAN_ITEMS; ++i) {
    if (base + i * 64 >= n) break;
    const uint64_t at = base + i * 64 + l, incl = wave_incl_scan_u64(v[i]);
    if (at < n) out[at] = run + incl - v[i];
    run += readlane_u64(incl, 63);
  }
}

// One launch up to a tile, two up to ADD_TILES tiles (blocks adding up the sums
// before theirs read ADD_TILES^2 / 2 of them at most, 64 MiB); beyond, the sums
// are scanned in turn.  (One block that scanned up to 65,536 values by itself
// took 43 us on average and up to 110 in the length passes of capped batches.)
constexpr uint64_t ADD_TILES = 4096;

void scan_u64(gem_ctx *c, const uint64_t *d_in, uint64_t *d_out, uint64_t n, uint64_t *d_total) {
  const uint64_t tiles = std::max<uint64_t>(1, (n + SCAN_TILE - 1) / SCAN_TILE);
  DevBuf sums, base;
  if (tiles > 1) {
    sums.alloc(tiles * 8, c->stream);
    k_tile_sums_u64<<<(uint32_t)tiles, SCAN_THREADS, 0, c->stream>>>(d_in, n, sums.as<uint64_t>());
    GEM_LAUNCH_CHECK("k_tile_sums_u64");
  }
  if (tiles > ADD_TILES) {
    base.alloc((tiles + 1) * 8, c->stream);
    scan_u64(c, sums.as<uint64_t>(), base.as<uint64_t>(), tiles);
    k_tile_scan_u64<false><<<(uint32_t)tiles, SCAN_THREADS, 0, c->stream>>>(d_in, n, base.as<uint64_t>(), d_out, d_total);
  } else {
    k_tile_scan_u64<true><<<(uint32_t)tiles, SCAN_THREADS, 0, c->stream>>>(d_in, n, sums.as<uint64_t>(), d_out, d_total);
  }
  GEM_LAUNCH_CHECK("k_tile_scan_u64");
}

// Many independent in-place scans: segments in chunks of SEG_CHUNK entries,
// chunk sums first (left out when no segment has two chunks), then each block
// adds up the sums of its segment's chunks before its own and scans it: wave w
// holds entries [w, w + 1) * 1024, lane = entry modulo 64.  One block per
// segment took 75 us for the 30 tables of a 16-vertex query on 2^22 vertices.
constexpr uint32_t SEG_STEPS = 16, SEG_CHUNK = 4 * 64 * SEG_STEPS;
uint32_t scan_chunks(uint64_t n) { return (uint32_t)std::max<uint64_t>(1, (n + SEG_CHUNK - 1) / SEG_CHUNK); }

__device__ __forceinline__ uint32_t seg_of_chunk(const ScanSeg *segs, uint32_t nseg, uint32_t chunk) {
  uint32_t lo = 0, hi = nseg;  // the last segment whose first chunk is <= chunk
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) / 2;
    if (segs[mid].first_chunk <= chunk)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

__global__ void __launch_bounds__(256) k_seg_sums(const ScanSeg *__restrict__ segs, uint32_t nseg,
                                                 uint64_t *__restrict__ sums) {
  __shared__ uint64_t sm[4];
  const ScanSeg sg = segs[seg_of_chunk(segs, nseg, blockIdx.x)];
  const uint64_t base = (uint64_t)(blockIdx.x - sg.first_chunk) * SEG_CHUNK;
  uint64_t x = 0;
#pragma unroll
  for (uint32_t i = 0; i < SEG_STEPS; ++i) {
    const uint64_t at = base + i * 256 + threadIdx.x;
    if (at < sg.n) x += sg.p[at];
  }
  x = wave_sum_u64(x);
  if (threadIdx.x % 64 == 0) sm[threadIdx.x / 64] = x;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = sm[0] + sm[1] + sm[2] + sm[3];
}

__global__ void __launch_bounds__(256) k_seg_scan(const ScanSeg *__restrict__ segs, uint32_t nseg,
                                                 const uint64_t *__restrict__ sums, uint64_t *__restrict__ totals) {
  __shared__ uint64_t sm[4], before[4];
  const uint32_t k = seg_of_chunk(segs, nseg, blockIdx.x);
  const ScanSeg sg = segs[k];
  const uint32_t chunk = blockIdx.x - sg.first_chunk, w = threadIdx.x / 64, l = threadIdx.x % 64;
  const uint64_t base = (uint64_t)chunk * SEG_CHUNK + w * 64 * SEG_STEPS;
  uint64_t v[SEG_STEPS], x = 0, y = 0;
#pragma unroll
  for (uint32_t i = 0; i < SEG_STEPS; ++i) {
    const uint64_t at = base + i * 64 + l;
    v[i] = at < sg.n ? sg.p[at] : 0;
    x += v[i];
  }
  for (uint32_t c = threadIdx.x; c < chunk; c += 256) y += sums[sg.first_chunk + c];
  x = wave_sum_u64(x);
  y = wave_sum_u64(y);
  if (l == 0) {
    sm[w] = x;
    before[w] = y;
  }
  __syncthreads();
  uint64_t run = before[0] + before[1] + before[2] + before[3];
  for (uint32_t i = 0; i < w; ++i) run += sm[i];
  if ((uint64_t)(chunk + 1) * SEG_CHUNK >= sg.n && threadIdx.x == 192) {  // the last chunk's last wave
    sg.p[sg.n] = run + sm[3];
    totals[k] = run + sm[3];
  }
#pragma unroll
  for (uint32_t i = 0; i < SEG_STEPS; ++i) {
    if (base + i * 64 >= sg.n) break;
    const uint64_t at = base + i * 64 + l, incl = wave_incl_scan_u64(v[i]);
    if (at < sg.n) sg.p[at] = run + incl - v[i];
    run += readlane_u64(incl, 63);
  }
}

void scan_segments_u64(gem_ctx *c, const ScanSeg *d_segs, uint32_t nseg, uint32_t chunks, uint64_t *d_totals) {
  if (!nseg) return;
  DevBuf sums;
  if (chunks > nseg) {
    sums.alloc((uint64_t)chunks * 8, c->stream);
    k_seg_sums<<<chunks, 256, 0, c->stream>>>(d_segs, nseg, sums.as<uint64_t>());
    GEM_LAUNCH_CHECK("k_seg_sums");
  }
  k_seg_scan<<<chunks, 256, 0, c->stream>>>(d_segs, nseg, sums.as<uint64_t>(), d_totals);
  GEM_LAUNCH_CHECK("k_seg_scan");
}

}  // namespace gemd
