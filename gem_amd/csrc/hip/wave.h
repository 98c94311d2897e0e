// Wave64 building blocks for gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace gemd {

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Load / store through the global address space.  Pointers read from memory
// (list addresses, row pointers) are generic to the compiler, which then
// emits flat instructions: those also count against the LDS wait counter, so
// every wait on them waits for LDS traffic too.  All such pointers here are
// device memory or mapped host memory, which global instructions reach.
template <class T>
__device__ __forceinline__ T ldg(const T *p) {
  return *(const __attribute__((address_space(1))) T *)p;
}
template <class T>
__device__ __forceinline__ void stg(T *p, T v) {
  *(__attribute__((address_space(1))) T *)p = v;
}

// Two neighbouring offsets (start and end of a list) in one 16-byte load.
typedef uint64_t u64x2 __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ u64x2 ld_pair(const uint64_t *p) {
  return *(const __attribute__((address_space(1))) u64x2 *)p;
}

// Up to four consecutive words in one store.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ void st_words(uint32_t *p, u32x4 x, uint32_t n) {
  if (n == 4)
    *(__attribute__((address_space(1))) u32x4 *)p = x;
  else if (n == 3)
    *(__attribute__((address_space(1))) u32x3 *)p = u32x3{x[0], x[1], x[2]};
  else if (n == 2)
    *(__attribute__((address_space(1))) u32x2 *)p = u32x2{x[0], x[1]};
  else
    stg(p, x[0]);
}

// popcount of the bits of `m` below this lane (v_mbcnt_lo/hi)
__device__ __forceinline__ uint32_t rank_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ uint32_t readlane_u32(uint32_t x, uint32_t lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, (int)lane);
}
__device__ __forceinline__ uint64_t readlane_u64(uint64_t x, uint32_t lane) {
  uint32_t lo = readlane_u32((uint32_t)x, lane), hi = readlane_u32((uint32_t)(x >> 32), lane);
  return ((uint64_t)hi << 32) | lo;
}

// Inclusive wave scan (all lanes active): within rows of 16 lanes, then the
// rows' totals handed on, all by DPP moves (shuffles go through LDS).
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t x) {
  x += dpp_or_zero<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8
  x += dpp_or_zero<0x112, 0xf>(x);
  x += dpp_or_zero<0x114, 0xf>(x);
  x += dpp_or_zero<0x118, 0xf>(x);
  x += dpp_or_zero<0x142, 0xa>(x);  // lane 15 of a row to the next one (rows 1 and 3)
  x += dpp_or_zero<0x143, 0xc>(x);  // lane 31 to rows 2 and 3
  return x;
}
__device__ __forceinline__ uint64_t wave_incl_scan_u64(uint64_t x) {
  const uint32_t l = lane_id();
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    uint64_t y = __shfl_up(x, d, 64);
    if (l >= d) x += y;
  }
  return x;
}
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t x) {
#pragma unroll
  for (uint32_t d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d, 64);
  return x;
}

// Block-wide exclusive scan of one u64 per thread (blockDim.x a multiple of
// 64, at most 8 waves per smem slot count); returns the block total.
__device__ __forceinline__ uint64_t block_excl_scan_u64(uint64_t x, uint64_t *excl, uint64_t *smem /*[nwaves]*/) {
  const uint32_t t = threadIdx.x, w = t / 64, l = t % 64;
  const uint32_t nw = blockDim.x / 64;
  uint64_t inc = wave_incl_scan_u64(x);
  if (l == 63) smem[w] = inc;
  __syncthreads();
  uint64_t wbase = 0, tot = 0;
  for (uint32_t i = 0; i < nw; ++i) {
    uint64_t s = smem[i];
    if (i < w) wbase += s;
    tot += s;
  }
  __syncthreads();
  *excl = wbase + inc - x;
  return tot;
}

// Largest r in [0, 64) with starts[r] <= item (starts ascending, starts[0] == 0).
__device__ __forceinline__ uint32_t seg_of(const uint32_t *starts, uint32_t item) {
  uint32_t lo = 0;
#pragma unroll
  for (uint32_t step = 32; step >= 1; step >>= 1)
    if (starts[lo + step] <= item && lo + step < 64) lo += step;
  return lo;
}

// Binary search for v in sorted a[0..n) (device or mapped host memory); true
// if present.
template <class T>
__device__ __forceinline__ bool sorted_contains(const T *a, uint64_t n, T v) {
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    uint64_t mid = (lo + hi) >> 1;
    T x = ldg(a + mid);
    if (x < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo < n && ldg(a + lo) == v;
}

// First index of sorted a[0..n) whose value is >= v (lower) or > v (upper).
__device__ __forceinline__ uint32_t lower_bound_u32(const uint32_t *a, uint32_t n, uint32_t v) {
  uint32_t lo = 0;
  while (n) {
    const uint32_t h = n >> 1;
    if (ldg(a + lo + h) < v) {
      lo += h + 1;
      n -= h + 1;
    } else {
      n = h;
    }
  }
  return lo;
}
__device__ __forceinline__ uint32_t upper_bound_u32(const uint32_t *a, uint32_t n, uint32_t v) {
  uint32_t lo = 0;
  while (n) {
    const uint32_t h = n >> 1;
    if (ldg(a + lo + h) <= v) {
      lo += h + 1;
      n -= h + 1;
    } else {
      n = h;
    }
  }
  return lo;
}

// Two membership tests at once in one list (the same in every lane): k0 says
// whether v0, k1 whether v1 is in sorted a[0..n); false ones stay false.  A
// search keeps the last place whose value is not above its own, so it is a
// load, a compare and a select a step, and the lanes step together.
// GLOBAL: the list is in device or mapped host memory (else in LDS).
template <bool GLOBAL = true>
__device__ __forceinline__ void contains_pair(const uint32_t *a, uint32_t n, uint32_t v0, bool &k0, uint32_t v1,
                                              bool &k1) {
  auto at = [&](uint32_t i) { return GLOBAL ? ldg(a + i) : a[i]; };
  if (!n) {
    k0 = k1 = false;
    return;
  }
  uint32_t o0 = 0, o1 = 0;
  for (; n > 1; n -= n >> 1) {
    const uint32_t h = n >> 1;
    const uint32_t x0 = at(o0 + h), x1 = at(o1 + h);
    o0 += x0 <= v0 ? h : 0;
    o1 += x1 <= v1 ? h : 0;
  }
  const uint32_t x0 = at(o0), x1 = at(o1);
  k0 = k0 && x0 == v0;
  k1 = k1 && x1 == v1;
}

// Four membership tests at once: v[g] in sorted a[g][0..n[g]) (each lane its
// own lists); k[g] enters as "still wanted" and leaves as the result.  The four
// searches advance in lockstep, so up to four loads of one lane are in flight
// at every stage.  A search that has ended or is not wanted goes on loading the
// place it found, or `any` (one readable word), instead of masking its lane
// off: the steps are selects and not branches (with four branches a step, the
// walk kernel ran more scalar than vector instructions), and the last place not
// above the value is kept instead of a flag for an equal one (8 vector
// instructions a step instead of 14).
__device__ __forceinline__ void contains_quad(const uint32_t *const a[4], const uint32_t n_in[4],
                                              const uint32_t v[4], bool k[4], const uint32_t *any) {
  const uint32_t *p[4];
  uint32_t n[4], o[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    k[g] = k[g] && n_in[g];
    p[g] = k[g] ? a[g] : any;
    n[g] = k[g] ? n_in[g] : 1;
    o[g] = 0;
  }
  while (__any((n[0] | n[1] | n[2] | n[3]) > 1)) {
    uint32_t x[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) x[g] = ldg(p[g] + (o[g] + (n[g] >> 1)));
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t h = n[g] >> 1;
      o[g] += x[g] <= v[g] ? h : 0;
      n[g] -= h;
    }
  }
  uint32_t x[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) x[g] = ldg(p[g] + o[g]);
#pragma unroll
  for (int g = 0; g < 4; ++g) k[g] = k[g] && x[g] == v[g];
}

// Map a hardware workgroup id to a logical one so that consecutive logical
// blocks run on the same XCD (workgroups are dispatched round-robin over the
// 8 XCDs); neighbouring row blocks then share one L2.
__device__ __forceinline__ uint32_t xcd_swizzle(uint32_t hw, uint32_t nblocks) {
  constexpr uint32_t X = 8;
  const uint32_t per = nblocks / X;
  if (per == 0) return hw;
  const uint32_t full = per * X;
  if (hw >= full) return hw;
  return (hw % X) * per + hw / X;
}

}  // namespace gemd
