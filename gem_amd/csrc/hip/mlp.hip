// Order-cost model: a 3-layer MLP (in -> 128 -> 128 -> 1, ReLU) with bf16
// weights and fp32 accumulation, trained and evaluated on the GPU by the
// kernels below (no library GEMM).  It predicts the cost of a join order from
// int32 order features; the batched path uses it to pick among candidate
// orders (the reference has no learned component; GEM's order stays a
// candidate and the fallback).
//
// Models of the shipped width (h = 128, in a multiple of 16 up to 272) run as
// one forward kernel, one kernel for the input gradients and one MFMA kernel
// for the weight gradients; other shapes run as a sequence of k_gemm.
//
// Parameters (fp32 master copy, flat): W1[in x h], b1[h], W2[h x h], b2[h],
// W3[h], b3[1]; forward and backward use bf16 copies of W1..W3 (rounded to
// nearest even).  Loss: mean squared error / 2.  Optimiser: Adam.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "../host/host_graph.h"
#include "ctx.h"

namespace gemd {

// fp32 -> bf16 bits, round to nearest even (NaN kept quiet)
__host__ __device__ inline uint16_t f32_to_bf16(float f) {
  uint32_t x = __builtin_bit_cast(uint32_t, f);
  if ((x & 0x7F800000u) == 0x7F800000u && (x & 0x007FFFFFu)) return (uint16_t)((x >> 16) | 0x40);
  x += 0x7FFFu + ((x >> 16) & 1u);
  return (uint16_t)(x >> 16);
}
__host__ __device__ inline float bf16_to_f32(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

constexpr int TM = 64, TN = 64, TK = 16;

// C[M x N] = op(A) op(B) (+ bias[N]) with an epilogue:
//   EPI 0: store; 1: bias + ReLU; 2: bias; 3: multiply by (mask[m][n] > 0)
// A is fp32: element (m, k) at A[m*lda + k] (TA = false) or A[k*lda + m].
// B is fp32 or bf16 (BBF): element (k, n) at B[k*ldb + n] (TB = false) or
// B[n*ldb + k].  256 threads, each a 4x4 block of C.
template <bool TA, bool TB, bool BBF, int EPI>
__global__ void __launch_bounds__(256) k_gemm(int M, int N, int K, const float *__restrict__ A, int lda,
                                             const void *__restrict__ Bv, int ldb, const float *__restrict__ bias,
                                             const float *__restrict__ mask, float *__restrict__ C, int ldc) {
  __shared__ float As[TK][TM + 1];
  __shared__ float Bs[TK][TN + 1];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  float acc[4][4] = {};
  const float *Bf = reinterpret_cast<const float *>(Bv);
  const uint16_t *Bh = reinterpret_cast<const uint16_t *>(Bv);
  for (int k0 = 0; k0 < K; k0 += TK) {
    for (int i = threadIdx.x; i < TK * TM; i += 256) {
      const int kk = i / TM, mm = i % TM;
      const int m = m0 + mm, k = k0 + kk;
      float v = 0.f;
      if (m < M && k < K) v = TA ? A[(size_t)k * lda + m] : A[(size_t)m * lda + k];
      As[kk][mm] = v;
    }
    for (int i = threadIdx.x; i < TK * TN; i += 256) {
      const int kk = i / TN, nn = i % TN;
      const int n = n0 + nn, k = k0 + kk;
      float v = 0.f;
      if (n < N && k < K) {
        const size_t idx = TB ? (size_t)n * ldb + k : (size_t)k * ldb + n;
        v = BBF ? bf16_to_f32(Bh[idx]) : Bf[idx];
      }
      Bs[kk][nn] = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (EPI == 1) v = fmaxf(v + bias[n], 0.f);
      if (EPI == 2) v = v + bias[n];
      if (EPI == 3) v = mask[(size_t)m * ldc + n] > 0.f ? v : 0.f;
      C[(size_t)m * ldc + n] = v;
    }
  }
}

// ------------------------------------------------ models of width 128
constexpr uint32_t MH = 128;      // hidden width
constexpr uint32_t MF_MAX = 272;  // widest input whose weights and rows fit the LDS
constexpr float FEAT_SCALE = 1.0f / 64.0f;

// Where the parameters of a model of F inputs stand in the flat vector.
struct MlpLayout {
  uint32_t F;
  __host__ __device__ uint32_t b1() const { return F * MH; }
  __host__ __device__ uint32_t W2() const { return b1() + MH; }
  __host__ __device__ uint32_t b2() const { return W2() + MH * MH; }
  __host__ __device__ uint32_t W3() const { return b2() + MH; }
  __host__ __device__ uint32_t b3() const { return W3() + MH; }
};

__device__ __forceinline__ float bf_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }

// W[2i][c] and W[2i + 1][c] (bf16, row-major [rows x 128]) as one word at
// P[i * 128 + c].
__device__ __forceinline__ void load_pairs(const uint16_t *__restrict__ W, uint32_t rows, uint32_t *P) {
  for (uint32_t i = threadIdx.x; i < rows / 2 * (MH / 8); i += blockDim.x) {
    const uint32_t r = i / (MH / 8), c = i % (MH / 8) * 8;
    const uint4 a = *reinterpret_cast<const uint4 *>(W + (size_t)(2 * r) * MH + c);
    const uint4 b = *reinterpret_cast<const uint4 *>(W + (size_t)(2 * r + 1) * MH + c);
    const uint32_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      P[r * MH + c + 2 * k] = (x[k] & 0xFFFFu) | (y[k] << 16);
      P[r * MH + c + 2 * k + 1] = (x[k] >> 16) | (y[k] & 0xFFFF0000u);
    }
  }
}

// acc[r] += sum over k ascending of x[r][k] * W[k][col], W as pairs in LDS.
template <int R>
__device__ __forceinline__ void dot_rows(const float *x, uint32_t stride, uint32_t K, const uint32_t *P, uint32_t col,
                                         float (&acc)[R]) {
  for (uint32_t k = 0; k < K; k += 4) {
    const uint32_t p0 = P[(k / 2) * MH + col], p1 = P[(k / 2 + 1) * MH + col];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float4 v = *reinterpret_cast<const float4 *>(x + r * stride + k);
      acc[r] = fmaf(v.x, bf_lo(p0), acc[r]);
      acc[r] = fmaf(v.y, bf_hi(p0), acc[r]);
      acc[r] = fmaf(v.z, bf_lo(p1), acc[r]);
      acc[r] = fmaf(v.w, bf_hi(p1), acc[r]);
    }
  }
}

// The three layers in one launch: a block holds all weights in LDS (103 KB of
// 160) and takes 8 R rows at a time, thread (c, g) column c of rows g R ... of
// them.  Each sum runs over its inputs in ascending order in one accumulator
// (as k_gemm's do).  Scoring a query's 8 candidates is bound by latency: three
// k_gemm launches of two blocks took 85 us, this one takes 11.
constexpr uint32_t MROW = MH + 4;  // floats of a hidden row in LDS
template <int R, bool STORE>
__global__ void __launch_bounds__(1024) k_mlp_forward(const int32_t *__restrict__ feats, uint32_t n, MlpLayout L,
                                                     const float *__restrict__ p, const uint16_t *__restrict__ wb,
                                                     float *__restrict__ H1, float *__restrict__ H2,
                                                     float *__restrict__ Y) {
  extern __shared__ uint4 mlp_lds[];
  const uint32_t F = L.F;
  uint32_t *P1 = reinterpret_cast<uint32_t *>(mlp_lds), *P2 = P1 + F / 2 * MH;
  float *w3 = reinterpret_cast<float *>(P2 + MH / 2 * MH);
  float *h1 = w3 + MH, *xs = h1 + 8 * R * MROW;  // xs: 8 R x F, then the second hidden rows
  load_pairs(wb, F, P1);
  load_pairs(wb + (size_t)F * MH, MH, P2);
  const uint32_t col = threadIdx.x % MH, g = threadIdx.x / MH;
  if (g == 0) w3[col] = bf16_to_f32(wb[(size_t)F * MH + MH * MH + col]);
  const float b1 = p[L.b1() + col], b2 = p[L.b2() + col], b3 = p[L.b3()];
  for (uint32_t r0 = blockIdx.x * 8 * R; r0 < n; r0 += gridDim.x * 8 * R) {
    const uint32_t rows = n - r0 < 8 * R ? n - r0 : 8 * R;
    __syncthreads();  // weights stand; the last rows are done with
    for (uint32_t i = threadIdx.x; i < 8 * R * (F / 4); i += 1024) {
      int4 f = make_int4(0, 0, 0, 0);
      if (i < rows * (F / 4)) f = reinterpret_cast<const int4 *>(feats + (size_t)r0 * F)[i];
      reinterpret_cast<float4 *>(xs)[i] = make_float4((float)f.x * FEAT_SCALE, (float)f.y * FEAT_SCALE,
                                                      (float)f.z * FEAT_SCALE, (float)f.w * FEAT_SCALE);
    }
    __syncthreads();
    float acc[R] = {};
    dot_rows<R>(xs + g * R * F, F, F, P1, col, acc);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float v = fmaxf(acc[r] + b1, 0.f);
      h1[(g * R + r) * MROW + col] = v;
      if (STORE && g * R + r < rows) H1[(size_t)(r0 + g * R + r) * MH + col] = v;
      acc[r] = 0.f;
    }
    __syncthreads();
    dot_rows<R>(h1 + g * R * MROW, MROW, MH, P2, col, acc);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float v = fmaxf(acc[r] + b2, 0.f);
      xs[(g * R + r) * MROW + col] = v;
      if (STORE && g * R + r < rows) H2[(size_t)(r0 + g * R + r) * MH + col] = v;
    }
    __syncthreads();
    if (threadIdx.x < rows) {
      float a = 0.f;
      for (uint32_t k = 0; k < MH; k += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(xs + threadIdx.x * MROW + k);
        a = fmaf(v.x, w3[k], a);
        a = fmaf(v.y, w3[k + 1], a);
        a = fmaf(v.z, w3[k + 2], a);
        a = fmaf(v.w, w3[k + 3], a);
      }
      Y[r0 + threadIdx.x] = a + b3;
    }
  }
}

// Input gradients of 8 R rows at a time (thread (c, g) as above): dY = (y - t) / n,
// dH2 = dY W3 and dH1 = dH2 W2^T where the unit was active; and the block's
// sums over its rows for the gradients of W3 and the biases and for the loss:
// part[block] = db1[128], db2[128], dW3[128], db3, loss.
constexpr uint32_t MPART = 3 * MH + 2;
template <int R>
__global__ void __launch_bounds__(1024)
k_mlp_backward(const float *__restrict__ Y, const float *__restrict__ T, uint32_t n, MlpLayout L,
               const uint16_t *__restrict__ wb, const float *__restrict__ H1, const float *__restrict__ H2,
               float *__restrict__ dH1, float *__restrict__ dH2, float *__restrict__ part) {
  __shared__ uint32_t P[MH / 2 * MH];  // W2^T in pairs: (W2[c][2i], W2[c][2i + 1]) at P[i * 128 + c]
  __shared__ __align__(16) float d2[8 * R * MROW];
  __shared__ float sums[8][3][MH], tail[2][8];
  const uint16_t *W2 = wb + (size_t)L.F * MH;
  for (uint32_t i = threadIdx.x; i < MH * (MH / 8); i += 1024) {
    const uint32_t c = i % MH, k = i / MH * 8;
    const uint4 a = *reinterpret_cast<const uint4 *>(W2 + (size_t)c * MH + k);
    P[(k / 2) * MH + c] = a.x;
    P[(k / 2 + 1) * MH + c] = a.y;
    P[(k / 2 + 2) * MH + c] = a.z;
    P[(k / 2 + 3) * MH + c] = a.w;
  }
  const uint32_t col = threadIdx.x % MH, g = threadIdx.x / MH;
  const float w3 = bf16_to_f32(W2[MH * MH + col]);
  float s1 = 0.f, s2 = 0.f, s3 = 0.f, sy = 0.f, sl = 0.f;
  for (uint32_t r0 = blockIdx.x * 8 * R; r0 < n; r0 += gridDim.x * 8 * R) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t row = r0 + g * R + r;
      float d = 0.f;
      if (row < n) {
        const float e = Y[row] - T[row], dy = e / (float)n, h2 = H2[(size_t)row * MH + col];
        d = h2 > 0.f ? dy * w3 : 0.f;
        dH2[(size_t)row * MH + col] = d;
        s2 += d;
        s3 = fmaf(h2, dy, s3);
        sy += dy;
        sl += 0.5f * e * e / (float)n;
      }
      d2[(g * R + r) * MROW + col] = d;
    }
    __syncthreads();
    float acc[R] = {};
    dot_rows<R>(d2 + g * R * MROW, MROW, MH, P, col, acc);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t row = r0 + g * R + r;
      if (row < n) {
        const float d = H1[(size_t)row * MH + col] > 0.f ? acc[r] : 0.f;
        dH1[(size_t)row * MH + col] = d;
        s1 += d;
      }
    }
  }
  sums[g][0][col] = s1;
  sums[g][1][col] = s2;
  sums[g][2][col] = s3;
  if (col == 0) {
    tail[0][g] = sy;
    tail[1][g] = sl;
  }
  __syncthreads();
  float *out = part + (size_t)blockIdx.x * MPART;
  if (threadIdx.x < 3 * MH) {
    float v = 0.f;
    for (int i = 0; i < 8; ++i) v += sums[i][threadIdx.x / MH][threadIdx.x % MH];
    out[threadIdx.x] = v;
  } else if (threadIdx.x < MPART) {
    float v = 0.f;
    for (int i = 0; i < 8; ++i) v += tail[threadIdx.x - 3 * MH][i];
    out[threadIdx.x] = v;
  }
}

// Weight gradients dW1 = X^T dH1 and dW2 = H1^T dH2 by fp32 MFMA (16x16x4):
// a wave takes 16 rows of one of them (all 128 columns, 32 accumulators) over
// one of gridDim.y slices of the n samples, whose partial sums k_mlp_reduce
// adds.  The contraction is over the samples and the result is small, so the
// slices are what fills the chip: as tiles of the result with the whole sum in
// one block (k_gemm), 20,480 samples took 11.8 ms, so 71 us.  Lane l holds samples
// s + l / 16; its eight columns (l % 16) * 8 ... are column l % 16 of eight
// tiles, so the right-hand rows are loaded 16 bytes at a time.
typedef float f32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) k_mlp_wgrad(const int32_t *__restrict__ feats, const float *__restrict__ H1,
                                                  const float *__restrict__ dH1, const float *__restrict__ dH2,
                                                  uint32_t n, uint32_t F, uint32_t slice, float *__restrict__ part) {
  const uint32_t tile = blockIdx.x * 4 + threadIdx.x / 64, l = threadIdx.x % 64;
  if (tile >= (F + MH) / 16) return;
  const bool first = tile < F / 16;  // a tile of dW1
  const uint32_t m = (first ? tile : tile - F / 16) * 16 + l % 16;
  const uint32_t lda = first ? F : MH;
  const float *B = first ? dH1 : dH2;
  const uint32_t s0 = blockIdx.y * slice, s1 = n - s0 < slice ? n : s0 + slice;
  f32x4 acc[8] = {};
  auto step = [&](uint32_t r) {
    const float a = first ? (float)feats[(size_t)r * lda + m] * FEAT_SCALE : H1[(size_t)r * lda + m];
    const f32x4 *q = reinterpret_cast<const f32x4 *>(B + (size_t)r * MH + (l % 16) * 8);
    const f32x4 b[2] = {q[0], q[1]};
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[j / 4][j % 4], acc[j], 0, 0, 0);
  };
  const uint32_t full = (s1 - s0) / 16;  // groups of 16 samples: four steps' loads in flight
  for (uint32_t i = 0; i < full; ++i)
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) step(s0 + 16 * i + 4 * u + l / 16);
  uint32_t s = s0 + 16 * full;
  for (; s + 4 <= s1; s += 4) step(s + l / 16);
  if (s < s1) {  // the last samples: lanes past the end add nothing
    const uint32_t r = s + l / 16;
    float a = 0.f;
    f32x4 b[2] = {};
    if (r < s1) {
      a = first ? (float)feats[(size_t)r * lda + m] * FEAT_SCALE : H1[(size_t)r * lda + m];
      const f32x4 *q = reinterpret_cast<const f32x4 *>(B + (size_t)r * MH + (l % 16) * 8);
      b[0] = q[0];
      b[1] = q[1];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[j / 4][j % 4], acc[j], 0, 0, 0);
  }
  // accumulator i of tile j: result row tile * 16 + 4 (l / 16) + i, column (l % 16) * 8 + j
  float *out = part + ((size_t)blockIdx.y * (F + MH) + tile * 16) * MH;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x4 v[2];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j / 4][j % 4] = acc[j][i];
    f32x4 *q = reinterpret_cast<f32x4 *>(out + (size_t)(4 * (l / 16) + i) * MH + (l % 16) * 8);
    q[0] = v[0];
    q[1] = v[1];
  }
}

// Partial sums -> gradients (flat, as the parameters) and the loss: a thread
// per weight over the slices, then a wave per block sum over the row blocks.
__global__ void __launch_bounds__(256) k_mlp_reduce(const float *__restrict__ wpart, uint32_t slices,
                                                   const float *__restrict__ part, uint32_t blocks, MlpLayout L,
                                                   float *__restrict__ grads, float *__restrict__ loss) {
  const uint32_t nw = (L.F + MH) * MH, wb = nw / 256;
  if (blockIdx.x < wb) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    float v = 0.f;
#pragma unroll 8
    for (uint32_t s = 0; s < slices; ++s) v += wpart[(size_t)s * nw + i];
    grads[i < L.F * MH ? i : L.W2() + (i - L.F * MH)] = v;
    return;
  }
  const uint32_t x = (blockIdx.x - wb) * 4 + threadIdx.x / 64, l = threadIdx.x % 64;
  if (x >= MPART) return;
  double v = 0;
  for (uint32_t b = l; b < blocks; b += 64) v += part[(size_t)b * MPART + x];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if (l) return;
  if (x < MH)
    grads[L.b1() + x] = (float)v;
  else if (x < 2 * MH)
    grads[L.b2() + x - MH] = (float)v;
  else if (x < 3 * MH + 1)
    grads[L.W3() + x - 2 * MH] = (float)v;  // and b3, which follows
  else
    *loss = (float)v;
}

// column sums of X[rows x cols] into out[cols]
__global__ void k_colsum(const float *__restrict__ X, int rows, int cols, float *__restrict__ out) {
  const int c = blockIdx.x;
  float s = 0.f;
  for (int r = threadIdx.x; r < rows; r += blockDim.x) s += X[(size_t)r * cols + c];
  __shared__ float sm[256];
  sm[threadIdx.x] = s;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sm[threadIdx.x] += sm[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = sm[0];
}

__global__ void k_feat_to_f32(const int32_t *__restrict__ f, size_t n, float scale, float *__restrict__ x) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = (float)f[i] * scale;
}

// dY = (Y - T) / n ; partial loss sums (one per block)
__global__ void k_mse_grad(const float *__restrict__ Y, const float *__restrict__ T, int n, float *__restrict__ dY,
                           float *__restrict__ part) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.f;
  if (i < n) {
    const float d = Y[i] - T[i];
    dY[i] = d / (float)n;
    l = 0.5f * d * d / (float)n;
  }
  __shared__ float sm[256];
  sm[threadIdx.x] = l;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sm[threadIdx.x] += sm[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sm[0];
}

__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                       size_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void k_to_bf16(const float *__restrict__ src, size_t n, uint16_t *__restrict__ dst) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = f32_to_bf16(src[i]);
}

}  // namespace gemd

using namespace gemd;

struct gem_mlp {
  gem_ctx *ctx;
  uint32_t in, h;
  size_t P;
  // offsets into the flat parameter vector
  size_t oW1, ob1, oW2, ob2, oW3, ob3;
  DevBuf params, grads, adam_m, adam_v, wbf;  // wbf: bf16 W1 | W2 | W3
  uint64_t adam_t = 0;
  float margin = 0.f;  // a candidate replaces GEM's order only if predicted cheaper by more
};

namespace {

void refresh_bf16(gem_mlp *m) {
  hipStream_t s = m->ctx->stream;
  const float *p = m->params.as<float>();
  uint16_t *b = m->wbf.as<uint16_t>();
  const size_t n1 = (size_t)m->in * m->h, n2 = (size_t)m->h * m->h, n3 = m->h;
  k_to_bf16<<<(uint32_t)((n1 + 255) / 256), 256, 0, s>>>(p + m->oW1, n1, b);
  k_to_bf16<<<(uint32_t)((n2 + 255) / 256), 256, 0, s>>>(p + m->oW2, n2, b + n1);
  k_to_bf16<<<(uint32_t)((n3 + 255) / 256), 256, 0, s>>>(p + m->oW3, n3, b + n1 + n2);
  GEM_LAUNCH_CHECK("k_to_bf16");
}

template <bool TA, bool TB, bool BBF, int EPI>
void gemm(hipStream_t s, int M, int N, int K, const float *A, int lda, const void *B, int ldb, const float *bias,
          const float *mask, float *C, int ldc) {
  dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
  k_gemm<TA, TB, BBF, EPI><<<grid, 256, 0, s>>>(M, N, K, A, lda, B, ldb, bias, mask, C, ldc);
  GEM_LAUNCH_CHECK("k_gemm");
}

// Rows up to which a forward block takes 8 rows at a time (more blocks, less
// work each); beyond, 32 (each weight read from LDS serves four rows).
constexpr uint32_t SMALL_ROWS = 2048;
constexpr uint32_t MLP_BLOCKS = 256;

bool wide(const gem_mlp *m) { return m->h == MH && m->in % 16 == 0 && m->in <= MF_MAX; }

size_t forward_lds(uint32_t F, uint32_t R) {
  const size_t rows = std::max<size_t>((size_t)8 * R * F, (size_t)8 * R * MROW);
  return 4 * ((size_t)(F + MH) / 2 * MH + MH + 8 * R * MROW + rows);
}

// A training set on the device.
struct DevSet {
  DevBuf feats, targets;
  uint32_t n = 0;
};

void upload(gem_mlp *m, const int32_t *h_feat, const float *h_target, uint32_t n, DevSet &d) {
  hipStream_t s = m->ctx->stream;
  d.n = n;
  d.feats.alloc((size_t)n * m->in * 4, s);
  GEM_HIP_CHECK(hipMemcpyAsync(d.feats.p, h_feat, (size_t)n * m->in * 4, hipMemcpyHostToDevice, s));
  if (!h_target) return;
  d.targets.alloc((size_t)n * 4, s);
  GEM_HIP_CHECK(hipMemcpyAsync(d.targets.p, h_target, (size_t)n * 4, hipMemcpyHostToDevice, s));
}

struct Acts {
  DevBuf X, H1, H2, Y;
};

template <int R, bool STORE>
void launch_forward(gem_mlp *m, const DevSet &d, Acts &a) {
  const uint32_t blocks = std::min<uint32_t>((d.n + 8 * R - 1) / (8 * R), MLP_BLOCKS);
  const size_t lds = forward_lds(m->in, R);
  GEM_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mlp_forward<R, STORE>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_mlp_forward<R, STORE><<<blocks, 1024, lds, m->ctx->stream>>>(d.feats.as<int32_t>(), d.n, MlpLayout{m->in},
                                                                 m->params.as<float>(), m->wbf.as<uint16_t>(),
                                                                 a.H1.as<float>(), a.H2.as<float>(), a.Y.as<float>());
  GEM_LAUNCH_CHECK("k_mlp_forward");
}

// Loss and gradients of a wide model (grads and *d_loss on the device).
void gradient_wide(gem_mlp *m, const DevSet &d, Acts &a, float *d_loss) {
  hipStream_t s = m->ctx->stream;
  const uint32_t n = d.n, F = m->in;
  const MlpLayout L{F};
  DevBuf dH1, dH2, part, wpart;
  dH1.alloc((size_t)n * MH * 4, s);
  dH2.alloc((size_t)n * MH * 4, s);
  const bool small = n <= SMALL_ROWS;
  const uint32_t blocks = std::min<uint32_t>(small ? (n + 7) / 8 : (n + 31) / 32, MLP_BLOCKS);
  part.alloc((size_t)blocks * MPART * 4, s);
  auto rows = small ? k_mlp_backward<1> : k_mlp_backward<4>;
  rows<<<blocks, 1024, 0, s>>>(a.Y.as<float>(), d.targets.as<float>(), n, L, m->wbf.as<uint16_t>(), a.H1.as<float>(),
                               a.H2.as<float>(), dH1.as<float>(), dH2.as<float>(), part.as<float>());
  GEM_LAUNCH_CHECK("k_mlp_backward");
  // slices of at least 64 samples, at most 64 of them: 25 tiles of 16 rows
  // (272 inputs) x 64 are 1,600 waves
  const uint32_t slice = std::max<uint32_t>(64, ((n + 63) / 64 + 3) / 4 * 4), slices = (n + slice - 1) / slice;
  wpart.alloc((size_t)slices * (F + MH) * MH * 4, s);
  k_mlp_wgrad<<<dim3(((F + MH) / 16 + 3) / 4, slices), 256, 0, s>>>(d.feats.as<int32_t>(), a.H1.as<float>(),
                                                                    dH1.as<float>(), dH2.as<float>(), n, F, slice,
                                                                    wpart.as<float>());
  GEM_LAUNCH_CHECK("k_mlp_wgrad");
  k_mlp_reduce<<<(F + MH) * MH / 256 + (MPART + 3) / 4, 256, 0, s>>>(wpart.as<float>(), slices, part.as<float>(), blocks,
                                                                   L, m->grads.as<float>(), d_loss);
  GEM_LAUNCH_CHECK("k_mlp_reduce");
}

// store: keep the hidden rows, for a backward pass.
void forward(gem_mlp *m, const DevSet &d, Acts &a, bool store) {
  hipStream_t s = m->ctx->stream;
  const uint32_t n = d.n;
  const size_t nf = (size_t)n * m->in;
  a.Y.alloc((size_t)n * 4, s);
  if (store || !wide(m)) {
    a.H1.alloc((size_t)n * m->h * 4, s);
    a.H2.alloc((size_t)n * m->h * 4, s);
  }
  if (wide(m)) {
    if (n <= SMALL_ROWS)
      store ? launch_forward<1, true>(m, d, a) : launch_forward<1, false>(m, d, a);
    else
      store ? launch_forward<4, true>(m, d, a) : launch_forward<4, false>(m, d, a);
    return;
  }
  a.X.alloc(nf * 4, s);
  k_feat_to_f32<<<(uint32_t)((nf + 255) / 256), 256, 0, s>>>(d.feats.as<int32_t>(), nf, FEAT_SCALE, a.X.as<float>());
  GEM_LAUNCH_CHECK("k_feat_to_f32");
  const float *p = m->params.as<float>();
  const uint16_t *wb = m->wbf.as<uint16_t>();
  const int H = (int)m->h, F = (int)m->in;
  gemm<false, false, true, 1>(s, n, H, F, a.X.as<float>(), F, wb, H, p + m->ob1, nullptr, a.H1.as<float>(), H);
  gemm<false, false, true, 1>(s, n, H, H, a.H1.as<float>(), H, wb + (size_t)F * H, H, p + m->ob2, nullptr,
                              a.H2.as<float>(), H);
  gemm<false, false, true, 2>(s, n, 1, H, a.H2.as<float>(), H, wb + (size_t)F * H + (size_t)H * H, 1, p + m->ob3,
                              nullptr, a.Y.as<float>(), 1);
}

// Loss and gradients; m->grads holds the gradients.
float backward(gem_mlp *m, const DevSet &d, Acts &a) {
  hipStream_t s = m->ctx->stream;
  const uint32_t n = d.n;
  if (wide(m)) {
    DevBuf dl;
    dl.alloc(4, s);
    gradient_wide(m, d, a, dl.as<float>());
    float *h = pinned<float>(m->ctx, 1);
    GEM_HIP_CHECK(hipMemcpyAsync(h, dl.p, 4, hipMemcpyDeviceToHost, s));
    GEM_HIP_CHECK(hipStreamSynchronize(s));
    return *h;
  }
  const int H = (int)m->h, F = (int)m->in;
  DevBuf dY, dH2, dH1, part;
  dY.alloc((size_t)n * 4, s);
  dH2.alloc((size_t)n * H * 4, s);
  dH1.alloc((size_t)n * H * 4, s);
  const uint32_t nb = (n + 255) / 256;
  part.alloc(nb * 4, s);
  k_mse_grad<<<nb, 256, 0, s>>>(a.Y.as<float>(), d.targets.as<float>(), (int)n, dY.as<float>(), part.as<float>());
  GEM_LAUNCH_CHECK("k_mse_grad");
  float *g = m->grads.as<float>();
  const uint16_t *wb = m->wbf.as<uint16_t>();
  const uint16_t *W2b = wb + (size_t)F * H, *W3b = wb + (size_t)F * H + (size_t)H * H;
  // layer 3
  gemm<true, false, false, 0>(s, H, 1, n, a.H2.as<float>(), H, dY.as<float>(), 1, nullptr, nullptr, g + m->oW3, 1);
  k_colsum<<<1, 256, 0, s>>>(dY.as<float>(), (int)n, 1, g + m->ob3);
  gemm<false, false, true, 3>(s, n, H, 1, dY.as<float>(), 1, W3b, H, nullptr, a.H2.as<float>(), dH2.as<float>(), H);
  // layer 2
  gemm<true, false, false, 0>(s, H, H, n, a.H1.as<float>(), H, dH2.as<float>(), H, nullptr, nullptr, g + m->oW2, H);
  k_colsum<<<H, 256, 0, s>>>(dH2.as<float>(), (int)n, H, g + m->ob2);
  gemm<false, true, true, 3>(s, n, H, H, dH2.as<float>(), H, W2b, H, nullptr, a.H1.as<float>(), dH1.as<float>(), H);
  // layer 1
  gemm<true, false, false, 0>(s, F, H, n, a.X.as<float>(), F, dH1.as<float>(), H, nullptr, nullptr, g + m->oW1, H);
  k_colsum<<<H, 256, 0, s>>>(dH1.as<float>(), (int)n, H, g + m->ob1);
  GEM_LAUNCH_CHECK("k_colsum");
  std::vector<float> hp(nb);
  GEM_HIP_CHECK(hipMemcpyAsync(hp.data(), part.p, nb * 4, hipMemcpyDeviceToHost, s));
  GEM_HIP_CHECK(hipStreamSynchronize(s));
  double loss = 0;
  for (float x : hp) loss += x;
  return (float)loss;
}

template <class F>
int mguard(gem_mlp *m, F &&f) {
  if (!m) return GEM_E_INVALID;
  if (!m->ctx) return GEM_E_STATE;  // its context was destroyed first
  try {
    GEM_HIP_CHECK(hipSetDevice(m->ctx->device));
    f();
    return GEM_OK;
  } catch (const Error &e) {
    m->ctx->err = e.msg;
    return e.code;
  } catch (const std::exception &e) {
    m->ctx->err = e.what();
    return GEM_E_INVALID;
  }
}

}  // namespace

namespace gemd {
float mlp_margin(const gem_mlp *m) { return m->margin; }

void mlp_detach(gem_mlp *m) {
  m->params.reset();
  m->grads.reset();
  m->adam_m.reset();
  m->adam_v.reset();
  m->wbf.reset();
  m->ctx = nullptr;
}
}  // namespace gemd

extern "C" {

int gem_mlp_create(gem_ctx *ctx, uint32_t in_dim, uint32_t hidden, uint64_t seed, gem_mlp **out) {
  if (!ctx || !out || in_dim == 0 || hidden == 0) return GEM_E_INVALID;
  auto *m = new gem_mlp();
  m->ctx = ctx;
  m->in = in_dim;
  m->h = hidden;
  m->oW1 = 0;
  m->ob1 = m->oW1 + (size_t)in_dim * hidden;
  m->oW2 = m->ob1 + hidden;
  m->ob2 = m->oW2 + (size_t)hidden * hidden;
  m->oW3 = m->ob2 + hidden;
  m->ob3 = m->oW3 + hidden;
  m->P = m->ob3 + 1;
  int st = mguard(m, [&]() {
    hipStream_t s = ctx->stream;
    m->params.alloc(m->P * 4, s);
    m->grads.alloc(m->P * 4, s);
    m->adam_m.alloc(m->P * 4, s);
    m->adam_v.alloc(m->P * 4, s);
    m->wbf.alloc(((size_t)in_dim * hidden + (size_t)hidden * hidden + hidden) * 2, s);
    // He-uniform weights, zero biases (seeded, host side)
    std::vector<float> p(m->P, 0.f);
    gemh::Rng rng(seed);
    auto fill = [&](size_t o, size_t cnt, double fan_in) {
      const double lim = std::sqrt(6.0 / fan_in);
      for (size_t i = 0; i < cnt; ++i) p[o + i] = (float)((2.0 * rng.uniform() - 1.0) * lim);
    };
    fill(m->oW1, (size_t)in_dim * hidden, in_dim);
    fill(m->oW2, (size_t)hidden * hidden, hidden);
    fill(m->oW3, hidden, hidden);
    GEM_HIP_CHECK(hipMemcpyAsync(m->params.p, p.data(), m->P * 4, hipMemcpyHostToDevice, s));
    GEM_HIP_CHECK(hipMemsetAsync(m->adam_m.p, 0, m->P * 4, s));
    GEM_HIP_CHECK(hipMemsetAsync(m->adam_v.p, 0, m->P * 4, s));
    refresh_bf16(m);
    GEM_HIP_CHECK(hipStreamSynchronize(s));
  });
  if (st) {
    delete m;
    return st;
  }
  ctx->mlps.push_back(m);
  *out = m;
  return GEM_OK;
}

void gem_mlp_destroy(gem_mlp *m) {
  if (!m) return;
  if (gem_ctx *c = m->ctx) {
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    c->mlps.erase(std::remove(c->mlps.begin(), c->mlps.end(), m), c->mlps.end());
  }
  delete m;
}

uint64_t gem_mlp_num_params(const gem_mlp *m) { return m ? m->P : 0; }

int gem_mlp_set_margin(gem_mlp *m, float margin) {
  if (!m || !(margin >= 0.f)) return GEM_E_INVALID;
  m->margin = margin;
  return GEM_OK;
}

int gem_mlp_get_params(gem_mlp *m, float *out) {
  return mguard(m, [&]() {
    if (!out) throw Error{GEM_E_INVALID, "null output"};
    GEM_HIP_CHECK(hipMemcpyAsync(out, m->params.p, m->P * 4, hipMemcpyDeviceToHost, m->ctx->stream));
    GEM_HIP_CHECK(hipStreamSynchronize(m->ctx->stream));
  });
}

int gem_mlp_set_params(gem_mlp *m, const float *in) {
  return mguard(m, [&]() {
    if (!in) throw Error{GEM_E_INVALID, "null input"};
    GEM_HIP_CHECK(hipMemcpyAsync(m->params.p, in, m->P * 4, hipMemcpyHostToDevice, m->ctx->stream));
    refresh_bf16(m);
    GEM_HIP_CHECK(hipStreamSynchronize(m->ctx->stream));
  });
}

int gem_mlp_predict(gem_mlp *m, const int32_t *feats, uint32_t n, float *out) {
  return mguard(m, [&]() {
    if (!n) return;
    if (!feats || !out) throw Error{GEM_E_INVALID, "null argument"};
    Acts a;
    DevSet d;
    upload(m, feats, nullptr, n, d);
    forward(m, d, a, false);
    GEM_HIP_CHECK(hipMemcpyAsync(out, a.Y.p, (size_t)n * 4, hipMemcpyDeviceToHost, m->ctx->stream));
    GEM_HIP_CHECK(hipStreamSynchronize(m->ctx->stream));
  });
}

int gem_mlp_loss_grad(gem_mlp *m, const int32_t *feats, const float *targets, uint32_t n, float *loss, float *grad) {
  return mguard(m, [&]() {
    if (!n || !feats || !targets) throw Error{GEM_E_INVALID, "empty or null batch"};
    Acts a;
    DevSet d;
    upload(m, feats, targets, n, d);
    forward(m, d, a, true);
    const float l = backward(m, d, a);
    if (loss) *loss = l;
    if (grad) {
      GEM_HIP_CHECK(hipMemcpyAsync(grad, m->grads.p, m->P * 4, hipMemcpyDeviceToHost, m->ctx->stream));
      GEM_HIP_CHECK(hipStreamSynchronize(m->ctx->stream));
    }
  });
}

int gem_mlp_train(gem_mlp *m, const int32_t *feats, const float *targets, uint32_t n, uint32_t iters, float lr,
                  float *losses) {
  return mguard(m, [&]() {
    if (!n || !feats || !targets) throw Error{GEM_E_INVALID, "empty or null batch"};
    hipStream_t s = m->ctx->stream;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    DevSet d;
    upload(m, feats, targets, n, d);
    for (uint32_t it = 0; it < iters; ++it) {
      Acts a;
      forward(m, d, a, true);
      const float l = backward(m, d, a);
      if (losses) losses[it] = l;
      ++m->adam_t;
      const float c1 = 1.f - std::pow(b1, (float)m->adam_t), c2 = 1.f - std::pow(b2, (float)m->adam_t);
      k_adam<<<(uint32_t)((m->P + 255) / 256), 256, 0, s>>>(m->params.as<float>(), m->grads.as<float>(),
                                                            m->adam_m.as<float>(), m->adam_v.as<float>(), m->P, lr, b1,
                                                            b2, eps, c1, c2);
      GEM_LAUNCH_CHECK("k_adam");
      refresh_bf16(m);
    }
    GEM_HIP_CHECK(hipStreamSynchronize(s));
  });
}

}  // extern "C"
