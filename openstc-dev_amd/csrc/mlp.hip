// BF16 MFMA kernels of the chemistry surrogate MLP (gfx950).
//
// One tiled GEMM covers every product of training and inference:
//   C[M x N] = op(A)[M x K] * op(B)[K x N]      (f32 accumulation)
// with op = identity or transpose of row-major operands held in FP32 or
// BF16, staged through LDS as BF16, multiplied with
// v_mfma_f32_16x16x32_bf16 and finished by a fused epilogue (bias, GELU,
// GELU' of a saved pre-activation, FP32 / BF16 stores, or FP32 atomic
// accumulation for split-K weight gradients).
//
// Tile: 64 x 64 outputs per workgroup of 4 wavefronts (each 32 x 32 = 2 x 2
// MFMA tiles), K step 64, the next step's operands loaded into registers
// while the current one is multiplied.  The products of a mini-batch are
// short (K = 24 to 264 forward, shares of 256 or 384 of 8,192 rows backward), so
// a tile's time is a few global-load latencies: K steps of 32 that waited for
// their own loads, with LDS moved in 2-byte pieces, took 13 / 17 / 20 us for
// the forward, input-gradient and weight-gradient products of 8,192 rows;
// this takes 10.5 / 15.5 / 14.0 us.
// LDS rows are 68 BF16 long: the 8-byte reads of a fragment and the 4-byte
// writes of a transposed operand (two K rows paired) spread over the banks.
//
// MFMA 16x16x32 BF16 operand layout (lane l of a wave64):
//   A fragment: row l%16, k = 8*(l/16) + 0..7
//   B fragment: col l%16, k = 8*(l/16) + 0..7
//   C/D f32x4 : col l%16, row = 4*(l/16) + 0..3
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "mlp.h"

namespace ostc {

namespace {

constexpr int BM = 64, BN = 64, BK = 64, LDK = 68;

__device__ inline __bf16 to_bf(float x) { return (__bf16)x; }
__device__ inline float from_bf(__bf16 x) { return (float)x; }

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;

// eight consecutive values as one or two 16-byte loads (launch_gemm checks
// the alignment)
template <typename T>
struct Oct;
template <>
struct Oct<float> {
  f32x4 lo, hi;
  __device__ void load(const float *p) {
    lo = *(const f32x4 *)p;
    hi = *(const f32x4 *)(p + 4);
  }
  __device__ void clear() { lo = hi = f32x4{0.f, 0.f, 0.f, 0.f}; }
  __device__ __bf16 bf(int e) const { return to_bf(e < 4 ? lo[e & 3] : hi[e & 3]); }
};
template <>
struct Oct<__bf16> {
  bf16x8 v;
  __device__ void load(const __bf16 *p) { v = *(const bf16x8 *)p; }
  __device__ void clear() {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (__bf16)0.f;
  }
  __device__ __bf16 bf(int e) const { return v[e]; }
};

// One operand's 64 x 64 tile, 16 values a thread: rows of the tile are the
// operand's M (or N) index, columns its K index.  KMAJOR: stored K x M, M
// contiguous -- the thread holds 8 values of two adjacent K rows and writes
// them in pairs; otherwise M x K, K contiguous.
template <typename T>
struct TileLoader {
  Oct<T> a, b;

  __device__ void load(bool kmajor, const T *p, int ld, int m0, int M, int k0, int k1, int tid) {
    a.clear();
    b.clear();
    if (!kmajor) {
      const int m = m0 + (tid >> 2), k = k0 + (tid & 3) * 16;
      if (m < M) {
        const T *q = p + (int64_t)m * ld + k;
        if (k < k1) a.load(q);
        if (k + 8 < k1) b.load(q + 8);
      }
    } else {
      const int k = k0 + (tid >> 3) * 2, m = m0 + (tid & 7) * 8;
      if (m < M) {
        const T *q = p + (int64_t)k * ld + m;
        if (k < k1) a.load(q);
        if (k + 1 < k1) b.load(q + ld);
      }
    }
  }

  __device__ void store(bool kmajor, __bf16 (*t)[LDK], int tid) const {
    if (!kmajor) {
      __bf16 *q = &t[tid >> 2][(tid & 3) * 16];
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        *(bf16x4 *)(q + e) = bf16x4{a.bf(e), a.bf(e + 1), a.bf(e + 2), a.bf(e + 3)};
        *(bf16x4 *)(q + 8 + e) = bf16x4{b.bf(e), b.bf(e + 1), b.bf(e + 2), b.bf(e + 3)};
      }
    } else {
      const int k = (tid >> 3) * 2, m = (tid & 7) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) *(bf16x2 *)&t[m + e][k] = bf16x2{a.bf(e), b.bf(e)};
    }
  }
};

template <typename TA, typename TB>
__global__ void __launch_bounds__(256) k_gemm(GemmArgs g, const TA *__restrict__ A, const TB *__restrict__ B) {
  __shared__ __attribute__((aligned(16))) __bf16 As[BM][LDK];
  __shared__ __attribute__((aligned(16))) __bf16 Bs[BN][LDK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  // split-K: blockIdx.z owns K range [kz0, kz1)
  // (chunks are whole K steps so every 8-element load stays 16-byte aligned)
  const int kchunk = (((g.K + (int)gridDim.z - 1) / (int)gridDim.z) + BK - 1) / BK * BK;
  const int kz0 = blockIdx.z * kchunk, kz1 = min(g.K, kz0 + kchunk);
  const bool ka = g.transA != 0, kb = g.transB == 0;  // operand stored with K as its row
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  TileLoader<TA> la;
  TileLoader<TB> lb;
  if (kz0 < kz1) {
    la.load(ka, A, g.lda, m0, g.M, kz0, kz1, tid);
    lb.load(kb, B, g.ldb, n0, g.N, kz0, kz1, tid);
  }
  for (int k0 = kz0; k0 < kz1; k0 += BK) {
    la.store(ka, As, tid);
    lb.store(kb, Bs, tid);
    __syncthreads();
    if (k0 + BK < kz1) {
      la.load(ka, A, g.lda, m0, g.M, k0 + BK, kz1, tid);
      lb.load(kb, B, g.ldb, n0, g.N, k0 + BK, kz1, tid);
    }
#pragma unroll
    for (int ks = 0; ks < BK; ks += 32) {
      bf16x8 af[2], bfr[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const __bf16 *ra = &As[wm * 32 + t * 16 + (lane & 15)][ks + 8 * (lane >> 4)];
        const __bf16 *rb = &Bs[wn * 32 + t * 16 + (lane & 15)][ks + 8 * (lane >> 4)];
        const bf16x4 a0 = *(const bf16x4 *)ra, a1 = *(const bf16x4 *)(ra + 4);
        const bf16x4 b0 = *(const bf16x4 *)rb, b1 = *(const bf16x4 *)(rb + 4);
        af[t] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
        bfr[t] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0);
    }
    __syncthreads();
  }

  // ---- epilogue ----
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = m0 + wm * 32 + a * 16 + 4 * (lane >> 4) + e;
        const int col = n0 + wn * 32 + b * 16 + (lane & 15);
        if (row >= g.M || col >= g.N) continue;
        float v = acc[a][b][e];
        const int64_t o = (int64_t)row * g.ldc + col;
        if (g.mode == EPI_ATOMIC) {
          atomicAdd(&g.Cf[o], v);
          continue;
        }
        if (g.bias) v += g.bias[col];
        if (g.mode == EPI_GELU) {
          if (g.Z) g.Z[o] = v;
          v = gelu(v);
        } else if (g.mode == EPI_GELU_GRAD) {
          v *= gelu_grad(g.Zin[o]);
        }
        if (g.Cf) g.Cf[o] = v;
        if (g.Cb) g.Cb[o] = to_bf(v);
      }
}

}  // namespace

hipError_t launch_gemm(const GemmArgs &g, const void *A, bool a_bf16, const void *B, bool b_bf16, int split_k,
                       hipStream_t s) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return hipSuccess;
  auto r8 = [](int v) { return (v + 7) / 8 * 8; };
  // every 8-wide operand load must stay inside its row
  if (g.K % 8 || g.lda % 8 || g.ldb % 8) return hipErrorInvalidValue;
  if (g.transA ? g.lda < r8(g.M) : g.lda < g.K) return hipErrorInvalidValue;
  if (g.transB ? g.ldb < g.K : g.ldb < r8(g.N)) return hipErrorInvalidValue;
  if (g.ldc < g.N || (!g.Cf && !g.Cb)) return hipErrorInvalidValue;
  if (g.mode == EPI_ATOMIC && !g.Cf) return hipErrorInvalidValue;
  if (g.mode == EPI_GELU_GRAD && !g.Zin) return hipErrorInvalidValue;
  if (((uintptr_t)A | (uintptr_t)B) % 16) return hipErrorInvalidValue;
  if (split_k < 1) split_k = 1;
  if (split_k > 1 && g.mode != EPI_ATOMIC) return hipErrorInvalidValue;
  // shares are whole K steps (k_gemm), so fewer than asked for may cover K; an
  // empty one would only add zeros to every output
  const int share = ((g.K + split_k - 1) / split_k + BK - 1) / BK * BK;
  split_k = (g.K + share - 1) / share;
  const dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM, split_k), blk(256);
  if (a_bf16 && b_bf16)
    hipLaunchKernelGGL((k_gemm<__bf16, __bf16>), grid, blk, 0, s, g, (const __bf16 *)A, (const __bf16 *)B);
  else if (a_bf16 && !b_bf16)
    hipLaunchKernelGGL((k_gemm<__bf16, float>), grid, blk, 0, s, g, (const __bf16 *)A, (const float *)B);
  else if (!a_bf16 && b_bf16)
    hipLaunchKernelGGL((k_gemm<float, __bf16>), grid, blk, 0, s, g, (const float *)A, (const __bf16 *)B);
  else
    hipLaunchKernelGGL((k_gemm<float, float>), grid, blk, 0, s, g, (const float *)A, (const float *)B);
  return hipGetLastError();
}

namespace {

__global__ void k_to_bf16(const float *__restrict__ src, __bf16 *__restrict__ dst, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = to_bf(src[i]);
}

__global__ void k_fill_cols_bf16(__bf16 *__restrict__ dst, int64_t rows, int cols, int c0,
                                 const float *__restrict__ vals) {
  const int w = cols - c0;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * w) return;
  const int64_t r = i / w;
  const int c = (int)(i - r * w);
  dst[r * cols + c0 + c] = to_bf(vals[c]);
}

// MSE over the first nout of ld columns: loss = sum (y - t)^2 / (M nout),
// G = d loss / d y (zero in the padding columns).  At most kMseBlocks
// workgroups, since each adds its share to one address and those additions
// queue up: 8,192 rows of 16 8.3 -> 6.4 us, 65,536 rows 54 -> 38 us, 131,072
// rows 107 -> 73 us against a workgroup per 256 values
constexpr int kMseBlocks = 64;
__global__ void k_mse(const float *__restrict__ Y, const float *__restrict__ T, int M, int nout, int ld,
                      float *__restrict__ G, float *__restrict__ loss_acc) {
  float l = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < (int64_t)M * ld; i += (int64_t)gridDim.x * 256) {
    const int c = (int)(i % ld);
    float g = 0.f;
    if (c < nout) {
      const float d = Y[i] - T[i];
      l += d * d;
      g = 2.f * d / ((float)M * (float)nout);
    }
    G[i] = g;
  }
  for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
  __shared__ float part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float b = part[0] + part[1] + part[2] + part[3];
    if (b != 0.f) atomicAdd(loss_acc, b / ((float)M * (float)nout));
  }
}

// Adam with bias correction on FP32 master weights
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m1, float *__restrict__ m2,
                       int64_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  w[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// gather rows idx[0..m) of a row-major matrix with `cols` columns
template <typename T>
__global__ void k_gather_rows(const T *__restrict__ src, const int *__restrict__ idx, int m, int cols,
                              T *__restrict__ dst) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)m * cols) return;
  const int r = (int)(i / cols), c = (int)(i % cols);
  dst[i] = src[(int64_t)idx[r] * cols + c];
}

inline unsigned nb(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

hipError_t launch_to_bf16(const float *src, __bf16 *dst, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_to_bf16, dim3(nb(n)), dim3(256), 0, s, src, dst, n);
  return hipGetLastError();
}

hipError_t launch_fill_cols_bf16(__bf16 *dst, int64_t rows, int cols, int c0, const float *vals, hipStream_t s) {
  if (rows <= 0 || c0 >= cols) return hipSuccess;
  hipLaunchKernelGGL(k_fill_cols_bf16, dim3(nb(rows * (cols - c0))), dim3(256), 0, s, dst, rows, cols, c0, vals);
  return hipGetLastError();
}

hipError_t launch_mse(const float *Y, const float *T, int M, int nout, int ld, float *G, float *loss_acc,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_mse, dim3(std::min<unsigned>(kMseBlocks, nb((int64_t)M * ld))), dim3(256), 0, s, Y, T, M, nout, ld, G, loss_acc);
  return hipGetLastError();
}

hipError_t launch_adam(float *w, const float *g, float *m1, float *m2, int64_t n, float lr, float b1, float b2,
                       float eps, int step, hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(nb(n)), dim3(256), 0, s, w, g, m1, m2, n, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t launch_gather_rows_bf16(const __bf16 *src, const int *idx, int m, int cols, __bf16 *dst, hipStream_t s) {
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_rows<__bf16>, dim3(nb((int64_t)m * cols)), dim3(256), 0, s, src, idx, m, cols, dst);
  return hipGetLastError();
}

hipError_t launch_gather_rows_f32(const float *src, const int *idx, int m, int cols, float *dst, hipStream_t s) {
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_rows<float>, dim3(nb((int64_t)m * cols)), dim3(256), 0, s, src, idx, m, cols, dst);
  return hipGetLastError();
}

}  // namespace ostc
