// Rank-predictor MLP on the GPU: forward, backward and Adam, complex-free
// FP32 (the learned part of the chosen form; no counterpart in the
// reference).
//
// Network: y = W3 gelu(W2 gelu(W1 a0 + b1) + b2) + b3 with a0 the input
// column (nin features; the first min(64, nin), the previous bond spectrum,
// enter as log10(max(x, 1e-16)) / 8, i.e. in [-2, 0]).  Activations are column-major (features x
// batch).  Parameters are one flat float array: W1 (width x nin), b1, W2
// (width x width), b2, W3 (1 x width), b3, each block column-major.
// GELU is the exact form 0.5 z (1 + erf(z / sqrt 2)).
#include <algorithm>
#include <cmath>
#include <vector>

#include "qtn_internal.hpp"

struct qtn_mlp {
  qtn_ctx* ctx = nullptr;
  int nin = 0, width = 0;
  int64_t np = 0;          // number of parameters
  float* params = nullptr; // device
  float* grads = nullptr;
  float* m1 = nullptr;     // Adam moments
  float* m2 = nullptr;
  int64_t step = 0;
  void* arena = nullptr;
};

namespace qtn {
namespace {

constexpr int kSlotA0 = 100, kSlotZ1 = 101, kSlotA1 = 102, kSlotZ2 = 103,
              kSlotA2 = 104, kSlotY = 105, kSlotD1 = 106, kSlotD2 = 107,
              kSlotIn = 108, kSlotT = 109, kSlotLoss = 110, kSlotPart = 111;
constexpr int kNLog = 64;

unsigned grid_for(int64_t n) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256,
                                                          8192));
}

// C (M x N) = op(A) op(B) [+ bias broadcast over columns] [+ C], FP32,
// column-major.  op(A) is A (M x K, lda) or A^T (A is K x M); op(B) is B
// (K x N) or B^T.  32 x 32 output tile per 256-thread block, 4 per thread,
// K staged through LDS in slices of 16.
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void sgemm(int64_t M, int64_t N, int64_t K,
                                             const float* __restrict__ A,
                                             int64_t lda,
                                             const float* __restrict__ B,
                                             int64_t ldb, float* __restrict__ C,
                                             int64_t ldc,
                                             const float* __restrict__ bias,
                                             int accumulate) {
  __shared__ float As[16][33];  // [k][m]
  __shared__ float Bs[16][33];  // [k][n]
  const int tid = threadIdx.x;
  const int64_t m0 = (int64_t)blockIdx.x * 32, n0 = (int64_t)blockIdx.y * 32;
  const int tm = tid % 32, tn = tid / 32;  // tn 0..7, each 4 columns
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t k0 = 0; k0 < K; k0 += 16) {
    for (int idx = tid; idx < 16 * 32; idx += 256) {
      const int kk = idx / 32, i = idx % 32;
      const int64_t gm = m0 + i, gk = k0 + kk;
      float a = 0.f;
      if (gm < M && gk < K) a = TA ? A[gk + gm * lda] : A[gm + gk * lda];
      As[kk][i] = a;
      const int64_t gn = n0 + i;
      float b = 0.f;
      if (gn < N && gk < K) b = TB ? B[gn + gk * ldb] : B[gk + gn * ldb];
      Bs[kk][i] = b;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const float a = As[kk][tm];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += a * Bs[kk][tn * 4 + j];
    }
    __syncthreads();
  }
  const int64_t gm = m0 + tm;
  if (gm >= M) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t gn = n0 + tn * 4 + j;
    if (gn >= N) continue;
    float v = acc[j];
    if (bias) v += bias[gm];
    if (accumulate) v += C[gm + gn * ldc];
    C[gm + gn * ldc] = v;
  }
}

template <bool TA, bool TB>
int32_t launch_sgemm(hipStream_t s, int64_t M, int64_t N, int64_t K,
                     const float* A, int64_t lda, const float* B, int64_t ldb,
                     float* C, int64_t ldc, const float* bias,
                     int accumulate) {
  dim3 grid((unsigned)((M + 31) / 32), (unsigned)((N + 31) / 32));
  hipLaunchKernelGGL((sgemm<TA, TB>), grid, dim3(256), 0, s, M, N, K, A, lda,
                     B, ldb, C, ldc, bias, accumulate);
  QTN_CHECK_HIP(hipGetLastError());
  return QTN_OK;
}

__global__ void prep_input(const float* __restrict__ X, int nin, int64_t nb,
                           float* __restrict__ A0) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
       i < (int64_t)nin * nb; i += (int64_t)gridDim.x * blockDim.x) {
    const int f = (int)(i % nin);
    const float x = X[i];
    A0[i] = f < kNLog ? 0.125f * log10f(fmaxf(x, 1e-16f)) : x;
  }
}

__device__ __forceinline__ float gelu_f(float z) {
  return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
}

__device__ __forceinline__ float gelu_d(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) +
         z * expf(-0.5f * z * z) * 0.39894228040143268f;
}

__global__ void gelu_fwd(const float* __restrict__ Z, float* __restrict__ A,
                         int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    A[i] = gelu_f(Z[i]);
}

// D <- D * gelu'(Z)
__global__ void gelu_bwd(const float* __restrict__ Z, float* __restrict__ D,
                         int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    D[i] *= gelu_d(Z[i]);
}

// dY = 2 (Y - T) / nb; loss[0] = sum (Y - T)^2 / nb (one workgroup).
__global__ __launch_bounds__(256) void mse_grad(const float* __restrict__ Y,
                                                const float* __restrict__ T,
                                                int64_t nb,
                                                float* __restrict__ dY,
                                                float* __restrict__ loss) {
  float s = 0.f;
  const float inv = 1.0f / (float)nb;
  for (int64_t i = threadIdx.x; i < nb; i += 256) {
    const float r = Y[i] - T[i];
    dY[i] = 2.0f * r * inv;
    s += r * r;
  }
  __shared__ float red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = red[0] * inv;
}

// db[r] = sum_b D[r + rows * b] (one wave per row).  grid ceil(rows/4).
__global__ __launch_bounds__(256) void row_sum(const float* __restrict__ D,
                                               int64_t rows, int64_t nb,
                                               float* __restrict__ db) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;
  float s = 0.f;
  for (int64_t b = lane; b < nb; b += 64) s += D[r + rows * b];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) db[r] = s;
}

__global__ void adam_step(float* __restrict__ p, const float* __restrict__ g,
                          float* __restrict__ m1, float* __restrict__ m2,
                          int64_t n, float lr, float b1, float b2, float eps,
                          float c1, float c2) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float v = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = v;
    p[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
  }
}

struct Offsets {
  int64_t W1, b1, W2, b2, W3, b3;
};

Offsets offsets(int nin, int w) {
  Offsets o;
  o.W1 = 0;
  o.b1 = o.W1 + (int64_t)w * nin;
  o.W2 = o.b1 + w;
  o.b2 = o.W2 + (int64_t)w * w;
  o.W3 = o.b2 + w;
  o.b3 = o.W3 + w;
  return o;
}

// ---- one launch per pass ----------------------------------------------------
// Networks of width 16, 32, .. 128 and at most 128 inputs run forward and
// backward in one launch: a workgroup takes 16 samples at a time through all
// layers with the activations in LDS (feature x sample), every product on
// FP32 MFMA tiles of 16 features x 16 samples, and keeps its share of the
// weight gradients in accumulators; a second launch adds the shares and takes
// the Adam step.  The training step is bound by its chain of dependent
// launches: sixteen of them took 146 us at 256 samples (72-128-128-1).
// The two take 27 + 5 us; 128 steps on 4096 samples 18.6 -> 4.5 ms.
typedef float f4_t __attribute__((ext_vector_type(4)));
constexpr int kMaxW = 128, kMaxIn = 128;
constexpr int kAct = 20;       // sample stride of an activation row
constexpr int kMaxGroups = 256;

// Floats of one workgroup's share: the gradient, the loss, 16-byte padding.
__host__ __device__ inline int64_t share_size(int64_t np) {
  return (np + 4) / 4 * 4;
}

// At every batch: gradient of 72-128-128-1, host copies included, layer by
// layer / one pass: 1 sample 0.19 / 0.12 ms, 256 0.29 / 0.17, 4096 1.8 / 0.6,
// 65536 26 / 8.7, 262144 117 / 35 (256 workgroups walk their tiles in series,
// the layers' FP32 products do not use the matrix cores).
bool one_pass(int nin, int w) {
  return w % 16 == 0 && w <= kMaxW && nin <= kMaxIn;
}

__device__ __forceinline__ f4_t mfma4(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The weights of a wave's two row tiles t = wave, wave + 4 of a layer, all
// loaded together once per launch: element s of tile i is W[16 t + l % 16,
// 4 s + l / 16] (W column-major, K columns).  Tiles and columns behind the
// last are read as the last (no select, which would make every load wait for
// the one before): such tiles are not used, such columns are cleared once all
// loads are under way (clear_behind).
__device__ __forceinline__ void load_layer(const float* __restrict__ W, int w,
                                           int K, int wave,
                                           float (&r)[2][32]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float* Wm = W + 16 * min(wave + 4 * i, w / 16 - 1) + (lane & 15);
#pragma unroll
    for (int s = 0; s < 32; ++s)
      r[i][s] = Wm[min(4 * s + (lane >> 4), K - 1) * w];
  }
}

// The same of W^T (W w x w), with the inner indices in the order 16 g +
// 4 (l / 16) + e, s = 4 g + e, so that a lane's four lie together.
__device__ __forceinline__ void load_layer_t(const float* __restrict__ W,
                                             int w, int wave,
                                             float (&r)[2][32]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float* Wm =
        W + (16 * min(wave + 4 * i, w / 16 - 1) + (lane & 15)) * w;
#pragma unroll
    for (int s = 0; s < 32; ++s)
      r[i][s] = Wm[min(16 * (s >> 2) + 4 * (lane >> 4) + (s & 3), w - 1)];
  }
}

// Zero in place of the columns from K on: against zero activations an
// infinite weight read there would give NaN.
__device__ __forceinline__ void clear_behind(int K, float (&r)[2][32]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int s = 0; s < 32; ++s)
    if (4 * s + 4 > K) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        r[i][s] = 4 * s + (lane >> 4) < K ? r[i][s] : 0.f;
    }
}

// 16 rows x 16 samples: the tile's weights times act (K rows, zero padded to
// a multiple of 16).
template <bool kT>
__device__ __forceinline__ f4_t layer_tile(const float (&r)[32], int K,
                                           const float (*act)[kAct]) {
  const int lane = threadIdx.x & 63;
  f4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    if (16 * g >= K) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = kT ? 16 * g + 4 * (lane >> 4) + e
                       : 16 * g + 4 * e + (lane >> 4);
      acc = mfma4(r[4 * g + e], act[k][lane & 15], acc);
    }
  }
  return acc;
}

// acc += rows of tile t of D times (rows of tile u of E)^T over the samples.
__device__ __forceinline__ f4_t grad_tile(const float (*D)[kAct],
                                          const float (*E)[kAct], int t,
                                          int u, f4_t acc) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k0 = 0; k0 < 16; k0 += 4) {
    const int k = k0 + (lane >> 4);
    acc = mfma4(D[16 * t + (lane & 15)][k], E[16 * u + (lane & 15)][k], acc);
  }
  return acc;
}

// Y (when given) = the network's output; with kGrad also this workgroup's
// share of the gradient (part[blockIdx.x * share_size(np) ..], laid out as the
// parameters, then its share of the loss).  Workgroups take the 16-sample
// tiles blockIdx.x, blockIdx.x + gridDim.x, ...
template <bool kGrad>
__global__ __launch_bounds__(256) void mlp_pass(
    const float* __restrict__ P, Offsets o, int64_t np, int nin, int w,
    const float* __restrict__ X, const float* __restrict__ T, int64_t nb,
    float* __restrict__ Y, float* __restrict__ part) {
  // zero rows behind the inputs pad them to whole tiles
  __shared__ float A0[kMaxIn][kAct], Z1[kMaxW][kAct], A1[kMaxW][kAct],
      Z2[kMaxW][kAct], A2[kMaxW][kAct];
  __shared__ float ys[16][17], dy[16];
  __shared__ float B1[kMaxW], B2[kMaxW], W3[kMaxW], B3;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wt = w / 16, it = (nin + 15) / 16;  // feature tiles
  // gradients of W2 and W1: tile (t, u) for t = wave, wave + 4
  f4_t g2[2][8], g1[2][8];
  float gw3 = 0.f, gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, gl = 0.f;
  if constexpr (kGrad) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) g2[i][u][e] = g1[i][u][e] = 0.f;
  }
  // the parameters, all in flight at once
  if (tid < w) {
    B1[tid] = P[o.b1 + tid];
    B2[tid] = P[o.b2 + tid];
    W3[tid] = P[o.W3 + tid];
  }
  if (tid == 0) B3 = P[o.b3];
  float w1[2][32], w2[2][32], w2t[2][32];
  load_layer(P + o.W1, w, nin, wave, w1);
  load_layer(P + o.W2, w, w, wave, w2);
  if constexpr (kGrad) load_layer_t(P + o.W2, w, wave, w2t);
  clear_behind(nin, w1);
  const float inv = 1.0f / (float)nb;
  for (int64_t n0 = (int64_t)blockIdx.x * 16; n0 < nb;
       n0 += (int64_t)gridDim.x * 16) {
    __syncthreads();
    {
      // sample n, features f0, f0 + 16, ..: read in range, then select
      const int n = tid >> 4, f0 = tid & 15;
      const float* x = X + min(n0 + n, nb - 1) * nin;
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = x[min(f0 + 16 * u, nin - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int f = f0 + 16 * u;
        const float a =
            u < 4 ? 0.125f * log10f(fmaxf(v[u], 1e-16f)) : v[u];
        if (u < it) A0[f][n] = (f < nin && n0 + n < nb) ? a : 0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = wave + 4 * i;
      if (t >= wt) break;
      const f4_t acc = layer_tile<false>(w1[i], 16 * it, A0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = 16 * t + 4 * (lane >> 4) + e;
        const float z = acc[e] + B1[m];
        Z1[m][lane & 15] = z;
        A1[m][lane & 15] = gelu_f(z);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = wave + 4 * i;
      if (t >= wt) break;
      const f4_t acc = layer_tile<false>(w2[i], w, A1);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = 16 * t + 4 * (lane >> 4) + e;
        const float z = acc[e] + B2[m];
        Z2[m][lane & 15] = z;
        A2[m][lane & 15] = gelu_f(z);
      }
    }
    __syncthreads();
    {
      const int n = tid & 15, q = tid >> 4;
      float y = 0.f;
      for (int m = q; m < w; m += 16) y += W3[m] * A2[m][n];
      ys[q][n] = y;
    }
    __syncthreads();
    if (tid < 16) {
      float y = B3;
#pragma unroll
      for (int q = 0; q < 16; ++q) y += ys[q][tid];
      const bool on = n0 + tid < nb;
      if (Y && on) Y[n0 + tid] = y;
      if constexpr (kGrad) {
        const float r = on ? y - T[n0 + tid] : 0.f;
        const float g = 2.0f * r * inv;
        dy[tid] = g;
        gl += r * r;
        gb3 += g;
      }
    }
    if constexpr (kGrad) {
      __syncthreads();
      // dZ2 over Z2
      for (int idx = tid; idx < 16 * w; idx += 256) {
        const int n = idx & 15, m = idx >> 4;
        Z2[m][n] = W3[m] * dy[n] * gelu_d(Z2[m][n]);
      }
      if (tid < w) {
#pragma unroll
        for (int n = 0; n < 16; ++n) gw3 += dy[n] * A2[tid][n];
      }
      __syncthreads();
      // dZ1 over Z1
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = wave + 4 * i;
        if (t >= wt) break;
        const f4_t acc = layer_tile<true>(w2t[i], w, Z2);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = 16 * t + 4 * (lane >> 4) + e;
          Z1[m][lane & 15] = acc[e] * gelu_d(Z1[m][lane & 15]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = wave + 4 * i;
        if (t >= wt) break;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (u < wt) g2[i][u] = grad_tile(Z2, A1, t, u, g2[i][u]);
          if (u < it) g1[i][u] = grad_tile(Z1, A0, t, u, g1[i][u]);
        }
      }
      if (tid < w) {
#pragma unroll
        for (int n = 0; n < 16; ++n) {
          gb1 += Z1[tid][n];
          gb2 += Z2[tid][n];
        }
      }
    }
  }
  if constexpr (kGrad) {
    float* G = part + (int64_t)blockIdx.x * share_size(np);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = wave + 4 * i;
      if (t >= wt) break;
      // four rows of a column per store (w and the blocks' offsets are
      // multiples of 16)
      const int m = 16 * t + 4 * (lane >> 4);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int c = 16 * u + (lane & 15);
        if (u < wt) *(f4_t*)(G + o.W2 + m + c * w) = g2[i][u];
        if (c < nin) *(f4_t*)(G + o.W1 + m + c * w) = g1[i][u];
      }
    }
    if (tid < w) {
      G[o.W3 + tid] = gw3;
      G[o.b1 + tid] = gb1;
      G[o.b2 + tid] = gb2;
    }
    if (tid < 16) {
      // the sixteen samples' shares, in one wave
#pragma unroll
      for (int sh = 8; sh > 0; sh >>= 1) {
        gb3 += __shfl_xor(gb3, sh, 16);
        gl += __shfl_xor(gl, sh, 16);
      }
      if (tid == 0) {
        G[o.b3] = gb3;
        G[np] = gl * inv;
      }
    }
  }
}

// Adds the workgroups' shares of the gradient (in order) into g; with kAdam
// takes the step instead.  The last entry is the loss.
template <bool kAdam>
__global__ __launch_bounds__(256) void mlp_reduce(
    const float* __restrict__ part, int parts, int64_t np,
    float* __restrict__ g, float* __restrict__ loss, float* __restrict__ p,
    float* __restrict__ m1, float* __restrict__ m2, float lr, float b1,
    float b2, float eps, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i > np) return;
  float s = 0.f;
#pragma unroll 8
  for (int q = 0; q < parts; ++q) s += part[q * share_size(np) + i];
  if (i == np) {
    loss[0] = s;
    return;
  }
  if constexpr (kAdam) {
    const float a = b1 * m1[i] + (1.f - b1) * s;
    const float v = b2 * m2[i] + (1.f - b2) * s * s;
    m1[i] = a;
    m2[i] = v;
    p[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
  } else {
    g[i] = s;
  }
}

// Forward and backward of one batch into the workgroups' shares.
int32_t pass_grad(qtn_mlp* m, int64_t nb, const float* X, const float* T,
                  float** part, int* parts) {
  qtn_ctx* ctx = m->ctx;
  const int groups = (int)std::min<int64_t>((nb + 15) / 16, kMaxGroups);
  void* p;
  QTN_TRY(ctx->buffer(kSlotPart, (size_t)groups * share_size(m->np) * sizeof(float),
                      &p));
  hipLaunchKernelGGL(mlp_pass<true>, dim3(groups), dim3(256), 0, ctx->stream,
                     (const float*)m->params, offsets(m->nin, m->width),
                     m->np, m->nin, m->width, X, T, nb, (float*)nullptr,
                     (float*)p);
  QTN_CHECK_HIP(hipGetLastError());
  *part = (float*)p;
  *parts = groups;
  return QTN_OK;
}

struct Acts {
  float *A0, *Z1, *A1, *Z2, *A2, *Y;
};

// Forward pass on device inputs X (nin x nb); keep: activations for the
// backward pass (layer by layer).
int32_t forward(qtn_mlp* m, int64_t nb, const float* X, Acts& a, bool keep) {
  qtn_ctx* ctx = m->ctx;
  hipStream_t s = ctx->stream;
  const int w = m->width, nin = m->nin;
  void* p;
  QTN_TRY(ctx->buffer(kSlotY, (size_t)nb * sizeof(float), &p));
  a.Y = (float*)p;
  const Offsets o = offsets(nin, w);
  const float* P = m->params;
  if (!keep && one_pass(nin, w)) {
    // Two workgroups per CU walk the samples with the weights they loaded.
    // One per 16 samples against 512, us at 262144 samples: 335 / 237
    // (72-128-128-1), 146 / 65 (10-16-16-1; layer by layer 84); even up to
    // 8192 samples.
    const int groups = (int)std::min<int64_t>((nb + 15) / 16, 512);
    hipLaunchKernelGGL(mlp_pass<false>, dim3(groups), dim3(256), 0, s, P, o,
                       m->np, nin, w, X, (const float*)nullptr, nb, a.Y,
                       (float*)nullptr);
    QTN_CHECK_HIP(hipGetLastError());
    return QTN_OK;
  }
  QTN_TRY(ctx->buffer(kSlotA0, (size_t)nin * nb * sizeof(float), &p));
  a.A0 = (float*)p;
  QTN_TRY(ctx->buffer(kSlotZ1, (size_t)w * nb * sizeof(float), &p));
  a.Z1 = (float*)p;
  QTN_TRY(ctx->buffer(kSlotA1, (size_t)w * nb * sizeof(float), &p));
  a.A1 = (float*)p;
  QTN_TRY(ctx->buffer(kSlotZ2, (size_t)w * nb * sizeof(float), &p));
  a.Z2 = (float*)p;
  QTN_TRY(ctx->buffer(kSlotA2, (size_t)w * nb * sizeof(float), &p));
  a.A2 = (float*)p;
  hipLaunchKernelGGL(prep_input, dim3(grid_for((int64_t)nin * nb)),
                     dim3(256), 0, s, X, nin, nb, a.A0);
  QTN_CHECK_HIP(hipGetLastError());
  QTN_TRY((launch_sgemm<false, false>(s, w, nb, nin, P + o.W1, w, a.A0, nin,
                                      a.Z1, w, P + o.b1, 0)));
  hipLaunchKernelGGL(gelu_fwd, dim3(grid_for((int64_t)w * nb)), dim3(256), 0,
                     s, a.Z1, a.A1, (int64_t)w * nb);
  QTN_TRY((launch_sgemm<false, false>(s, w, nb, w, P + o.W2, w, a.A1, w,
                                      a.Z2, w, P + o.b2, 0)));
  hipLaunchKernelGGL(gelu_fwd, dim3(grid_for((int64_t)w * nb)), dim3(256), 0,
                     s, a.Z2, a.A2, (int64_t)w * nb);
  QTN_TRY((launch_sgemm<false, false>(s, 1, nb, w, P + o.W3, 1, a.A2, w, a.Y,
                                      1, P + o.b3, 0)));
  QTN_CHECK_HIP(hipGetLastError());
  return QTN_OK;
}

// Loss and gradient into m->grads for device inputs X and targets T.
int32_t loss_grad(qtn_mlp* m, int64_t nb, const float* X, const float* T,
                  float* loss_dev) {
  qtn_ctx* ctx = m->ctx;
  hipStream_t s = ctx->stream;
  const int w = m->width, nin = m->nin;
  if (one_pass(nin, w)) {
    float* part;
    int parts;
    QTN_TRY(pass_grad(m, nb, X, T, &part, &parts));
    hipLaunchKernelGGL(mlp_reduce<false>,
                       dim3((unsigned)((m->np + 256) / 256)), dim3(256), 0, s,
                       (const float*)part, parts, m->np, m->grads, loss_dev,
                       (float*)nullptr, (float*)nullptr, (float*)nullptr, 0.f,
                       0.f, 0.f, 0.f, 0.f, 0.f);
    QTN_CHECK_HIP(hipGetLastError());
    return QTN_OK;
  }
  Acts a;
  QTN_TRY(forward(m, nb, X, a, true));
  const Offsets o = offsets(nin, w);
  const float* P = m->params;
  float* G = m->grads;
  void *pd1, *pd2, *pdy;
  QTN_TRY(ctx->buffer(kSlotD1, (size_t)w * nb * sizeof(float), &pd1));
  QTN_TRY(ctx->buffer(kSlotD2, (size_t)w * nb * sizeof(float), &pd2));
  QTN_TRY(ctx->buffer(kSlotT, (size_t)nb * sizeof(float) * 2, &pdy));
  float* dZ1 = (float*)pd1;
  float* dZ2 = (float*)pd2;
  float* dY = (float*)pdy + nb;
  hipLaunchKernelGGL(mse_grad, dim3(1), dim3(256), 0, s, a.Y, T, nb, dY,
                     loss_dev);
  // dW3 = dY A2^T (1 x w), db3 = sum dY
  QTN_TRY((launch_sgemm<false, true>(s, 1, w, nb, dY, 1, a.A2, w, G + o.W3,
                                     1, nullptr, 0)));
  hipLaunchKernelGGL(row_sum, dim3(1), dim3(256), 0, s, dY, 1, nb, G + o.b3);
  // dZ2 = W3^T dY * gelu'(Z2)
  QTN_TRY((launch_sgemm<true, false>(s, w, nb, 1, P + o.W3, 1, dY, 1, dZ2, w,
                                     nullptr, 0)));
  hipLaunchKernelGGL(gelu_bwd, dim3(grid_for((int64_t)w * nb)), dim3(256), 0,
                     s, a.Z2, dZ2, (int64_t)w * nb);
  // dW2 = dZ2 A1^T, db2
  QTN_TRY((launch_sgemm<false, true>(s, w, w, nb, dZ2, w, a.A1, w, G + o.W2,
                                     w, nullptr, 0)));
  hipLaunchKernelGGL(row_sum, dim3((w + 3) / 4), dim3(256), 0, s, dZ2, w, nb,
                     G + o.b2);
  // dZ1 = W2^T dZ2 * gelu'(Z1)
  QTN_TRY((launch_sgemm<true, false>(s, w, nb, w, P + o.W2, w, dZ2, w, dZ1,
                                     w, nullptr, 0)));
  hipLaunchKernelGGL(gelu_bwd, dim3(grid_for((int64_t)w * nb)), dim3(256), 0,
                     s, a.Z1, dZ1, (int64_t)w * nb);
  // dW1 = dZ1 A0^T, db1
  QTN_TRY((launch_sgemm<false, true>(s, w, nin, nb, dZ1, w, a.A0, nin,
                                     G + o.W1, w, nullptr, 0)));
  hipLaunchKernelGGL(row_sum, dim3((w + 3) / 4), dim3(256), 0, s, dZ1, w, nb,
                     G + o.b1);
  QTN_CHECK_HIP(hipGetLastError());
  return QTN_OK;
}

int32_t upload(qtn_ctx* ctx, int slot, const float* host, size_t n,
               float** dev) {
  void* p;
  QTN_TRY(ctx->buffer(slot, std::max<size_t>(n, 1) * sizeof(float), &p));
  QTN_CHECK_HIP(hipMemcpyAsync(p, host, n * sizeof(float),
                               hipMemcpyHostToDevice, ctx->stream));
  *dev = (float*)p;
  return QTN_OK;
}

}  // namespace

// Prediction for device features (used by the learned two-site update):
// Y (nb floats, device) = mlp(X) for X (nin x nb, device).
int32_t mlp_predict_device(qtn_mlp* m, int64_t nb, const float* X,
                           float** Y) {
  Acts a;
  QTN_TRY(forward(m, nb, X, a, false));
  *Y = a.Y;
  return QTN_OK;
}

int mlp_nin(const qtn_mlp* m) { return m->nin; }
qtn_ctx* mlp_ctx(const qtn_mlp* m) { return m->ctx; }

}  // namespace qtn

using namespace qtn;

extern "C" {

int32_t qtn_mlp_create(qtn_ctx* ctx, int32_t nin, int32_t width,
                       const float* params, qtn_mlp** out) try {
  clear_error();
  QTN_ARG(ctx && params && out, "qtn_mlp_create: NULL argument");
  QTN_ARG(nin >= 1 && nin <= 4096 && width >= 1 && width <= 4096,
          "qtn_mlp_create: bad sizes");
  QTN_CHECK_HIP(hipSetDevice(ctx->device));
  qtn_mlp* m = new qtn_mlp();
  m->ctx = ctx;
  m->nin = nin;
  m->width = width;
  m->np = (int64_t)width * nin + width + (int64_t)width * width + width +
          width + 1;
  const size_t bytes = (size_t)m->np * 4 * sizeof(float);
  hipError_t e = hipMalloc(&m->arena, bytes);
  if (e != hipSuccess) {
    delete m;
    set_error("qtn_mlp_create: hipMalloc failed");
    return QTN_ERR_OOM;
  }
  m->params = (float*)m->arena;
  m->grads = m->params + m->np;
  m->m1 = m->grads + m->np;
  m->m2 = m->m1 + m->np;
  QTN_CHECK_HIP(hipMemsetAsync(m->arena, 0, bytes, ctx->stream));
  QTN_CHECK_HIP(hipMemcpyAsync(m->params, params, m->np * sizeof(float),
                               hipMemcpyHostToDevice, ctx->stream));
  QTN_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  *out = m;
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

int32_t qtn_mlp_destroy(qtn_mlp* m) try {
  clear_error();
  if (!m) return QTN_OK;
  QTN_CHECK_HIP(hipSetDevice(m->ctx->device));
  QTN_CHECK_HIP(hipStreamSynchronize(m->ctx->stream));
  if (m->arena) QTN_CHECK_HIP(hipFree(m->arena));
  delete m;
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

int32_t qtn_mlp_get_params(const qtn_mlp* m, float* params) try {
  clear_error();
  QTN_ARG(m && params, "qtn_mlp_get_params: NULL argument");
  QTN_CHECK_HIP(hipSetDevice(m->ctx->device));
  QTN_CHECK_HIP(hipMemcpyAsync(params, m->params, m->np * sizeof(float),
                               hipMemcpyDeviceToHost, m->ctx->stream));
  QTN_CHECK_HIP(hipStreamSynchronize(m->ctx->stream));
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

int32_t qtn_mlp_forward(qtn_mlp* m, int64_t nb, const float* X, float* Y) try {
  clear_error();
  QTN_ARG(m && X && Y, "qtn_mlp_forward: NULL argument");
  QTN_ARG(nb >= 1, "qtn_mlp_forward: empty batch");
  qtn_ctx* ctx = m->ctx;
  QTN_CHECK_HIP(hipSetDevice(ctx->device));
  float* dX;
  QTN_TRY(upload(ctx, kSlotIn, X, (size_t)m->nin * nb, &dX));
  float* dY;
  QTN_TRY(mlp_predict_device(m, nb, dX, &dY));
  QTN_CHECK_HIP(hipMemcpyAsync(Y, dY, nb * sizeof(float),
                               hipMemcpyDeviceToHost, ctx->stream));
  QTN_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

int32_t qtn_mlp_loss_grad(qtn_mlp* m, int64_t nb, const float* X,
                          const float* T, float* loss, float* grad) try {
  clear_error();
  QTN_ARG(m && X && T && loss && grad, "qtn_mlp_loss_grad: NULL argument");
  QTN_ARG(nb >= 1, "qtn_mlp_loss_grad: empty batch");
  qtn_ctx* ctx = m->ctx;
  QTN_CHECK_HIP(hipSetDevice(ctx->device));
  float *dX, *dT;
  QTN_TRY(upload(ctx, kSlotIn, X, (size_t)m->nin * nb, &dX));
  void* pt;
  QTN_TRY(ctx->buffer(kSlotT, (size_t)nb * sizeof(float) * 2, &pt));
  dT = (float*)pt;
  QTN_CHECK_HIP(hipMemcpyAsync(dT, T, nb * sizeof(float),
                               hipMemcpyHostToDevice, ctx->stream));
  void* pl;
  QTN_TRY(ctx->buffer(kSlotLoss, sizeof(float), &pl));
  QTN_TRY(loss_grad(m, nb, dX, dT, (float*)pl));
  QTN_CHECK_HIP(hipMemcpyAsync(loss, pl, sizeof(float),
                               hipMemcpyDeviceToHost, ctx->stream));
  QTN_CHECK_HIP(hipMemcpyAsync(grad, m->grads, m->np * sizeof(float),
                               hipMemcpyDeviceToHost, ctx->stream));
  QTN_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

int32_t qtn_mlp_train(qtn_mlp* m, int64_t nb, const float* X, const float* T,
                      int32_t steps, int64_t minibatch, float lr,
                      float* loss_hist) try {
  clear_error();
  QTN_ARG(m && X && T, "qtn_mlp_train: NULL argument");
  QTN_ARG(nb >= 1 && steps >= 0, "qtn_mlp_train: bad sizes");
  qtn_ctx* ctx = m->ctx;
  hipStream_t s = ctx->stream;
  QTN_CHECK_HIP(hipSetDevice(ctx->device));
  const int64_t mb = (minibatch > 0 && minibatch < nb) ? minibatch : nb;
  // the whole training set stays on the device; step t trains on the
  // contiguous slice starting at (t * mb) mod nb (the caller shuffles)
  float *dX, *dT;
  QTN_TRY(upload(ctx, kSlotIn, X, (size_t)m->nin * nb, &dX));
  void* pt;
  QTN_TRY(ctx->buffer(kSlotT + 10, (size_t)nb * sizeof(float), &pt));
  dT = (float*)pt;
  QTN_CHECK_HIP(hipMemcpyAsync(dT, T, nb * sizeof(float),
                               hipMemcpyHostToDevice, s));
  void* pl;
  QTN_TRY(ctx->buffer(kSlotLoss, (size_t)std::max(1, steps) * sizeof(float),
                      &pl));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int t = 0; t < steps; ++t) {
    const int64_t start = ((int64_t)t * mb) % nb;
    const int64_t cnt = std::min(mb, nb - start);
    const float c1 = 1.f - powf(b1, (float)(m->step + 1));
    const float c2 = 1.f - powf(b2, (float)(m->step + 1));
    if (one_pass(m->nin, m->width)) {
      float* part;
      int parts;
      QTN_TRY(pass_grad(m, cnt, dX + start * m->nin, dT + start, &part,
                        &parts));
      hipLaunchKernelGGL(mlp_reduce<true>,
                         dim3((unsigned)((m->np + 256) / 256)), dim3(256), 0,
                         s, (const float*)part, parts, m->np, (float*)nullptr,
                         (float*)pl + t, m->params, m->m1, m->m2, lr, b1, b2,
                         eps, c1, c2);
      QTN_CHECK_HIP(hipGetLastError());
      m->step += 1;
      continue;
    }
    QTN_TRY(loss_grad(m, cnt, dX + start * m->nin, dT + start,
                      (float*)pl + t));
    hipLaunchKernelGGL(adam_step, dim3(grid_for(m->np)), dim3(256), 0, s,
                       m->params, (const float*)m->grads, m->m1, m->m2, m->np,
                       lr, b1, b2, eps, c1, c2);
    QTN_CHECK_HIP(hipGetLastError());
    m->step += 1;
  }
  if (loss_hist && steps > 0)
    QTN_CHECK_HIP(hipMemcpyAsync(loss_hist, pl, steps * sizeof(float),
                                 hipMemcpyDeviceToHost, s));
  QTN_CHECK_HIP(hipStreamSynchronize(s));
  return QTN_OK;
} catch (...) {
  return qtn::abi_exception();
}

}  // extern "C"
