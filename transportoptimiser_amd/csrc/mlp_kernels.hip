// Surrogate MLP kernels (FP32): an ensemble of E networks
// n_in -> H -> H -> n_out with tanh hidden layers, trained by Adam on the
// mean squared error.  The reference fits its GA surrogate with kNN local
// regression on a grid (SimulateGPU.cu:2934-3155, 5533-5968); this network
// replaces that fit and full Monte Carlo stays as the fallback.
//
// Parameter layout of one member: W1[n_in][H], b1[H], W2[H][H], b2[H],
// W3[H][n_out], b3[n_out] (row-major, input index first).
#include <hip/hip_runtime.h>

#include "mlp_kernels.h"

namespace roadmc {

constexpr int kMlpH = 64;
constexpr int kMlpThreads = 512;  // 8 waves

__host__ __device__ inline int mlp_n_params(int n_in, int n_out) {
  return n_in * kMlpH + kMlpH + kMlpH * kMlpH + kMlpH + kMlpH * n_out + n_out;
}

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Row strides of the LDS arrays.  A lane reads element (l % 16, l / 16) of a
// 16 x 4 operand: at stride 68 (4 mod 64 banks) the 16 rows and 4 consecutive
// columns, at stride 80 (16 mod 64) the 4 rows and 16 consecutive columns, lie
// in 64 different banks.
constexpr int kSA = 68, kSB = 80;

// One 16 x 16 output tile of A . B over K terms on v_mfma_f32_16x16x4_f32,
// operand (row, k) at A[row * ar + k * ak], (k, column) at B[k * bk + col *
// bc].  Lane l's item r is the tile's (4 (l / 16) + r, l % 16).
template <int K>
__device__ __forceinline__ floatx4 mlp_tile(const float* A, int ar, int ak, const float* B, int bk,
                                            int bc) {
  const int l = threadIdx.x & 63, i = l & 15, k0 = l >> 4;
  const float* a = A + i * ar + k0 * ak;
  const float* b = B + k0 * bk + i * bc;
  floatx4 acc = {};
#pragma unroll
  for (int k = 0; k < K; k += 4)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k * ak], b[k * bk], acc, 0, 0, 0);
  return acc;
}

// The forward pass of 32 samples through member e, shared by the gradient and
// the prediction: weights and activations in LDS, the 64 x 64 layer on the
// FP32 matrix cores (one 16 x 16 tile a wave), the small layers on the VALU.
struct MlpLds {
  float *W1, *b1, *W2, *b2, *W3, *b3;  // W2 at stride kSB
  float *x, *h1, *h2;                  // [S][n_in], [S][kSA], [S][kSA]
  float* y;                            // [S][n_out]
};

__host__ __device__ inline int mlp_fwd_floats(int n_in, int n_out) {
  const int S = kMlpChunk, H = kMlpH;
  return n_in * H + H + H * kSB + H + H * n_out + n_out + S * n_in + 2 * S * kSA + S * n_out;
}

__device__ __forceinline__ MlpLds mlp_lds(float* sm, int NI, int NO) {
  constexpr int S = kMlpChunk, H = kMlpH;
  MlpLds m;
  m.h1 = sm;
  m.h2 = m.h1 + S * kSA;
  m.W2 = m.h2 + S * kSA;
  m.W1 = m.W2 + H * kSB;
  m.b1 = m.W1 + NI * H;
  m.b2 = m.b1 + H;
  m.W3 = m.b2 + H;
  m.b3 = m.W3 + H * NO;
  m.x = m.b3 + NO;
  m.y = m.x + S * NI;
  return m;
}

__device__ __forceinline__ void mlp_forward(const MlpLds& m, const float* __restrict__ w, int NI,
                                            int NO, const float* __restrict__ X, int n, int s0) {
  constexpr int S = kMlpChunk, H = kMlpH;
  const int tid = threadIdx.x;
  const float* w2 = w + NI * H + H;
  const float* w3 = w2 + H * H + H;
  for (int i = tid; i < NI * H + H; i += kMlpThreads) m.W1[i] = w[i];  // W1, b1
  for (int i = tid; i < H * H; i += kMlpThreads) m.W2[(i >> 6) * kSB + (i & 63)] = w2[i];
  for (int i = tid; i < H; i += kMlpThreads) m.b2[i] = w2[H * H + i];
  for (int i = tid; i < H * NO + NO; i += kMlpThreads) m.W3[i] = w3[i];  // W3, b3
  for (int i = tid; i < S * NI; i += kMlpThreads)
    m.x[i] = (size_t)s0 * NI + i < (size_t)n * NI ? X[(size_t)s0 * NI + i] : 0.0f;
  __syncthreads();
  // h1 = tanh(x W1 + b1)
#pragma unroll
  for (int i = tid; i < S * H; i += kMlpThreads) {
    const int s = i >> 6, j = i & 63;
    float v = m.b1[j];
    for (int k = 0; k < NI; ++k) v += m.x[s * NI + k] * m.W1[k * H + j];
    m.h1[s * kSA + j] = tanhf(v);
  }
  __syncthreads();
  // h2 = tanh(h1 W2 + b2)
  {
    const int l = tid & 63, wave = tid >> 6, r0 = (wave & 1) * 16, c0 = (wave >> 1) * 16;
    const floatx4 a = mlp_tile<H>(m.h1 + r0 * kSA, kSA, 1, m.W2 + c0, kSB, 1);
    const int j = c0 + (l & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      m.h2[(r0 + 4 * (l >> 4) + r) * kSA + j] = tanhf(a[r] + m.b2[j]);
  }
  __syncthreads();
  // y = h2 W3 + b3, eight lanes an output.
  for (int i = tid >> 3; i < S * NO; i += kMlpThreads / 8) {
    const int s = i / NO, k = i - s * NO, q = tid & 7;
    float v = 0.0f;
#pragma unroll
    for (int j = 0; j < H; j += 8) v += m.h2[s * kSA + j + q] * m.W3[(j + q) * NO + k];
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    if (q == 0) m.y[i] = v + m.b3[k];
  }
  __syncthreads();
}

// One block: member e = blockIdx.y, samples [32 chunk, 32 chunk + 32).  The
// three 64-wide products (h1 W2, d2 W2^T, h1^T d2) run on the FP32 matrix
// cores from LDS; the work is a chain of short phases, so small chunks (256
// blocks for 2,048 samples of 4 members) shorten it.  One thread per output
// with scalar LDS loops over 64-sample chunks took 159 us a launch at that
// size; this one 15 us (a pass of 400 steps 68.9 -> 8.4 ms).
__global__ __launch_bounds__(kMlpThreads) void mlp_grad_kernel(MlpArgs a,
                                                               const float* __restrict__ X,
                                                               const float* __restrict__ Y, int n,
                                                               float* __restrict__ partial,
                                                               float* __restrict__ loss_part) {
  constexpr int H = kMlpH, S = kMlpChunk;
  const int NI = a.n_in, NO = a.n_out, NP = mlp_n_params(NI, NO);
  const int e = blockIdx.y, chunk = blockIdx.x, s0 = chunk * S;
  extern __shared__ float sm[];
  __shared__ float red[kMlpThreads / 64];
  const MlpLds m = mlp_lds(sm, NI, NO);
  float* d1 = m.y + S * NO;    // [S][kSA]
  float* d2 = d1 + S * kSA;    // [S][kSA]
  float* W2t = d2 + S * kSA;   // W2 at stride kSA, for d2 W2^T
  const int tid = threadIdx.x, l = tid & 63, wave = tid >> 6;
  const float* w = a.params + (size_t)e * NP;
  for (int i = tid; i < H * H; i += kMlpThreads)
    W2t[(i >> 6) * kSA + (i & 63)] = w[NI * H + H + i];
  mlp_forward(m, w, NI, NO, X, n, s0);
  // MSE over n samples and NO outputs; y becomes its gradient.
  float lsum = 0.0f;
  const float scale = 2.0f / ((float)n * (float)NO);
  for (int i = tid; i < S * NO; i += kMlpThreads) {
    float g = 0.0f;
    if (s0 + i / NO < n) {
      const float r = m.y[i] - Y[(size_t)s0 * NO + i];
      lsum += r * r;
      g = scale * r;
    }
    m.y[i] = g;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
  if (l == 0) red[wave] = lsum;
  __syncthreads();
  // d2 = (dy W3^T) o (1 - h2^2)
#pragma unroll
  for (int i = tid; i < S * H; i += kMlpThreads) {
    const int s = i >> 6, j = i & 63;
    float v = 0.0f;
    for (int k = 0; k < NO; ++k) v += m.y[s * NO + k] * m.W3[j * NO + k];
    const float h = m.h2[s * kSA + j];
    d2[s * kSA + j] = v * (1.0f - h * h);
  }
  __syncthreads();
  // d1 = (d2 W2^T) o (1 - h1^2)
  {
    const int r0 = (wave & 1) * 16, c0 = (wave >> 1) * 16;
    const floatx4 t = mlp_tile<H>(d2 + r0 * kSA, kSA, 1, W2t + c0 * kSA, 1, kSA);
    const int j = c0 + (l & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int at = (r0 + 4 * (l >> 4) + r) * kSA + j;
      const float h = m.h1[at];
      d1[at] = t[r] * (1.0f - h * h);
    }
  }
  // Weight gradients summed over the block's samples (fixed order).
  float* g = partial + ((size_t)e * gridDim.x + chunk) * NP;
  float* gW2 = g + NI * H + H;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int i0 = (wave & 3) * 16, j0 = ((wave >> 2) * 2 + t) * 16;
    const floatx4 v = mlp_tile<S>(m.h1 + i0, 1, kSA, d2 + j0, kSA, 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) gW2[(i0 + 4 * (l >> 4) + r) * H + j0 + (l & 15)] = v[r];
  }
  __syncthreads();
  // The others: W1, b1, then b2, W3, b3.
  const int n1 = NI * H + H, n3 = H + H * NO + NO;
  for (int p = tid; p < n1 + n3; p += kMlpThreads) {
    const float *u = nullptr, *d;  // sum over the samples of u (or 1) times d
    int us = 0, ds = kSA;
    if (p < n1) {
      const int i = p >> 6;
      if (i < NI) {
        u = m.x + i;
        us = NI;
      }
      d = d1 + (p & 63);
    } else if (p < n1 + H) {
      d = d2 + (p - n1);
    } else {
      const int q = p - n1 - H, i = q / NO;
      if (i < H) {
        u = m.h2 + i;
        us = kSA;
      }
      d = m.y + (q - i * NO);
      ds = NO;
    }
    float v = 0.0f;
#pragma unroll 8
    for (int s = 0; s < S; ++s) v += u ? u[s * us] * d[s * ds] : d[s * ds];
    g[p < n1 ? p : p + H * H] = v;
  }
  if (tid == 0) {
    float t = 0.0f;
    for (int i = 0; i < kMlpThreads / 64; ++i) t += red[i];
    loss_part[(size_t)e * gridDim.x + chunk] = t / ((float)n * (float)NO);
  }
}

// Sums the block partials (fixed order: four interleaved sums, then those) and,
// when lr > 0, applies one Adam step; grad_out (optional) receives the summed
// gradient.  64 parameters a block, four threads a parameter, sixteen loads in
// flight.
__global__ __launch_bounds__(256) void mlp_adam_kernel(MlpArgs a,
                                                       const float* __restrict__ partial,
                                                       int nchunk, float* __restrict__ grad_out,
                                                       float lr, float bc1, float bc2) {
  __shared__ float part[4][64];
  const int NP = mlp_n_params(a.n_in, a.n_out);
  const int e = blockIdx.y, x = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + x;
  float g = 0.0f;
  if (p < NP) {
    const float* src = partial + (size_t)e * nchunk * NP + p;
#pragma unroll 16
    for (int c = q; c < nchunk; c += 4) g += src[(size_t)c * NP];
  }
  part[q][x] = g;
  __syncthreads();
  if (q || p >= NP) return;
  g = (part[0][x] + part[1][x]) + (part[2][x] + part[3][x]);
  const size_t i = (size_t)e * NP + p;
  if (grad_out) grad_out[i] = g;
  if (lr > 0.0f) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float m = b1 * a.m[i] + (1.0f - b1) * g;
    const float v = b2 * a.v[i] + (1.0f - b2) * g * g;
    a.m[i] = m;
    a.v[i] = v;
    a.params[i] -= lr * (m / bc1) / (sqrtf(v / bc2) + eps);
  }
}

__global__ void mlp_loss_kernel(const float* __restrict__ loss_part, int nchunk, int E,
                                float* __restrict__ loss) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  float l = 0.0f;
  for (int c = 0; c < nchunk; ++c) l += loss_part[(size_t)e * nchunk + c];
  loss[e] = l;
}

// out[e][s][k], 32 samples of a member per block.
__global__ __launch_bounds__(kMlpThreads) void mlp_predict_kernel(MlpArgs a,
                                                                  const float* __restrict__ X,
                                                                  int n, float* __restrict__ out) {
  const int NI = a.n_in, NO = a.n_out, e = blockIdx.y, s0 = blockIdx.x * kMlpChunk;
  extern __shared__ float sm[];
  const MlpLds m = mlp_lds(sm, NI, NO);
  mlp_forward(m, a.params + (size_t)e * mlp_n_params(NI, NO), NI, NO, X, n, s0);
  for (int i = threadIdx.x; i < kMlpChunk * NO; i += kMlpThreads)
    if (s0 + i / NO < n) out[((size_t)e * n + s0) * NO + i] = m.y[i];
}

int mlp_param_count(int n_in, int n_out) { return mlp_n_params(n_in, n_out); }

namespace {

size_t mlp_predict_lds(int n_in, int n_out) { return sizeof(float) * mlp_fwd_floats(n_in, n_out); }

size_t mlp_grad_lds(int n_in, int n_out) {
  return mlp_predict_lds(n_in, n_out) +
         sizeof(float) * (2 * kMlpChunk * kSA + kMlpH * kSA);
}

}  // namespace

hipError_t mlp_set_lds_limit(int n_in, int n_out) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_grad_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)mlp_grad_lds(n_in, n_out));
  return e != hipSuccess ? e
                         : hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_predict_kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)mlp_predict_lds(n_in, n_out));
}

hipError_t launch_mlp_grad(const MlpArgs& a, const float* X, const float* Y, int n, float* partial,
                           float* loss_part, hipStream_t s) {
  hipLaunchKernelGGL(mlp_grad_kernel, dim3(mlp_chunks(n), a.E), dim3(kMlpThreads),
                     mlp_grad_lds(a.n_in, a.n_out), s, a, X, Y, n, partial, loss_part);
  return hipGetLastError();
}

hipError_t launch_mlp_update(const MlpArgs& a, const float* partial, int nchunk, float* grad_out,
                             float lr, float bc1, float bc2, const float* loss_part, float* loss,
                             hipStream_t s) {
  hipLaunchKernelGGL(mlp_adam_kernel, dim3((mlp_n_params(a.n_in, a.n_out) + 63) / 64, a.E),
                     dim3(256), 0, s, a, partial, nchunk, grad_out, lr, bc1, bc2);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !loss) return e;
  hipLaunchKernelGGL(mlp_loss_kernel, dim3(1), dim3(64), 0, s, loss_part, nchunk, a.E, loss);
  return hipGetLastError();
}

hipError_t launch_mlp_predict(const MlpArgs& a, const float* X, int n, float* out, hipStream_t s) {
  hipLaunchKernelGGL(mlp_predict_kernel, dim3(mlp_chunks(n), a.E), dim3(kMlpThreads),
                     mlp_predict_lds(a.n_in, a.n_out), s, a, X, n, out);
  return hipGetLastError();
}

}  // namespace roadmc
