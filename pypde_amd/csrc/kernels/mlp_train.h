// Kernels for training the Newton initial-guess MLP on the GPU (hipRTC-compiled
// once, independent of the PDE).  Matrices are row-major fp32 in memory with
// samples along columns ("feature-major"); products run on the matrix cores as
// BF16 x BF16 -> FP32 (v_mfma_f32_32x32x8bf16_1k).
//
// MFMA 32x32x8 operand layout (64 lanes, l = lane):
//   A (32 x 8):  a[i] = A[l % 32][4 (l / 32) + i]          i = 0..3
//   B (8 x 32):  b[i] = B[4 (l / 32) + i][l % 32]
//   C (32 x 32): c[j] = C[8 (j / 4) + 4 (l / 32) + j % 4][l % 32]   j = 0..15
#pragma once

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ short to_bf16(float x) {
  // round to nearest even (inputs here are finite)
  unsigned int b = __float_as_uint(x);
  b += 0x7FFFu + ((b >> 16) & 1u);
  return (short)(b >> 16);
}

__device__ __forceinline__ float bf16_to_f(short h) {
  return __uint_as_float(((unsigned int)(unsigned short)h) << 16);
}

// Four floats p[0], p[ld], p[2 ld], p[3 ld] as BF16, entries from `left` on
// read as 0 (left <= 0: none is read).  vec: ld = 1 and p is 16-byte aligned.
__device__ __forceinline__ bf16x4 load4(const float* __restrict__ p, long ld, int left, bool vec) {
  float x[4];
  if (vec && left >= 4) {
    const float4 q = *(const float4*)p;
    x[0] = q.x, x[1] = q.y, x[2] = q.z, x[3] = q.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = i < left ? p[i * ld] : 0.0f;
  }
  bf16x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = to_bf16(x[i]);
  return r;
}
__device__ __forceinline__ bf16x4 round4(float4 q) {
  const bf16x4 r = {to_bf16(q.x), to_bf16(q.y), to_bf16(q.z), to_bf16(q.w)};
  return r;
}
// Whether groups of four along a row of X (leading dimension ld) are aligned.
__device__ __forceinline__ bool vector_rows(const float* X, int ld) {
  return (ld & 3) == 0 && ((unsigned long long)X & 15ull) == 0;
}

// C = alpha op(A) op(B) + beta C;  op(A): M x K, op(B): K x N.
// A(m, k) = transA ? A[k * lda + m] : A[m * lda + k];  likewise B.
// A workgroup of 4 waves computes a 64 x 64 tile.  The network's products have
// K = 46..135 and a batch of columns, so what bounds them is the latency of
// one panel after another: K goes in chunks of 128, a thread's sixteen loads
// of four values all in flight, and both operands lie in LDS with k
// contiguous, so that a fragment is one 8-byte read (135 x 4096 x 128: 14.9 ->
// 7.7 us against chunks of 32 and B fragments gathered from four rows).
constexpr int GEMM_KC = 128;
extern "C" __global__ void __launch_bounds__(256)
k_gemm_bf16(const float* __restrict__ A, int lda, int transA, const float* __restrict__ B, int ldb,
            int transB, float* __restrict__ C, int ldc, int M, int N, int K, float alpha,
            float beta) {
  __shared__ __align__(16) short As[64][GEMM_KC + 8];
  __shared__ __align__(16) short Bs[64][GEMM_KC + 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  // op(X)'s panel, row index r0.. (op(A)'s rows, op(B)'s columns), as [row][k]
  auto stage = [&](const float* __restrict__ X, int ld, bool kfast, int r0, int rows, int k0,
                   short (*S)[GEMM_KC + 8]) {
    constexpr int G = GEMM_KC / 4;
    const bool vec = kfast && vector_rows(X, ld);
#pragma unroll
    for (int i = 0; i < 64 * G / 256; i++) {
      const int e = tid + 256 * i;
      // neighbouring threads read neighbouring addresses
      const int r = kfast ? e / G : e % 64, k = 4 * (kfast ? e % G : e / 64);
      const int gr = r0 + r, gk = k0 + k;
      bf16x4 v = {0, 0, 0, 0};
      if (gr < rows && gk < K)
        v = load4(kfast ? X + (long)gr * ld + gk : X + (long)gk * ld + gr, kfast ? 1 : ld, K - gk,
                  vec);
      *(bf16x4*)&S[r][k] = v;
    }
  };
  f32x16 acc;
#pragma unroll
  for (int j = 0; j < 16; j++) acc[j] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += GEMM_KC) {
    if (k0) __syncthreads();
    stage(A, lda, !transA, m0, M, k0, As);
    stage(B, ldb, transB != 0, n0, N, k0, Bs);
    __syncthreads();
    const int kc = K - k0 < GEMM_KC ? (K - k0 + 7) / 8 : GEMM_KC / 8;
#pragma unroll 4
    for (int kk = 0; kk < kc; kk++) {
      const bf16x4 a = *(const bf16x4*)&As[wr + (lane & 31)][kk * 8 + 4 * (lane >> 5)];
      const bf16x4 b = *(const bf16x4*)&Bs[wc + (lane & 31)][kk * 8 + 4 * (lane >> 5)];
      acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < 16; j++) {
    int r = m0 + wr + 8 * (j / 4) + 4 * (lane >> 5) + (j % 4);
    int c = n0 + wc + (lane & 31);
    if (r < M && c < N) {
      float v = alpha * acc[j];
      if (beta != 0.0f) v += beta * C[(long)r * ldc + c];
      C[(long)r * ldc + c] = v;
    }
  }
}

// C = alpha A B^T + beta C for a long K and a small C (weight gradients: K is
// the batch): with 64 x 64 tiles such a product fills two to six workgroups
// that walk the batch serially.  Here a workgroup of 16 waves computes a 16 x
// 16 tile, each wave taking one sixteenth of K straight from memory (k is
// contiguous in both operands) in chunks of 32, and the 16 partial tiles are
// summed in wave order, so results do not depend on timing.  Bound by each
// compute unit's line lookups (a load touches 16 rows); the workgroups start
// at different chunks, so that a power-of-two batch's rows do not meet in one
// L2 channel.  135 x 128 x 4096: 345 -> 16.5 us, x 16384: 2021 -> 59 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int TALL_WAVES = 16;
extern "C" __global__ void __launch_bounds__(64 * TALL_WAVES)
k_gemm_bf16_tall(const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
                 float* __restrict__ C, int ldc, int M, int N, int K, float alpha, float beta) {
  __shared__ float part[TALL_WAVES][16][17];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
  // rows past the edge repeat the last one; their results are not stored
  const int ra = m0 + (lane & 15) < M ? m0 + (lane & 15) : M - 1;
  const int rb = n0 + (lane & 15) < N ? n0 + (lane & 15) : N - 1;
  const float* const pa = A + (long)ra * lda;
  const float* const pb = B + (long)rb * ldb;
  const bool vec = vector_rows(A, lda) && vector_rows(B, ldb);
  // 16x16x16: a[i] = A[l % 16][4 (l / 16) + i], c[j] = C[4 (l / 16) + j][l % 16]
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int chunks = (K + 32 * TALL_WAVES - 1) / (32 * TALL_WAVES);  // per wave
  int c = (int)((blockIdx.x + blockIdx.y * gridDim.x) % chunks);
#pragma unroll 4
  for (int i = 0; i < chunks; i++) {
    const int k0 = 32 * (wave * chunks + c);
    c = c + 1 < chunks ? c + 1 : 0;
    if (vec && k0 + 32 <= K) {
      float4 x[2][2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = k0 + 16 * h + 4 * (lane >> 4);
        x[0][h] = *(const float4*)(pa + k);
        x[1][h] = *(const float4*)(pb + k);
      }
#pragma unroll
      for (int h = 0; h < 2; h++)
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(round4(x[0][h]), round4(x[1][h]), acc, 0,
                                                        0, 0);
    } else {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = k0 + 16 * h + 4 * (lane >> 4);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(load4(pa + k, 1, K - k, false),
                                                        load4(pb + k, 1, K - k, false), acc, 0, 0,
                                                        0);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++) part[wave][4 * (lane >> 4) + j][lane & 15] = acc[j];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    float v = part[0][r][c];
#pragma unroll
    for (int w = 1; w < TALL_WAVES; w++) v += part[w][r][c];
    if (m0 + r < M && n0 + c < N) {
      float* const o = C + (long)(m0 + r) * ldc + n0 + c;
      v = alpha * v;
      if (beta != 0.0f) v += beta * *o;
      *o = v;
    }
  }
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu_grad(float z) {
  float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// Z[r][c] += b[r]; H = act(Z) (act 1: SiLU, 0: identity).  H may alias Z only
// when act == 0.
extern "C" __global__ void k_bias_act(float* __restrict__ Z, const float* __restrict__ b,
                                      float* __restrict__ H, int rows, int cols, int act) {
  long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)rows * cols) return;
  int r = (int)(i / cols);
  float z = Z[i] + b[r];
  Z[i] = z;
  H[i] = act ? silu(z) : z;
}

// dZ = dH * SiLU'(Z)
extern "C" __global__ void k_act_grad(float* __restrict__ dZ, const float* __restrict__ dH,
                                      const float* __restrict__ Z, long n) {
  long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  dZ[i] = dH[i] * silu_grad(Z[i]);
}

// db[r] = sum_c dZ[r][c]  (one workgroup per row)
extern "C" __global__ void __launch_bounds__(256)
k_rowsum(const float* __restrict__ dZ, float* __restrict__ db, int rows, int cols) {
  __shared__ float red[256];
  int r = blockIdx.x;
  float s = 0.0f;
  for (int c = threadIdx.x; c < cols; c += 256) s += dZ[(long)r * cols + c];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) db[r] = red[0];
}

// mean-squared error over rows x cols: dY = 2 (Y - T) / (rows cols), loss
// accumulated (sum of squares / (rows cols)) into *loss.  At most 256
// workgroups stride over the array: their atomics on the one address are what
// bounds a launch with one per 256 entries (135 x 4096: 30.6 -> 8.2 us).
extern "C" __global__ void __launch_bounds__(256)
k_mse(const float* __restrict__ Y, const float* __restrict__ T, float* __restrict__ dY,
      float* __restrict__ loss, int rows, int cols) {
  __shared__ float red[256];
  long n = (long)rows * cols;
  float e = 0.0f;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256l * gridDim.x) {
    float d = Y[i] - T[i];
    dY[i] = 2.0f * d / (float)n;
    e += d * d / (float)n;
  }
  red[threadIdx.x] = e;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Adam step (Kingma & Ba) on fp32 master weights.
extern "C" __global__ void k_adam(float* __restrict__ w, const float* __restrict__ g,
                                  float* __restrict__ m, float* __restrict__ v, long n, float lr,
                                  float b1, float b2, float eps, float c1, float c2) {
  long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.0f - b1) * gi;
  float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
