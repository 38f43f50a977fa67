// learned_pc.hip -- forward / backward / Adam kernels of the learned
// SH-space preconditioner (see learned_pc.hpp) and its hooks into the
// Galerkin solver vector.
#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

#include "learned_pc.hpp"
#include "runtime.hpp"

namespace v3d {

namespace {
inline unsigned gb(long n) {
  long b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  return (unsigned)(b < 1 ? 1 : b);
}
#define GL(i, n) \
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (long)gridDim.x * blockDim.x)

constexpr float kC0 = 0.7978845608028654f;  // sqrt(2/pi)
constexpr float kC1 = 0.044715f;

__device__ __forceinline__ float gelu_f(float x) {
  return 0.5f * x * (1.0f + tanhf(kC0 * (x + kC1 * x * x * x)));
}
__device__ __forceinline__ float gelu_g(float x) {
  const float t = tanhf(kC0 * (x + kC1 * x * x * x));
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * kC0 * (1.0f + 3.0f * kC1 * x * x);
}

// splitmix64 -> uniform in [-1, 1)
__device__ __forceinline__ float hash_uniform(unsigned long long s) {
  s += 0x9E3779B97F4A7C15ULL;
  s = (s ^ (s >> 30)) * 0xBF58476D1CE4E5B9ULL;
  s = (s ^ (s >> 27)) * 0x94D049BB133111EBULL;
  s ^= s >> 31;
  return (float)((double)(s >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0);
}

__global__ void k_init_uniform(float *p, long n, float a, unsigned long long seed) {
  GL(i, n) p[i] = a * hash_uniform(seed * 0x100000001B3ULL + (unsigned long long)i);
}
__global__ void k_bias_gelu(float *A, const float *__restrict__ b, long B, int w, float *H) {
  GL(i, B * w) {
    const float a = A[i] + b[i % w];
    A[i] = a;
    H[i] = gelu_f(a);
  }
}
__global__ void k_add_bias(float *Y, const float *__restrict__ b, long B, int w) {
  GL(i, B * w) Y[i] += b[i % w];
}
// dY = (Y - T) / n, per-block partial sums of (Y - T)^2 in FP64
__global__ __launch_bounds__(256) void k_diff_loss(const float *__restrict__ Y,
                                                   const float *__restrict__ T, long n, float invn,
                                                   float *dY, double *part) {
  double acc = 0;
  GL(i, n) {
    const float d = Y[i] - T[i];
    dY[i] = d * invn;
    acc += (double)d * d;
  }
  __shared__ double sh[4];
  acc = wave_sum(acc);
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}
// The sum of v over a workgroup of 256 (in thread 0), in a fixed order.
__device__ __forceinline__ double block_sum(double v) {
  __shared__ double sh[4];
  v = wave_sum(v);
  __syncthreads();
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  return sh[0] + sh[1] + sh[2] + sh[3];
}
// Latency-bound: one workgroup over the partials, 1152 in a minibatch of 1024 rows
// at order 16 (4 us for 4096; one thread adding them in turn took 218 us).
__global__ __launch_bounds__(256) void k_sum_parts(const double *__restrict__ part, int n,
                                                   double scale, double *out) {
  double s = 0;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  s = block_sum(s);
  if (threadIdx.x == 0) out[0] = s * scale;
}
__global__ void k_gelu_back(float *dH, const float *__restrict__ A, long n) {
  GL(i, n) dH[i] *= gelu_g(A[i]);
}
// Bias gradients: the column sums of the three layers' output gradients
// D_l [B][w_l] in one launch.  Latency-bound (5 MB at a batch of 1024): a
// workgroup takes 32 columns, 32 threads down each in steps of 32 rows, so
// that the reads are 128-byte runs and every column has 32 chains of loads in
// flight; the 32 partial sums are added in FP64 in order.  One thread per
// column took 227 us per layer, 0.7 ms of a 1.2 ms minibatch.
struct BiasGrads {
  const float *D[3];
  float *g[3];
  int w[3];
};
__global__ __launch_bounds__(1024) void k_bias_grads(const BiasGrads a, long B) {
  __shared__ float sh[32][33];
  const int c = threadIdx.x & 31, q = threadIdx.x >> 5;
  int l = 0, blk = blockIdx.x;
  while (blk >= (a.w[l] + 31) / 32) blk -= (a.w[l++] + 31) / 32;
  const int w = a.w[l], col = blk * 32 + c;
  float s = 0;
  if (col < w) {
    const float *__restrict__ D = a.D[l] + col;
#pragma unroll 8
    for (long r = q; r < B; r += 32) s += D[r * w];
  }
  sh[q][c] = s;
  __syncthreads();
  if (q == 0 && col < w) {
    double t = 0;
#pragma unroll
    for (int k = 0; k < 32; ++k) t += (double)sh[k][c];
    a.g[l][col] = (float)t;
  }
}
// ---- BF16 activations on MFMA
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Every product of the network has its contracted index contiguous in both
// operands, C[m][n] = sum_k A[m lda + k] B[n ldb + k]: what a product reads
// transposed is written transposed by its producer (HT below, and W2^T, W3^T
// beside the weights), with rows of ldt = B rounded up to 8, zero past B.

// Y[r][c] = bf16(X[r][c]) (round to nearest even) and its transpose
// YT[c][r] (ldt >= rows, zeros past them); either may be null.  One 32 x 32
// tile per workgroup.
struct ToBf16 {
  const float *X;
  __bf16 *Y, *YT;
  int rows, cols, ldt;
};
__device__ __forceinline__ void store_transposed(const __bf16 (&sh)[32][34], int r0, int c0,
                                                 int cols, int ldt, __bf16 *__restrict__ YT) {
  const int c = threadIdx.x >> 3, r = (threadIdx.x & 7) * 4;
  if (c0 + c >= cols || r0 + r >= ldt) return;
  const bf16x4 v = {sh[r][c], sh[r + 1][c], sh[r + 2][c], sh[r + 3][c]};
  *(bf16x4 *)(YT + (long)(c0 + c) * ldt + r0 + r) = v;
}
__global__ __launch_bounds__(256) void k_to_bf16(const ToBf16 a0, const ToBf16 a1,
                                                 const ToBf16 a2) {
  __shared__ __bf16 sh[32][34];
  const ToBf16 a = blockIdx.y == 0 ? a0 : (blockIdx.y == 1 ? a1 : a2);
  const int ct = (a.cols + 31) / 32;
  const int r0 = (int)(blockIdx.x / ct) * 32, c0 = (int)(blockIdx.x % ct) * 32;
  if (r0 >= a.rows) return;
  const int r = r0 + (threadIdx.x >> 3), c = c0 + (threadIdx.x & 7) * 4;
  bf16x4 v = {};
  if (r < a.rows && c < a.cols) {  // cols is a multiple of 4
    const float *x = a.X + (long)r * a.cols + c;
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = (__bf16)x[u];
    if (a.Y) *(bf16x4 *)(a.Y + (long)r * a.cols + c) = v;
  }
  if (!a.YT) return;
#pragma unroll
  for (int u = 0; u < 4; ++u) sh[threadIdx.x >> 3][(threadIdx.x & 7) * 4 + u] = v[u];
  __syncthreads();
  store_transposed(sh, r0, c0, a.cols, a.ldt, a.YT);
}

// What becomes of the product's tile (FP32 sums v):
enum GemmOut {
  kOutStore,    // C = v
  kOutBias,     // C = v + bias
  kOutGelu,     // a = v + bias (to C if given); H = bf16(gelu(a)), HT its transpose
  kOutGeluOdd,  // H[m] = bf16(gelu(v + bias)), H[M + m] = bf16(gelu(-v + bias))
  kOutOdd,      // A holds 2 M rows: C = ((v + bias) - (v' + bias)) / 2, v' of row M + m
  kOutLoss,     // d = v + bias - T; C = d / n, H = bf16(C), HT; part = sum d^2 of the tile
  kOutBack      // C = v gelu'(P), H = bf16(C), HT (P the pre-activations)
};
struct GemmEpi {
  float *C = nullptr;
  const float *bias = nullptr, *P = nullptr, *T = nullptr;
  __bf16 *H = nullptr, *HT = nullptr;
  double *part = nullptr;
  float invn = 0.0f;
  int ldt = 0;
};

// The epilogue of the 32 x 32 tile at (m0, n0): four consecutive columns of one
// row per thread, value(h, row, column) the tile's sums (h = 1: row M + m).
template <GemmOut OUT, typename V>
__device__ __forceinline__ void finish_tile(int M, int N, int m0, int n0, const GemmEpi &e,
                                            __bf16 (&sh)[32][34], long tile, V value) {
  constexpr int NS = OUT == kOutOdd ? 2 : 1;
  const int tid = threadIdx.x, tr = tid >> 3, tc = (tid & 7) * 4;
  const int m = m0 + tr, n = n0 + tc;
  const bool row = m < M;
  const long o = (long)m * N + n;
  double d2 = 0;
  bf16x4 hv = {};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float v[NS];
#pragma unroll
    for (int h = 0; h < NS; ++h) v[h] = value(h, tr, tc + u);
    if (!row || n + u >= N) continue;
    if constexpr (OUT == kOutStore) {
      e.C[o + u] = v[0];
    } else if constexpr (OUT == kOutBias) {
      e.C[o + u] = v[0] + e.bias[n + u];
    } else if constexpr (OUT == kOutGelu) {
      const float a = v[0] + e.bias[n + u];
      if (e.C) e.C[o + u] = a;
      hv[u] = (__bf16)gelu_f(a);
    } else if constexpr (OUT == kOutGeluOdd) {
      e.H[o + u] = (__bf16)gelu_f(v[0] + e.bias[n + u]);
      e.H[(long)M * N + o + u] = (__bf16)gelu_f(-v[0] + e.bias[n + u]);
    } else if constexpr (OUT == kOutOdd) {
      e.C[o + u] = 0.5f * ((v[0] + e.bias[n + u]) - (v[NS - 1] + e.bias[n + u]));
    } else if constexpr (OUT == kOutLoss) {
      const float d = v[0] + e.bias[n + u] - e.T[o + u];
      e.C[o + u] = d * e.invn;
      hv[u] = (__bf16)(d * e.invn);
      d2 += (double)d * d;
    } else {
      const float g = v[0] * gelu_g(e.P[o + u]);
      e.C[o + u] = g;
      hv[u] = (__bf16)g;
    }
  }
  if constexpr (OUT == kOutGelu || OUT == kOutLoss || OUT == kOutBack) {
    if (e.H && row && n < N) *(bf16x4 *)(e.H + o) = hv;  // N is a multiple of 8
    if (e.HT) {
#pragma unroll
      for (int u = 0; u < 4; ++u) sh[tr][tc + u] = hv[u];
      __syncthreads();
      store_transposed(sh, m0, n0, N, e.ldt, e.HT);
    }
  }
  if constexpr (OUT == kOutLoss) {
    d2 = block_sum(d2);
    if (tid == 0) e.part[tile] = d2;
  }
}

// A workgroup computes a 32 x 32 tile; its four waves take every fourth slab
// of 32 k and add their sums through LDS in wave order.  The operands go
// straight from memory to the MFMA registers: lane l supplies row l % 16 of
// each 16-row strip at k = 8 (l / 16) .. + 7 of the slab, one 16-byte load
// (the same k for both operands, so the k order inside the instruction does
// not matter), and holds results of rows 4 (l / 16) + r, column l % 16.
// Bound: latency.  The products of a minibatch are 0.1-0.6 GFLOP, under a
// microsecond of matrix work, so what counts is one workgroup per CU and all
// its loads in flight at once: 64 x 64 tiles through LDS, one slab after the
// other, took 12-32 us per product, this form 6.5-11.5 us with its elementwise
// stage, at a batch of 1024.
// Rows past M or N are clamped to the last one and not stored.  The host
// requires K, lda and ldb multiples of 8 and 16-byte aligned bases, so a
// vector is whole in range or whole out of it (then zero).
template <GemmOut OUT>
__global__ __launch_bounds__(256) void k_gemm_bf16(int M, int N, int K,
                                                   const __bf16 *__restrict__ A, long lda,
                                                   const __bf16 *__restrict__ B, long ldb,
                                                   const GemmEpi e) {
  constexpr int NS = OUT == kOutOdd ? 2 : 1;  // tiles of A that meet the same tile of B
  __shared__ float red[4][NS][32][33];
  __shared__ __bf16 sh[32][34];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * 32, n0 = blockIdx.y * 32;
  const __bf16 *pa[NS][2], *pb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const long m = min(m0 + 16 * i + li, M - 1), n = min(n0 + 16 * i + li, N - 1);
#pragma unroll
    for (int h = 0; h < NS; ++h) pa[h][i] = A + (m + (long)h * M) * lda + 8 * lg;
    pb[i] = B + n * ldb + 8 * lg;
  }
  f32x4 acc[NS][2][2] = {};
  auto slab = [&](int k0, bool whole) {
    bf16x8 a[NS][2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool in = whole || k0 + 8 * lg < K;
#pragma unroll
      for (int h = 0; h < NS; ++h) a[h][i] = in ? *(const bf16x8 *)(pa[h][i] + k0) : bf16x8{};
      b[i] = in ? *(const bf16x8 *)(pb[i] + k0) : bf16x8{};
    }
#pragma unroll
    for (int h = 0; h < NS; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[h][i][j] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], b[j], acc[h][i][j], 0, 0, 0);
  };
  int k0 = 32 * w;
  for (; k0 + 3 * 128 + 32 <= K; k0 += 4 * 128) {
#pragma unroll
    for (int u = 0; u < 4; ++u) slab(k0 + 128 * u, true);
  }
  for (; k0 + 32 <= K; k0 += 128) slab(k0, true);
  if (k0 < K) slab(k0, false);
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[w][h][16 * i + 4 * lg + r][16 * j + li] = acc[h][i][j][r];
  __syncthreads();
  finish_tile<OUT>(M, N, m0, n0, e, sh, (long)blockIdx.y * gridDim.x + blockIdx.x,
                   [&](int h, int r, int c) {
                     return ((red[0][h][r][c] + red[1][h][r][c]) + red[2][h][r][c]) +
                            red[3][h][r][c];
                   });
}

// The same for large products: a 64 x 64 tile, each wave 32 x 32 of it over all
// of K, slabs of 32 k staged through LDS, so that an operand's row is read once
// per 64 columns.  Bound: the operands' reads; the form above reads twice as much
// (forward pass, 1152-1024-1024-1152, batch 4096: 103 us here, 208 there).
// Workgroups reach the XCDs in turn: an XCD's take the column tiles of one row
// tile one after the other, which then finds its A rows in that L2.
template <GemmOut OUT>
__global__ __launch_bounds__(256) void k_gemm_bf16_lds(int M, int N, int K,
                                                       const __bf16 *__restrict__ A, long lda,
                                                       const __bf16 *__restrict__ B, long ldb,
                                                       const GemmEpi e) {
  constexpr int NS = OUT == kOutOdd ? 2 : 1, kPitch = 40;
  __shared__ __attribute__((aligned(16))) __bf16 As[NS][64][kPitch];
  __shared__ __attribute__((aligned(16))) __bf16 Bs[64][kPitch];
  __shared__ float sums[NS][64][65];
  __shared__ __bf16 sh[32][34];
  const int nt = (N + 63) / 64;
  const long q = blockIdx.x / 8, m_tile = q / nt * 8 + blockIdx.x % 8;
  if (m_tile >= (M + 63) / 64) return;
  const int m0 = (int)m_tile * 64, n0 = (int)(q % nt) * 64;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lg = lane >> 4, wm = (w >> 1) * 32, wn = (w & 1) * 32;
  const int sr = tid >> 2, sk = (tid & 3) * 8;  // the vector that this thread stages
  f32x4 acc[NS][2][2] = {};
  for (int k0 = 0; k0 < K; k0 += 32) {
    const bool in = k0 + sk < K;
#pragma unroll
    for (int h = 0; h < NS; ++h)
      *(bf16x8 *)&As[h][sr][sk] =
          in && m0 + sr < M
              ? *(const bf16x8 *)(A + (m0 + sr + (long)h * M) * lda + k0 + sk)
              : bf16x8{};
    *(bf16x8 *)&Bs[sr][sk] =
        in && n0 + sr < N ? *(const bf16x8 *)(B + (n0 + sr) * ldb + k0 + sk) : bf16x8{};
    __syncthreads();
    bf16x8 b[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) b[j] = *(const bf16x8 *)&Bs[wn + 16 * j + li][8 * lg];
#pragma unroll
    for (int h = 0; h < NS; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8 a = *(const bf16x8 *)&As[h][wm + 16 * i + li][8 * lg];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[h][i][j] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j], acc[h][i][j], 0, 0, 0);
      }
    __syncthreads();
  }
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sums[h][wm + 16 * i + 4 * lg + r][wn + 16 * j + li] = acc[h][i][j][r];
  __syncthreads();
  const int mt32 = (M + 31) / 32;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) {
      const int m = m0 + 32 * i, n = n0 + 32 * j;
      if (m >= M || n >= N) continue;
      finish_tile<OUT>(M, N, m, n, e, sh, (long)(n / 32) * mt32 + m / 32,
                       [&](int h, int r, int c) { return sums[h][32 * i + r][32 * j + c]; });
      __syncthreads();  // sh is read
    }
}

template <GemmOut OUT>
int gemm_bf16(long M, int N, long K, const __bf16 *A, long lda, const __bf16 *B, long ldb,
              const GemmEpi &e, hipStream_t st) {
  if (M < 1 || N < 1 || K < 1 || K > 0x7fffff00L) return VES3D_INVALID_PARAMETER;
  if (K % 8 || N % 8 || lda % 8 || ldb % 8) return VES3D_INVALID_PARAMETER;
  if (((uintptr_t)A | (uintptr_t)B) & 15) return VES3D_INVALID_PARAMETER;
  const unsigned gy = cdiv(N, 32);
  if (M > 0x7fffff00L || gy > 65535) return VES3D_INVALID_PARAMETER;
  // The LDS form where its tiles give every CU two workgroups and the operands'
  // reads bound the product: forward pass 1152-512-512-1152, batch 4096 (512 tiles,
  // 2.4e9 multiplications) 102 / 72 us, 2000 (256 tiles) 56 / 62; the weight
  // gradients' few tiles (a quarter of these or less) take twice the time in it.
  const long mt = cdiv(M, 64), nt = cdiv(N, 64);
  if (mt * nt >= 512 && M * N * K >= 2000000000L) {
    const long groups = (mt + 7) / 8 * 8 * nt;
    if (groups > 0x7fffffffL) return VES3D_INVALID_PARAMETER;
    k_gemm_bf16_lds<OUT><<<(unsigned)groups, 256, 0, st>>>((int)M, N, (int)K, A, lda, B, ldb, e);
    return launch_status();
  }
  k_gemm_bf16<OUT><<<dim3(cdiv(M, 32), gy), 256, 0, st>>>((int)M, N, (int)K, A, lda, B, ldb, e);
  return launch_status();
}

// out = -in
__global__ void k_negate(const float *__restrict__ in, long n, float *out) {
  GL(i, n) out[i] = -in[i];
}
// Y = (Y - Yneg) / 2: the odd part g(z) - g(-z) of the network, so that the
// preconditioner satisfies P(-r) = -P(r) (with the row scaling, P(a r) =
// a P(r) for every real a)
__global__ void k_odd_part(float *Y, const float *__restrict__ Yneg, long n) {
  GL(i, n) Y[i] = 0.5f * (Y[i] - Yneg[i]);
}
// minibatch rows Zb[i] = sgn Zs[perm[i]], Tb[i] = sgn Ts[perm[i]], with
// sgn = -1 on odd batch rows: the samples enter with both signs, as the
// target map is odd
__global__ void k_gather_batch(const float *__restrict__ Zs, const float *__restrict__ Ts,
                               const int *__restrict__ perm, long B, int nin, float *Zb, float *Tb) {
  GL(i, B * nin) {
    const long r = i / nin;
    const long src = (long)perm[r] * nin + (i % nin);
    const float sg = (r & 1) ? -1.0f : 1.0f;
    Zb[i] = sg * Zs[src];
    Tb[i] = sg * Ts[src];
  }
}
// partial sums of (Y - T)^2 and T^2 per block into part[2 * block + {0, 1}]
__global__ __launch_bounds__(256) void k_sq_sums(const float *__restrict__ Y,
                                                 const float *__restrict__ T, long n,
                                                 double *part) {
  double a = 0, b = 0;
  GL(i, n) {
    const double d = (double)Y[i] - (double)T[i];
    a += d * d;
    b += (double)T[i] * (double)T[i];
  }
  __shared__ double sh[2][4];
  a = wave_sum(a);
  b = wave_sum(b);
  if (threadIdx.x % 64 == 0) {
    sh[0][threadIdx.x / 64] = a;
    sh[1][threadIdx.x / 64] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
    part[2 * blockIdx.x + 1] = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
  }
}
// acc[0..1] += sums of the nb partial pairs (one workgroup, fixed order)
__global__ __launch_bounds__(256) void k_acc_pairs(const double *__restrict__ part, int nb,
                                                   double *acc) {
  double a = 0, b = 0;
  for (int k = threadIdx.x; k < nb; k += 256) {
    a += part[2 * k];
    b += part[2 * k + 1];
  }
  a = block_sum(a);
  b = block_sum(b);
  if (threadIdx.x == 0) {
    acc[0] += a;
    acc[1] += b;
  }
}
// Adam (Kingma & Ba 2015, Algorithm 1) with decoupled weight decay wd
// (Loshchilov & Hutter 2019): P -= lr (m_hat / (sqrt(v_hat) + eps) + wd P)
__global__ void k_adam(float *P, const float *__restrict__ G, float *M, float *V, long n, float lr,
                       float c1, float c2, float wd) {
  GL(i, n) {
    const float g = G[i];
    const float m = 0.9f * M[i] + 0.1f * g;
    const float v = 0.999f * V[i] + 0.001f * g * g;
    M[i] = m;
    V[i] = v;
    P[i] -= lr * ((m / c1) / (sqrtf(v / c2) + 1e-8f) + wd * P[i]);
  }
}

// Row element j of vesicle v inside the order-major Galerkin vector.
__device__ __forceinline__ long row_index(long v, int j, long nv, int nc, const int2 *cinfo) {
  long base, f, nf;
  int c;
  if (j < 3 * nc) {
    const int d = j / nc;
    c = j % nc;
    f = 3 * v + d;
    nf = 3 * nv;
    base = 0;
  } else {
    c = j - 3 * nc;
    f = v;
    nf = nv;
    base = 3 * nv * (long)nc;
  }
  const int2 bl = cinfo[c];
  return base + nf * bl.x + f * bl.y + (c - bl.x);
}

// scale[v] = |row_v(y)|, one workgroup per vesicle
__global__ __launch_bounds__(256) void k_row_norms(const double *__restrict__ y, long nv, int nc,
                                                   const int2 *__restrict__ cinfo, double *scale) {
  const long v = blockIdx.x;
  double acc = 0;
  for (int j = threadIdx.x; j < 4 * nc; j += 256) {
    const double a = y[row_index(v, j, nv, nc, cinfo)];
    acc += a * a;
  }
  __shared__ double sh[4];
  acc = wave_sum(acc);
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = acc;
  __syncthreads();
  if (threadIdx.x == 0) scale[v] = sqrt(sh[0] + sh[1] + sh[2] + sh[3]) + 1e-300;
}
// Frames F_v (row-major 3x3 per vesicle, columns the vesicle's canonical
// axes; nullptr: identity) rotate the three velocity blocks of a vesicle's
// row into its canonical frame, z_d = sum_e F[e][d] x_e, and back,
// x_e = sum_d F[e][d] z_d.  The tension block is a scalar and not rotated.
__device__ __forceinline__ double to_canonical(const double *__restrict__ y, long v, int j, long nv,
                                               int nc, const int2 *__restrict__ cinfo,
                                               const double *__restrict__ frames) {
  if (j >= 3 * nc || frames == nullptr) return y[row_index(v, j, nv, nc, cinfo)];
  const int d = j / nc, c = j % nc;
  const double *F = frames + 9 * v;
  double z = 0;
#pragma unroll
  for (int e = 0; e < 3; ++e) z += F[3 * e + d] * y[row_index(v, e * nc + c, nv, nc, cinfo)];
  return z;
}

template <typename T>
__global__ void k_gather_rows(const double *__restrict__ y, long nv, int nc,
                              const int2 *__restrict__ cinfo, const double *__restrict__ scale,
                              const double *__restrict__ frames, T *Z) {
  const int nin = 4 * nc;
  GL(i, nv * nin) {
    const long v = i / nin;
    const int j = (int)(i % nin);
    Z[i] = (T)(float)(to_canonical(y, v, j, nv, nc, cinfo, frames) / scale[v]);
  }
}
// The correction skips the tension coefficients of degree > tcut: the
// surface divergence is low-pass filtered at that degree (src/Surface.cc:372),
// so those coefficients span the null space of the implicit operator, and
// the solution the diagonal-preconditioned solve reaches has them at zero.
__global__ void k_scatter_add(const float *__restrict__ Y, long nv, int nc, int p, int tcut,
                              const int2 *__restrict__ cinfo, const double *__restrict__ scale,
                              const double *__restrict__ frames, double *y) {
  const int nin = 4 * nc;
  GL(i, nv * nin) {
    const long v = i / nin;
    const int j = (int)(i % nin);
    double add;
    if (j >= 3 * nc) {
      const int c = j - 3 * nc;
      const int2 bl = cinfo[c];
      const int degree = (p + 1 - bl.y) + (c - bl.x);  // order m = p + 1 - block length
      if (degree > tcut) continue;
      add = (double)Y[i];
    } else if (frames == nullptr) {
      add = (double)Y[i];
    } else {
      const int e = j / nc, c = j % nc;
      const double *F = frames + 9 * v;
      const float *Yv = Y + v * nin;
      add = F[3 * e] * (double)Yv[c] + F[3 * e + 1] * (double)Yv[nc + c] +
            F[3 * e + 2] * (double)Yv[2 * nc + c];
    }
    y[row_index(v, j, nv, nc, cinfo)] += scale[v] * add;
  }
}
// samples in the canonical frames: Z = F^T Dr_v / s, T = F^T (e_v - Dr_v) / s,
// written at rows slot0 + v (mod cap)
__global__ void k_record(const double *__restrict__ Dr, const double *__restrict__ e, long nv,
                         int nc, const int2 *__restrict__ cinfo, const double *__restrict__ scale,
                         const double *__restrict__ frames, long slot0, long cap, float *Zs,
                         float *Ts) {
  const int nin = 4 * nc;
  GL(i, nv * nin) {
    const long v = i / nin;
    const int j = (int)(i % nin);
    const long row = (slot0 + v) % cap;
    const double s = scale[v];
    const double z = to_canonical(Dr, v, j, nv, nc, cinfo, frames);
    const double t = to_canonical(e, v, j, nv, nc, cinfo, frames);
    Zs[row * nin + j] = (float)(z / s);
    Ts[row * nin + j] = (float)((t - z) / s);
  }
}
}  // namespace

LearnedPC::~LearnedPC() {
  for (float *p : {P_, G_, M_, V_, Zs_, Ts_, A1_, H1_, A2_, H2_, Y_, dY_, dA2_, dA1_, Zb_, Tb_,
                   Zneg_, Yneg_})
    if (p) (void)hipFree(p);
  if (scale_) (void)hipFree(scale_);
  if (lossbuf_) (void)hipFree(lossbuf_);
  if (evalbuf_) (void)hipFree(evalbuf_);
  if (perm_) (void)hipFree(perm_);
  if (vidx_) (void)hipFree(vidx_);
  if (Pbest_) (void)hipFree(Pbest_);
  for (__bf16 *p : {Wh_, Zh_, H1h_, H2h_, dYh_, dA2h_, trh_})
    if (p) (void)hipFree(p);
  if (part_) (void)hipFree(part_);
  for (auto &kv : descs_) (void)hipFree(kv.second);
}

int LearnedPC::set_activations(int mode) {
  if (mode != 0 && mode != 1) return VES3D_INVALID_PARAMETER;
  if (mode == 1 && (nin_ % 8 || width_ % 8)) return VES3D_INVALID_PARAMETER;
  if (mode == 1 && !Wh_) {
    // [W1 | W2 | W3 | W2^T | W3^T]
    const long nw = (long)width_ * nin_ * 3 + 2L * width_ * width_;
    if (hipMalloc(&Wh_, sizeof(__bf16) * nw) != hipSuccess) return VES3D_MEMORY_ERROR;
  }
  act_ = mode;
  wdirty_ = true;
  // reallocate the batch buffers at the current capacity with the new
  // mode's operand buffers
  const long b = bcap_;
  bcap_ = 0;
  return b > 0 ? ensure_batch(b) : VES3D_SUCCESS;
}

int LearnedPC::refresh_bf16(hipStream_t st) {
  if (!wdirty_) return VES3D_SUCCESS;
  const int w = width_, n = nin_;
  const long wn = (long)w * n, ww = (long)w * w;
  const ToBf16 a1{P_ + oW1_, Wh_, nullptr, w, n, 0};
  const ToBf16 a2{P_ + oW2_, Wh_ + wn, Wh_ + 2 * wn + ww, w, w, w};
  const ToBf16 a3{P_ + oW3_, Wh_ + wn + ww, Wh_ + 2 * wn + 2 * ww, n, w, n};
  k_to_bf16<<<dim3(cdiv(w, 32) * std::max(cdiv(w, 32), cdiv(n, 32)), 3), 256, 0, st>>>(a1, a2, a3);
  V3D_CHECK(launch_status());
  wdirty_ = false;
  return VES3D_SUCCESS;
}

int LearnedPC::init(int nin, int width, long capacity, unsigned long long seed) {
  nin_ = nin;
  width_ = width;
  cap_ = capacity;
  seed_ = seed;
  oW1_ = 0;
  ob1_ = oW1_ + (long)width * nin;
  oW2_ = ob1_ + width;
  ob2_ = oW2_ + (long)width * width;
  oW3_ = ob2_ + width;
  ob3_ = oW3_ + (long)nin * width;
  np_ = ob3_ + nin;
  for (float **p : {&P_, &G_, &M_, &V_})
    if (hipMalloc(p, sizeof(float) * np_) != hipSuccess) return VES3D_MEMORY_ERROR;
  V3D_HIP(hipMemset(P_, 0, sizeof(float) * np_));
  V3D_HIP(hipMemset(M_, 0, sizeof(float) * np_));
  V3D_HIP(hipMemset(V_, 0, sizeof(float) * np_));
  // Glorot-uniform hidden layers; the output layer starts small so that
  // the untrained preconditioner is close to D.
  const float a1 = std::sqrt(6.0f / (nin + width)), a2 = std::sqrt(6.0f / (2.0f * width));
  k_init_uniform<<<gb((long)width * nin), 256>>>(P_ + oW1_, (long)width * nin, a1, seed * 3 + 1);
  k_init_uniform<<<gb((long)width * width), 256>>>(P_ + oW2_, (long)width * width, a2, seed * 3 + 2);
  k_init_uniform<<<gb((long)nin * width), 256>>>(P_ + oW3_, (long)nin * width, 0.01f * a1, seed * 3 + 3);
  V3D_CHECK(launch_status());
  if (cap_ > 0) {
    if (hipMalloc(&Zs_, sizeof(float) * cap_ * nin) != hipSuccess) return VES3D_MEMORY_ERROR;
    if (hipMalloc(&Ts_, sizeof(float) * cap_ * nin) != hipSuccess) return VES3D_MEMORY_ERROR;
  }
  if (hipMalloc(&lossbuf_, sizeof(double) * 4200) != hipSuccess) return VES3D_MEMORY_ERROR;
  if (hipMalloc(&evalbuf_, sizeof(double) * (2 + 2 * kEvalParts)) != hipSuccess)
    return VES3D_MEMORY_ERROR;
  return hip_status(hipDeviceSynchronize());
}

int LearnedPC::ensure_batch(long B) {
  if (B <= bcap_) return VES3D_SUCCESS;
  for (float *p : {A1_, H1_, A2_, H2_, Y_, dY_, dA2_, dA1_, Zb_, Tb_, Zneg_, Yneg_})
    if (p) (void)hipFree(p);
  if (scale_) (void)hipFree(scale_);
  const long w = width_, n = nin_;
  float **wb[] = {&A1_, &H1_, &A2_, &H2_, &dA2_, &dA1_};
  for (float **p : wb)
    if (hipMalloc(p, sizeof(float) * B * w) != hipSuccess) return VES3D_MEMORY_ERROR;
  float **nb[] = {&Y_, &dY_, &Zb_, &Tb_, &Zneg_, &Yneg_};
  for (float **p : nb)
    if (hipMalloc(p, sizeof(float) * B * n) != hipSuccess) return VES3D_MEMORY_ERROR;
  if (hipMalloc(&scale_, sizeof(double) * B) != hipSuccess) return VES3D_MEMORY_ERROR;
  for (__bf16 *p : {Zh_, H1h_, H2h_, dYh_, dA2h_, trh_})
    if (p) (void)hipFree(p);
  Zh_ = H1h_ = H2h_ = dYh_ = dA2h_ = trh_ = nullptr;
  if (part_) (void)hipFree(part_);
  part_ = nullptr;
  if (act_ == 1) {
    // the hidden activations hold both signs' rows (odd_forward)
    for (__bf16 **p : {&H1h_, &H2h_})
      if (hipMalloc(p, sizeof(__bf16) * 2 * B * w) != hipSuccess) return VES3D_MEMORY_ERROR;
    if (hipMalloc(&dA2h_, sizeof(__bf16) * B * w) != hipSuccess) return VES3D_MEMORY_ERROR;
    for (__bf16 **p : {&Zh_, &dYh_})
      if (hipMalloc(p, sizeof(__bf16) * B * n) != hipSuccess) return VES3D_MEMORY_ERROR;
    // transposed operands of the weight gradients: Z, dY, H1, H2, dA1, dA2
    const long bt = (B + 7) / 8 * 8;
    if (hipMalloc(&trh_, sizeof(__bf16) * bt * (2 * n + 4 * w)) != hipSuccess)
      return VES3D_MEMORY_ERROR;
    if (hipMalloc(&part_, sizeof(double) * cdiv(B, 32) * cdiv(n, 32)) != hipSuccess)
      return VES3D_MEMORY_ERROR;
  }
  bcap_ = B;
  return VES3D_SUCCESS;
}

// C[M][N] = A B with A(r,k) = A[r ars + k acs], B(k,c) = B[k brs + c bcs]
int LearnedPC::gemm(int M, int N, int K, const float *A, long ars, long acs, const float *Bm,
                    long brs, long bcs, float *C, hipStream_t st) {
  auto key = std::make_tuple(M, N, K, ars, acs, brs, bcs);
  GemmDesc h{};
  h.M = M;
  h.N = N;
  h.K = K;
  h.a_rs = ars;
  h.a_cs = acs;
  h.b_rs = brs;
  h.b_cs = bcs;
  h.c_rs = N;
  h.c_cs = 1;
  GemmDesc *d = nullptr;
  auto it = descs_.find(key);
  if (it != descs_.end()) {
    d = it->second;
  } else {
    d = upload_descs(&h, 1);
    if (!d) return VES3D_MEMORY_ERROR;
    descs_[key] = d;
  }
  return gemm_grouped<float>(d, 1, 1, M, N, A, Bm, C, 1.0f, 0.0f, st, gemm_pick_tile(&h, 1));
}

int LearnedPC::forward(const float *Z, long B, float *Y, hipStream_t st) {
  V3D_CHECK(ensure_batch(B));
  const int w = width_, n = nin_;
  if (act_ == 1) {
    // BF16 operands (weights rounded from the FP32 master copy), FP32
    // accumulation, pre-activations and output
    V3D_CHECK(refresh_bf16(st));
    const ToBf16 a{Z, Zh_, nullptr, (int)B, n, 0};
    k_to_bf16<<<cdiv(B, 32) * cdiv(n, 32), 256, 0, st>>>(a, a, a);
    V3D_CHECK(launch_status());
    GemmEpi e;
    e.bias = P_ + ob1_;
    e.H = H1h_;
    V3D_CHECK(gemm_bf16<kOutGelu>(B, w, n, Zh_, n, W1h(), n, e, st));
    e.bias = P_ + ob2_;
    e.H = H2h_;
    V3D_CHECK(gemm_bf16<kOutGelu>(B, w, w, H1h_, w, W2h(), w, e, st));
    GemmEpi y;
    y.bias = P_ + ob3_;
    y.C = Y;
    return gemm_bf16<kOutBias>(B, n, w, H2h_, w, W3h(), w, y, st);
  }
  V3D_CHECK(gemm((int)B, w, n, Z, n, 1, P_ + oW1_, 1, n, A1_, st));   // Z W1^T
  k_bias_gelu<<<gb(B * w), 256, 0, st>>>(A1_, P_ + ob1_, B, w, H1_);
  V3D_CHECK(launch_status());
  V3D_CHECK(gemm((int)B, w, w, H1_, w, 1, P_ + oW2_, 1, w, A2_, st));  // H1 W2^T
  k_bias_gelu<<<gb(B * w), 256, 0, st>>>(A2_, P_ + ob2_, B, w, H2_);
  V3D_CHECK(launch_status());
  V3D_CHECK(gemm((int)B, n, w, H2_, w, 1, P_ + oW3_, 1, w, Y, st));    // H2 W3^T
  k_add_bias<<<gb(B * n), 256, 0, st>>>(Y, P_ + ob3_, B, n);
  return launch_status();
}

int LearnedPC::bias_grads(long B, hipStream_t st) {
  const BiasGrads a{{dY_, dA2_, dA1_}, {G_ + ob3_, G_ + ob2_, G_ + ob1_}, {nin_, width_, width_}};
  k_bias_grads<<<cdiv(nin_, 32) + 2 * cdiv(width_, 32), 1024, 0, st>>>(a, B);
  return launch_status();
}

// BF16 operands of every product, FP32 pre-activations, gradients and bias sums
int LearnedPC::loss_grad_bf16(const float *Z, const float *T, long B, double *loss_host,
                              hipStream_t st) {
  V3D_CHECK(ensure_batch(B));
  V3D_CHECK(refresh_bf16(st));
  const int w = width_, n = nin_;
  const long tot = B * n, bt = (B + 7) / 8 * 8;
  __bf16 *Zt = trh_, *dYt = Zt + bt * n, *H1t = dYt + bt * n, *H2t = H1t + bt * w,
         *dA1t = H2t + bt * w, *dA2t = dA1t + bt * w;
  const ToBf16 a{Z, Zh_, Zt, (int)B, n, (int)bt};
  k_to_bf16<<<cdiv(B, 32) * cdiv(n, 32), 256, 0, st>>>(a, a, a);
  V3D_CHECK(launch_status());
  auto epi = [&](float *C, const float *bias, __bf16 *H, __bf16 *HT) {
    GemmEpi e;
    e.C = C;
    e.bias = bias;
    e.H = H;
    e.HT = HT;
    e.ldt = (int)bt;
    return e;
  };
  V3D_CHECK(gemm_bf16<kOutGelu>(B, w, n, Zh_, n, W1h(), n, epi(A1_, P_ + ob1_, H1h_, H1t), st));
  V3D_CHECK(gemm_bf16<kOutGelu>(B, w, w, H1h_, w, W2h(), w, epi(A2_, P_ + ob2_, H2h_, H2t), st));
  GemmEpi l = epi(dY_, P_ + ob3_, dYh_, dYt);
  l.T = T;
  l.invn = 1.0f / (float)tot;
  l.part = part_;
  V3D_CHECK(gemm_bf16<kOutLoss>(B, n, w, H2h_, w, W3h(), w, l, st));
  k_sum_parts<<<1, 256, 0, st>>>(part_, (int)(cdiv(B, 32) * cdiv(n, 32)), 0.5 / (double)tot,
                                 lossbuf_ + 4100);
  V3D_CHECK(launch_status());
  // input gradients, dY W3 and dA2 W2, through the activations
  GemmEpi g = epi(dA2_, nullptr, dA2h_, dA2t);
  g.P = A2_;
  V3D_CHECK(gemm_bf16<kOutBack>(B, w, n, dYh_, n, W3t(), n, g, st));
  g = epi(dA1_, nullptr, nullptr, dA1t);
  g.P = A1_;
  V3D_CHECK(gemm_bf16<kOutBack>(B, w, w, dA2h_, w, W2t(), w, g, st));
  // weight gradients dY^T H2, dA2^T H1, dA1^T Z: K is the batch, padded to bt
  V3D_CHECK(gemm_bf16<kOutStore>(n, w, bt, dYt, bt, H2t, bt, epi(G_ + oW3_, nullptr, nullptr, nullptr), st));
  V3D_CHECK(gemm_bf16<kOutStore>(w, w, bt, dA2t, bt, H1t, bt, epi(G_ + oW2_, nullptr, nullptr, nullptr), st));
  V3D_CHECK(gemm_bf16<kOutStore>(w, n, bt, dA1t, bt, Zt, bt, epi(G_ + oW1_, nullptr, nullptr, nullptr), st));
  V3D_CHECK(bias_grads(B, st));
  if (loss_host) {
    V3D_HIP(hipMemcpyAsync(loss_host, lossbuf_ + 4100, sizeof(double), hipMemcpyDeviceToHost, st));
    V3D_HIP(hipStreamSynchronize(st));
  }
  return VES3D_SUCCESS;
}

int LearnedPC::loss_grad(const float *Z, const float *T, long B, double *loss_host,
                         hipStream_t st) {
  const int w = width_, n = nin_;
  const long tot = B * n;
  if (act_ == 1) return loss_grad_bf16(Z, T, B, loss_host, st);
  V3D_CHECK(forward(Z, B, Y_, st));
  const int nb = (int)std::min<long>(4096, std::max<long>(1, (tot + 255) / 256));
  k_diff_loss<<<nb, 256, 0, st>>>(Y_, T, tot, 1.0f / (float)tot, dY_, lossbuf_);
  V3D_CHECK(launch_status());
  k_sum_parts<<<1, 256, 0, st>>>(lossbuf_, nb, 0.5 / (double)tot, lossbuf_ + 4100);
  V3D_CHECK(launch_status());
  // layer 3
  V3D_CHECK(gemm(n, w, (int)B, dY_, 1, n, H2_, w, 1, G_ + oW3_, st));  // dY^T H2
  V3D_CHECK(gemm((int)B, w, n, dY_, n, 1, P_ + oW3_, w, 1, dA2_, st));  // dY W3
  k_gelu_back<<<gb(B * w), 256, 0, st>>>(dA2_, A2_, B * w);
  V3D_CHECK(launch_status());
  // layer 2
  V3D_CHECK(gemm(w, w, (int)B, dA2_, 1, w, H1_, w, 1, G_ + oW2_, st));
  V3D_CHECK(gemm((int)B, w, w, dA2_, w, 1, P_ + oW2_, w, 1, dA1_, st));
  k_gelu_back<<<gb(B * w), 256, 0, st>>>(dA1_, A1_, B * w);
  V3D_CHECK(launch_status());
  // layer 1
  V3D_CHECK(gemm(w, n, (int)B, dA1_, 1, w, Z, n, 1, G_ + oW1_, st));
  V3D_CHECK(bias_grads(B, st));
  if (loss_host) {
    V3D_HIP(hipMemcpyAsync(loss_host, lossbuf_ + 4100, sizeof(double), hipMemcpyDeviceToHost, st));
    V3D_HIP(hipStreamSynchronize(st));
  }
  return VES3D_SUCCESS;
}

int LearnedPC::reset_optimizer() {
  V3D_HIP(hipMemset(M_, 0, sizeof(float) * np_));
  V3D_HIP(hipMemset(V_, 0, sizeof(float) * np_));
  t_ = 0;
  return VES3D_SUCCESS;
}

int LearnedPC::adam(float lr, hipStream_t st) {
  ++t_;
  const float c1 = 1.0f - std::pow(0.9f, (float)t_), c2 = 1.0f - std::pow(0.999f, (float)t_);
  k_adam<<<gb(np_), 256, 0, st>>>(P_, G_, M_, V_, np_, lr, c1, c2, wd_);
  wdirty_ = true;
  return launch_status();
}

int LearnedPC::subset_loss(const int *idx, long m, double *loss_host, double *target_ms_host,
                            hipStream_t st) {
  const long B = std::min<long>(std::max<long>(bcap_, 1), m);
  V3D_CHECK(ensure_batch(B));
  double *acc = evalbuf_, *part = evalbuf_ + 2;
  V3D_HIP(hipMemsetAsync(acc, 0, 2 * sizeof(double), st));
  for (long r0 = 0; r0 < m; r0 += B) {
    const long cnt = std::min(B, m - r0);
    k_gather_batch<<<gb(cnt * nin_), 256, 0, st>>>(Zs_, Ts_, idx + r0, cnt, nin_, Zb_, Tb_);
    V3D_CHECK(launch_status());
    V3D_CHECK(odd_forward(Zb_, cnt, Y_, st));
    const long tot = cnt * nin_;
    const int nb = (int)std::min<long>(kEvalParts, std::max<long>(1, (tot + 255) / 256));
    k_sq_sums<<<nb, 256, 0, st>>>(Y_, Tb_, tot, part);
    V3D_CHECK(launch_status());
    k_acc_pairs<<<1, 256, 0, st>>>(part, nb, acc);
    V3D_CHECK(launch_status());
  }
  double h[2];
  V3D_HIP(hipMemcpyAsync(h, acc, sizeof(h), hipMemcpyDeviceToHost, st));
  V3D_HIP(hipStreamSynchronize(st));
  const double n = (double)m * nin_;
  if (loss_host) *loss_host = 0.5 * h[0] / n;
  if (target_ms_host) *target_ms_host = h[1] / n;
  return VES3D_SUCCESS;
}

int LearnedPC::dataset_loss(long have, double *loss_host, double *target_ms_host,
                            hipStream_t st) {
  if (!perm_ && hipMalloc(&perm_, sizeof(int) * cap_) != hipSuccess) return VES3D_MEMORY_ERROR;
  std::vector<int> all(have);
  for (long i = 0; i < have; ++i) all[i] = (int)i;
  V3D_HIP(hipStreamSynchronize(st));
  V3D_HIP(hipMemcpy(perm_, all.data(), sizeof(int) * have, hipMemcpyHostToDevice));
  return subset_loss(perm_, have, loss_host, target_ms_host, st);
}

int LearnedPC::train(int epochs, int batch, float lr, double *last_loss, hipStream_t st) {
  const long have = std::min(count_, cap_);
  if (have < 2 || batch < 1 || epochs < 1) return VES3D_INVALID_PARAMETER;
  // a fixed tenth of the samples is held out; the kept parameters are those
  // with the lowest held-out loss (evaluated after every epoch)
  const long nval = std::max<long>(1, have / 10), ntr = have - nval;
  const long B = std::min<long>(batch, ntr);
  V3D_CHECK(ensure_batch(B));
  if (!perm_ && hipMalloc(&perm_, sizeof(int) * cap_) != hipSuccess) return VES3D_MEMORY_ERROR;
  if (!vidx_ && hipMalloc(&vidx_, sizeof(int) * cap_) != hipSuccess) return VES3D_MEMORY_ERROR;
  if (!Pbest_ && hipMalloc(&Pbest_, sizeof(float) * np_) != hipSuccess) return VES3D_MEMORY_ERROR;
  std::mt19937_64 split(seed_ + 777);
  std::vector<int> all(have);
  for (long i = 0; i < have; ++i) all[i] = (int)i;
  std::shuffle(all.begin(), all.end(), split);
  std::vector<int> tr(all.begin() + nval, all.end());
  V3D_HIP(hipStreamSynchronize(st));
  V3D_HIP(hipMemcpy(vidx_, all.data(), sizeof(int) * nval, hipMemcpyHostToDevice));
  std::mt19937_64 rng(seed_ + 12345 + (unsigned long long)t_);
  const long per_epoch = std::max<long>(1, ntr / B);
  const long total = epochs * per_epoch;
  // Adam over shuffled minibatches with a cosine learning-rate decay
  double best = 0;
  V3D_CHECK(subset_loss(vidx_, nval, &best, nullptr, st));
  V3D_HIP(hipMemcpyAsync(Pbest_, P_, sizeof(float) * np_, hipMemcpyDeviceToDevice, st));
  long k = 0;
  for (int ep = 0; ep < epochs; ++ep) {
    std::shuffle(tr.begin(), tr.end(), rng);
    V3D_HIP(hipStreamSynchronize(st));
    V3D_HIP(hipMemcpy(perm_, tr.data(), sizeof(int) * ntr, hipMemcpyHostToDevice));
    for (long b = 0; b < per_epoch; ++b, ++k) {
      k_gather_batch<<<gb(B * nin_), 256, 0, st>>>(Zs_, Ts_, perm_ + b * B, B, nin_, Zb_, Tb_);
      V3D_CHECK(launch_status());
      V3D_CHECK(loss_grad(Zb_, Tb_, B, nullptr, st));
      const double c = 0.5 * (1.0 + std::cos(M_PI * (double)k / (double)total));
      V3D_CHECK(adam((float)(lr * c), st));
    }
    double l = 0;
    V3D_CHECK(subset_loss(vidx_, nval, &l, nullptr, st));
    if (l < best) {
      best = l;
      best_epoch_ = ep + 1;
      V3D_HIP(hipMemcpyAsync(Pbest_, P_, sizeof(float) * np_, hipMemcpyDeviceToDevice, st));
    }
  }
  V3D_HIP(hipMemcpyAsync(P_, Pbest_, sizeof(float) * np_, hipMemcpyDeviceToDevice, st));
  wdirty_ = true;
  if (last_loss) *last_loss = best;
  trained_ = true;
  return hip_status(hipStreamSynchronize(st));
}

int LearnedPC::apply_inplace(double *y, long nv, int p, int tcut, const int2 *cinfo,
                             const double *frames, hipStream_t st) {
  const int nc = p * (p + 2);
  if (4 * nc != nin_) return VES3D_INVALID_PARAMETER;
  V3D_CHECK(ensure_batch(nv));
  k_row_norms<<<(unsigned)nv, 256, 0, st>>>(y, nv, nc, cinfo, scale_);
  V3D_CHECK(launch_status());
  if (act_ == 1) {
    k_gather_rows<<<gb(nv * nin_), 256, 0, st>>>(y, nv, nc, cinfo, scale_, frames, Zh_);
    V3D_CHECK(launch_status());
    V3D_CHECK(odd_forward_bf16(nv, Y_, st));
  } else {
    k_gather_rows<<<gb(nv * nin_), 256, 0, st>>>(y, nv, nc, cinfo, scale_, frames, Zb_);
    V3D_CHECK(launch_status());
    V3D_CHECK(odd_forward(Zb_, nv, Y_, st));
  }
  k_scatter_add<<<gb(nv * nin_), 256, 0, st>>>(Y_, nv, nc, p, tcut, cinfo, scale_, frames,
                                                y);
  return launch_status();
}

// The odd part on the rows of Zh_.  The first layer's product changes sign
// with its input, so it serves both signs; the hidden layers run on 2 B rows
// (z's, then -z's), and the last product forms half the difference.
int LearnedPC::odd_forward_bf16(long B, float *Y, hipStream_t st) {
  V3D_CHECK(refresh_bf16(st));
  const int w = width_, n = nin_;
  GemmEpi e;
  e.bias = P_ + ob1_;
  e.H = H1h_;
  V3D_CHECK(gemm_bf16<kOutGeluOdd>(B, w, n, Zh_, n, W1h(), n, e, st));
  e.bias = P_ + ob2_;
  e.H = H2h_;
  V3D_CHECK(gemm_bf16<kOutGelu>(2 * B, w, w, H1h_, w, W2h(), w, e, st));
  GemmEpi y;
  y.bias = P_ + ob3_;
  y.C = Y;
  return gemm_bf16<kOutOdd>(B, n, w, H2h_, w, W3h(), w, y, st);
}

int LearnedPC::odd_forward(const float *Z, long B, float *Y, hipStream_t st) {
  V3D_CHECK(ensure_batch(B));
  if (act_ == 1) {
    const ToBf16 a{Z, Zh_, nullptr, (int)B, nin_, 0};
    k_to_bf16<<<cdiv(B, 32) * cdiv(nin_, 32), 256, 0, st>>>(a, a, a);
    V3D_CHECK(launch_status());
    return odd_forward_bf16(B, Y, st);
  }
  const long n = B * nin_;
  V3D_CHECK(forward(Z, B, Y, st));
  k_negate<<<gb(n), 256, 0, st>>>(Z, n, Zneg_);
  V3D_CHECK(launch_status());
  V3D_CHECK(forward(Zneg_, B, Yneg_, st));
  k_odd_part<<<gb(n), 256, 0, st>>>(Y, Yneg_, n);
  return launch_status();
}

int LearnedPC::record(const double *Dr, const double *e, long nv, int p, const int2 *cinfo,
                      const double *frames, hipStream_t st) {
  const int nc = p * (p + 2);
  if (4 * nc != nin_ || cap_ < nv) return VES3D_INVALID_PARAMETER;
  V3D_CHECK(ensure_batch(nv));
  k_row_norms<<<(unsigned)nv, 256, 0, st>>>(Dr, nv, nc, cinfo, scale_);
  V3D_CHECK(launch_status());
  k_record<<<gb(nv * nin_), 256, 0, st>>>(Dr, e, nv, nc, cinfo, scale_, frames, head_, cap_,
                                           Zs_, Ts_);
  V3D_CHECK(launch_status());
  head_ = (head_ + nv) % cap_;
  count_ += nv;
  return VES3D_SUCCESS;
}

}  // namespace v3d
