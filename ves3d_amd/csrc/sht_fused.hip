// sht_fused.hip -- the spherical-harmonic transforms in one kernel each.
//
// As grouped GEMMs (sht.hip) a transform is two launches with the Legendre
// sums of every (function, latitude, frequency) in memory between them, and
// each skinny product pays a launch.  Here a workgroup takes FG functions
// through both stages with that intermediate in LDS:
//   synthesis: Legendre sums (VALU, a table entry serves FG functions), then
//     the Fourier sums on MFMA (16 rows of (function, latitude) by 16
//     longitudes);
//   analysis: the Fourier sums of the grid rows on MFMA, then the Legendre
//     sums.
// Orders 16 and 32 in FP64, here / as GEMMs in us (back to back): N = 6 functions
// synthesis 7.9 / 11.9, of three variants 8.7 / 30, analysis 8.4 / 11.6; N =
// 1536: 15 / 25, 30 / 61, 16 / 23; N = 6144: 35 / 56, 93 / 150, 54 / 55.
// Longitudes lon and lon + p lie pi apart, where the Fourier functions of
// order m differ by (-1)^m: the frequencies are kept as an even-order half E
// and an odd-order half O (p of each), a synthesis writes E + O and E - O, an
// analysis reads the sums and differences of the two half circles, and the
// products shrink by half.
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "mfma.hpp"
#include "sht.hpp"

namespace v3d {

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr size_t kLdsMost = 64 * 1024;  // two workgroups per CU
// Orders of the contracted side up to 32: at 33 to 48 a handful of functions is
// faster in one kernel (2 at order 48: 10.6 us, 16.7 as GEMMs), many are slower
// (6144: 196, 122 us), and more instances would have to be kept for the few.
constexpr int kMaxSteps = 8;
constexpr int kBatch = 8;               // table values a thread has in flight

__host__ __device__ __forceinline__ int up16(int v) { return (v + 15) & ~15; }

// Frequency block j holds order m = (j + 1) / 2, cosine for odd j and j = 0.
// Its place within the half of its parity:
__device__ __forceinline__ int half_place(int j) {
  const int m = (j + 1) / 2;
  return j == 0 ? 0 : m - 1 + (j & 1 ? 0 : 1);
}
// and the block at place e of the even (odd = 0) or odd half.
__host__ __device__ __forceinline__ int half_block(int odd, int e) {
  if (odd) return 2 * (e | 1) - 1 + (e & 1);
  return e == 0 ? 0 : 2 * ((e + 1) & ~1) - 1 + ((e - 1) & 1);
}
// Offset of block j's coefficients, and of order m's Legendre block with L
// columns per degree.
__device__ __forceinline__ int block_off(int p, int j) {
  if (j == 0) return 0;
  const int m = (j + 1) / 2;
  return (p + 1) * (2 * m - 1) - m * (m - 1) + (j & 1 ? 0 : p + 1 - m);
}
__device__ __forceinline__ int legendre_off(int p, int m, int L) {
  return L * (m * (p + 1) - m * (m - 1) / 2);
}

// The Fourier functions on half a circle in MFMA operand order: for every 16
// columns and half (even, odd), KS loads of 64 values, entry 4 s + lane / 16
// of column lane % 16 (zero past the orders).  A wave keeps its 16 columns in
// registers.
template <typename T, int KS>
struct Operand {
  T e[KS], o[KS];
  __device__ __forceinline__ void load(const T *__restrict__ frag, int c, int lane) {
    const T *f = frag + (long)c * 2 * KS * 64 + lane;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      e[s] = f[64 * s];
      o[s] = f[64 * (KS + s)];
    }
  }
};
// One 16 x 16 tile of E and of O from the row's two halves at a.
template <typename T, int KS>
__device__ __forceinline__ void tile_sums(const T *__restrict__ a, const Operand<T, KS> &f,
                                          typename Mfma<T>::v4 &E, typename Mfma<T>::v4 &O) {
  E = O = typename Mfma<T>::v4{T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    E = Mfma<T>::step(a[4 * s], f.e[s], E);
    O = Mfma<T>::step(a[4 * KS + 4 * s], f.o[s], O);
  }
}
// The columns and row tiles of a wave: with at most kWaves column tiles the
// waves share each column's rows, else a wave takes every kWaves-th column.
struct WaveTiles {
  int c, c_step, r, r_step;
};
__device__ __forceinline__ WaveTiles wave_tiles(int wave, int ct) {
  const int groups = max(1, kWaves / ct);
  if (ct > kWaves) return {wave, kWaves, 0, 1};
  if (wave >= groups * ct) return {ct, 1, 0, 1};  // nothing
  return {wave % ct, ct, wave / ct, groups};
}

template <typename T>
struct SynthArgs {
  const T *S;
  long N;
  int p0, p1;
  T alpha;
  const T *leg;
  int kind[kMaxSynth];
  const T *frag[kMaxSynth];
  T *X[kMaxSynth];
};

size_t synth_lds(int p0, int p1, int fg, size_t es) {
  const size_t K = up16(p0 * 2) / 2, L = p1 + 1;
  return es * (fg * L * (2 * K + 1) + (size_t)fg * sh_ncoef(p0));
}
size_t analysis_lds(int p0, int p1, int fg, size_t es) {
  const size_t K = up16(p0 * 2) / 2, L = p0 + 1;
  return es * (fg * L * (2 * K + 1) + fg * L * (2 * p1 + 1)) + sizeof(short) * sh_ncoef(p1);
}

// Latency-bound with few functions (one workgroup per function and variant),
// else by the writes (2112 per function and variant at order 32: 93 us for 6144
// functions and three variants are 3.4 TB/s).  A thread takes a latitude and its
// mirror together, whose sums share the products of the even and the odd
// degrees, and has kBatch table values in flight, past an order's last degree
// as zeros: one latitude per thread, with the last few values one by one, took
// 7.3 instead of 6.0 us for 6 functions at order 24, 106 instead of 93 us there.
// (The analysis gains nothing from either: its sums are bound by the LDS reads,
// which stay, 50 -> 60 us.)
template <typename T, int FG, int KS>
__global__ __launch_bounds__(kThreads) void k_synth(const SynthArgs<T> a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int K = 4 * KS, ldr = 2 * K + 1;
  const int p0 = a.p0, p1 = a.p1, L = p1 + 1, nc = p0 * (p0 + 2), R = FG * L;
  T *B = (T *)lds;      // [R][ldr] Legendre sums, even half then odd half
  T *C = B + R * ldr;   // [nc][FG] coefficients
  const int var = blockIdx.y, tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int ct = up16(p1) / 16;
  WaveTiles w = wave_tiles(tid >> 6, ct);
  Operand<T, KS> F;
  if (w.c < ct) F.load(a.frag[var], w.c, lane);
  const long f0 = (long)blockIdx.x * FG;
  const T *__restrict__ leg = a.leg;
  const int kind = a.kind[var];
#pragma unroll
  for (int f = 0; f < FG; ++f)
    for (int c = tid; c < nc; c += kThreads)
      C[c * FG + f] = f0 + f < a.N ? a.S[(f0 + f) * nc + c] : T(0);
  if (K > p0) {
    const int pad = K - p0;
    for (int i = tid; i < R * pad; i += kThreads) {
      T *b = B + (i / pad) * ldr + p0 + i % pad;
      b[0] = b[K] = T(0);
    }
  }
  __syncthreads();
  // a table value and its mirror latitude's differ by (-1)^(n - m) (the first
  // derivatives' by the opposite sign)
  const int Lh = (L + 1) / 2;
  const T mirror = kind == 1 || kind == 2 ? T(-1) : T(1);
  for (int i = tid; i < 2 * p0 * Lh; i += kThreads) {
    const int j = i / Lh, l = i % Lh, m = (j + 1) / 2, len = p0 + 1 - m;
    // an order's blocks of the four derivative kinds follow each other
    const T *__restrict__ t = leg + 4 * legendre_off(p0, m, L) + kind * len * L + l;
    const T *c = C + block_off(p0, j) * FG;
    T se[FG] = {}, so[FG] = {};
    for (int n0 = 0; n0 < len; n0 += kBatch) {
      T x[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) x[u] = t[min(n0 + u, len - 1) * L];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const T v = n0 + u < len ? x[u] : T(0);
        const T *cu = c + min(n0 + u, len - 1) * FG;
#pragma unroll
        for (int f = 0; f < FG; ++f) {
          if (u & 1)
            so[f] = fma(v, cu[f], so[f]);
          else
            se[f] = fma(v, cu[f], se[f]);
        }
      }
    }
    const int place = (m & 1 ? K : 0) + half_place(j), lm = L - 1 - l;
#pragma unroll
    for (int f = 0; f < FG; ++f) {
      B[(f * L + l) * ldr + place] = a.alpha * (se[f] + so[f]);
      if (lm != l) B[(f * L + lm) * ldr + place] = a.alpha * (mirror * (se[f] - so[f]));
    }
  }
  __syncthreads();
  const long rows = (a.N - f0) * L;  // rows left from this workgroup on
  T *__restrict__ X = a.X[var] + f0 * L * 2 * p1;
  for (int c = w.c; c < ct;) {
    const int col = 16 * c + li;
    for (int r0 = 16 * w.r; r0 < R; r0 += 16 * w.r_step) {
      typename Mfma<T>::v4 E, O;
      tile_sums<T, KS>(B + min(r0 + li, R - 1) * ldr + lk, F, E, O);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = r0 + Mfma<T>::row(lk, r);
        if (row < R && row < rows && col < p1) {
          X[(long)row * 2 * p1 + col] = E[r] + O[r];
          X[(long)row * 2 * p1 + p1 + col] = E[r] - O[r];
        }
      }
    }
    c += w.c_step;
    if (c < ct) F.load(a.frag[var], c, lane);
  }
}

// leg: per order m the block [latitude][degree].
template <typename T>
struct AnalysisArgs {
  const T *X;
  long N;
  int p0, p1;
  const T *frag, *leg;
  T *S;
};

template <typename T, int FG, int KS>
__global__ __launch_bounds__(kThreads) void k_analysis(const AnalysisArgs<T> a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int K = 4 * KS, ldr = 2 * K + 1;
  const int p0 = a.p0, p1 = a.p1, L = p0 + 1, nc = p1 * (p1 + 2);
  const int R = FG * L, ldg = 2 * p1 + 1;
  T *P = (T *)lds;                     // [R][ldr] sums then differences of the half circles
  T *G = P + R * ldr;                  // [R][ldg] Fourier sums, even half then odd half
  short *J = (short *)(G + R * ldg);   // coefficient -> block
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int ct = up16(p1) / 16;
  WaveTiles w = wave_tiles(tid >> 6, ct);
  Operand<T, KS> F;
  if (w.c < ct) F.load(a.frag, w.c, lane);
  const long f0 = (long)blockIdx.x * FG;
  const long rows = (a.N - f0) * L;
  const T *__restrict__ X = a.X + f0 * L * 2 * p0;
#pragma unroll 4
  for (int i = tid; i < R * K; i += kThreads) {
    const int row = i / K, lon = i % K;
    const bool in = lon < p0 && row < rows;
    const T x = in ? X[(long)row * 2 * p0 + lon] : T(0);
    const T y = in ? X[(long)row * 2 * p0 + p0 + lon] : T(0);
    P[row * ldr + lon] = x + y;
    P[row * ldr + K + lon] = x - y;
  }
  for (int j = tid; j < 2 * p1; j += kThreads) {
    const int o = block_off(p1, j);
    for (int n = 0; n <= p1 - (j + 1) / 2; ++n) J[o + n] = (short)j;
  }
  __syncthreads();
  for (int c = w.c; c < ct;) {
    const int col = 16 * c + li;
    for (int r0 = 16 * w.r; r0 < R; r0 += 16 * w.r_step) {
      typename Mfma<T>::v4 E, O;
      tile_sums<T, KS>(P + min(r0 + li, R - 1) * ldr + lk, F, E, O);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = r0 + Mfma<T>::row(lk, r);
        if (row < R && col < p1) {
          G[row * ldg + col] = E[r];
          G[row * ldg + p1 + col] = O[r];
        }
      }
    }
    c += w.c_step;
    if (c < ct) F.load(a.frag, c, lane);
  }
  __syncthreads();
  for (int c = tid; c < nc; c += kThreads) {
    const int j = J[c], m = (j + 1) / 2, n = c - block_off(p1, j);
    const int ls = p1 + 1 - m;
    const T *__restrict__ t = a.leg + legendre_off(p1, m, L) + n;
    const T *g = G + (m & 1 ? p1 : 0) + half_place(j);
    T s[FG] = {};
#pragma unroll 8
    for (int l = 0; l < L; ++l) {
      const T x = t[l * ls];
#pragma unroll
      for (int f = 0; f < FG; ++f) s[f] = fma(x, g[(f * L + l) * ldg], s[f]);
    }
#pragma unroll
    for (int f = 0; f < FG; ++f)
      if (f0 + f < a.N) a.S[(f0 + f) * nc + c] = s[f];
  }
}

// Operand tables, built once per (device, orders, kind): kinds 0, 1, 2 the
// longitude derivatives of MatFourier (synthesis), 3 MatFourierInv, 4 the
// transpose of MatFourier(p1, p0); kind 5 the transposed MatLegendre(p1, p0) by
// latitude, so that consecutive lanes (degrees) read consecutive words.
struct FragTable {
  double *d64 = nullptr;
  float *d32 = nullptr;
};
std::mutex g_frag_mu;
std::map<std::tuple<int, int, int, int>, FragTable> g_frags;

template <typename T>
const T *frag_ptr(const FragTable &t);
template <>
const double *frag_ptr<double>(const FragTable &t) { return t.d64; }
template <>
const float *frag_ptr<float>(const FragTable &t) { return t.d32; }

// Under g_frag_mu.
template <typename T>
const T *frag_upload(const std::tuple<int, int, int, int> &key, const std::vector<double> &f) {
  std::vector<float> f32(f.begin(), f.end());
  FragTable t;
  if (hipMalloc(&t.d64, sizeof(double) * f.size()) != hipSuccess) return nullptr;
  if (hipMalloc(&t.d32, sizeof(float) * f.size()) != hipSuccess ||
      hipMemcpy(t.d64, f.data(), sizeof(double) * f.size(), hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipMemcpy(t.d32, f32.data(), sizeof(float) * f.size(), hipMemcpyHostToDevice) !=
          hipSuccess) {
    (void)hipFree(t.d64);
    (void)hipFree(t.d32);
    return nullptr;
  }
  return frag_ptr<T>(g_frags[key] = t);
}

template <typename T>
const T *frag_table(int p0, int p1, int kind, const ShMatsHost &h) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_frag_mu);
  const auto key = std::make_tuple(dev, p0, p1, kind);
  auto it = g_frags.find(key);
  if (it != g_frags.end()) return frag_ptr<T>(it->second);
  std::vector<double> f;
  if (kind == 5) {
    for (int m = 0; m <= p1; ++m)
      for (int lat = 0; lat <= p0; ++lat)
        for (int n = 0; n <= p1 - m; ++n) f.push_back(h.data[h.MlT[m] + (long)n * (p0 + 1) + lat]);
    return frag_upload<T>(key, f);
  }
  // element (k, col) of a half: synthesis: order place k at longitude col,
  // analysis: longitude k of order place col
  const int KS = up16(2 * p0) / 8, ct = up16(p1) / 16;
  const double *M = &h.data[kind == 0   ? h.Mf
                            : kind == 1 ? h.Mdf
                            : kind == 2 ? h.Md2f
                            : kind == 3 ? h.Mfinv
                                        : h.MfT];
  f.assign((size_t)ct * 2 * KS * 64, 0.0);
  for (int c = 0; c < ct; ++c)
    for (int odd = 0; odd < 2; ++odd)
      for (int s = 0; s < KS; ++s)
        for (int lane = 0; lane < 64; ++lane) {
          const int k = 4 * s + lane / 16, col = 16 * c + lane % 16;
          if (k >= p0 || col >= p1) continue;
          f[((size_t)(c * 2 + odd) * KS + s) * 64 + lane] =
              kind < 3    ? M[(long)half_block(odd, k) * 2 * p1 + col]
              : kind == 3 ? M[(long)k * 2 * p1 + half_block(odd, col)]
                          : M[(long)half_block(odd, col) * 2 * p0 + k];
        }
  return frag_upload<T>(key, f);
}

// Whether n values at a and k values at b share memory.  A workgroup writes its
// functions over others that no workgroup has read yet; the GEMMs read all of
// their input into the work buffer before they write.
template <typename T>
bool overlap(const T *a, long n, const T *b, long k) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return x < y + sizeof(T) * k && y < x + sizeof(T) * n;
}

// Functions per workgroup: as many as share the tables without leaving CUs
// idle (0: the GEMMs run).
int functions_per_group(long N, int nvar, size_t (*lds)(int, int, int, size_t), int p0, int p1,
                        size_t es) {
  if (!gemm_is_default() || p0 > 4 * kMaxSteps || N >= (1L << 31)) return 0;
  for (int fg : {4, 2, 1}) {
    if (lds(p0, p1, fg, es) > kLdsMost) continue;
    if (fg == 1 || (N + fg - 1) / fg * nvar >= 512) return fg;
  }
  return 0;
}

template <typename T, int FG, int KS>
int launch(const SynthArgs<T> &a, int nvar, hipStream_t st) {
  k_synth<T, FG, KS><<<dim3(cdiv(a.N, FG), nvar), kThreads,
                       synth_lds(a.p0, a.p1, FG, sizeof(T)), st>>>(a);
  return launch_status();
}
template <typename T, int FG, int KS>
int launch(const AnalysisArgs<T> &a, int, hipStream_t st) {
  k_analysis<T, FG, KS><<<cdiv(a.N, FG), kThreads, analysis_lds(a.p0, a.p1, FG, sizeof(T)), st>>>(
      a);
  return launch_status();
}
template <typename T, int FG, typename A>
int launch_steps(const A &a, int nvar, hipStream_t st) {
  switch ((a.p0 + 7) / 8) {
    case 1: return launch<T, FG, 2>(a, nvar, st);
    case 2: return launch<T, FG, 4>(a, nvar, st);
    case 3: return launch<T, FG, 6>(a, nvar, st);
    default: return launch<T, FG, 8>(a, nvar, st);
  }
}
template <typename T, typename A>
int launch_groups(const A &a, int fg, int nvar, hipStream_t st) {
  return fg == 4   ? launch_steps<T, 4>(a, nvar, st)
         : fg == 2 ? launch_steps<T, 2>(a, nvar, st)
                   : launch_steps<T, 1>(a, nvar, st);
}

}  // namespace

namespace {

constexpr long kAlways = 1L << 60;

// The number of functions from which the GEMMs synthesise nvar variants of order
// p0 on the grid of p1.  A workgroup of 512 threads takes at most four functions,
// which is little work on a small grid, and forms the Legendre sums of every
// variant; the GEMMs share the tables over 64 functions and, of a value and its
// longitude derivative (nvar = 2), the sums.  Drawn from orders 1 to 32 with 512
// to 131072 functions; here / as GEMMs in us:
//  - FP64, three variants: orders 6 -> 6, N = 3072 / 4608: 17 / 21, 24 / 22; 6 ->
//    12, 6144 / 12288: 34 / 39, 71 / 57; 12 -> 12, 8192 / 16384: 59 / 59, 120 / 89;
//    16 -> 16, 12288: 110 / 110; one variant, 6 -> 6, 6144 / 8192: 11 / 11, 15 / 12
//  - order above 24 (two functions or one fit the LDS): 30 -> 20, 1536 / 3072: 43 /
//    56, 88 / 80; 32 -> 32, 3072 / 12288: 121 / 142, 569 / 473; one variant, 30 ->
//    30, 12288 / 16384: 152 / 163, 226 / 204
//  - the value and its longitude derivative: 12 -> 12, 6144 / 8192: 30 / 31, 40 / 34
//  - FP32, three variants: 6 -> 6, 4608 / 8192: 17 / 22, 28 / 23; 24 -> 12, 6144 /
//    8192: 50 / 55, 68 / 63; 32 -> 32, 16384 / 24000: 309 / 348, 575 / 514
template <typename T>
long synth_line(int p0, int p1, int nvar) {
  if (sizeof(T) == 8) {
    if (p0 > 24) return p1 < p0 ? 2048 : (nvar == 1 ? 12288 : 3072);
    if (p0 >= 20 && p1 < p0) return nvar == 2 ? 4096 : 6144;
    if (p1 >= 28) return p1 >= 36 && nvar > 1 ? 12288 : kAlways;
    if (p1 <= 8) return nvar == 1 ? 6144 : 4096;
    return p1 < 12 || (p1 == 12 && nvar == 2) ? 6144 : 12288;
  }
  if (p0 >= 20 && (p1 < p0 || (nvar == 2 && p1 == p0 && p0 <= 24))) return 6144;
  if (p0 > 24) return 20480;
  return p1 < 12 ? 6144 : (p1 < 28 ? 12288 : kAlways);
}

// The same for the analysis of grids of p0 to order p1.  Here / as GEMMs in us:
//  - small grids, FP64: 3 -> 3, N = 8192 / 12288: 9 / 11, 13 / 11; 6 -> 6, 24000 /
//    32768: 25 / 25, 34 / 26; 8 -> 8, 65536: 75 / 60; FP32: 3 -> 3, 12288 / 16384: 10
//    / 12, 13 / 12; 12 -> 12, 65536: 85 / 73; but FP64 8 -> 16, 65536: 94 / 126
//  - half the order, few results per function: FP64 8 -> 4, 12288: 14 / 14, 32 -> 16,
//    16384: 159 / 128; FP32 16 -> 8, 16384 / 32768: 25 / 25, 46 / 42
//  - both orders above 24, FP64, where one function (order 32) or two fit the LDS:
//    32 -> 32, 1024 / 1536: 29 / 33, 42 / 38; 28 -> 28, 4608 / 6144: 61 / 64, 80 / 75;
//    FP32, 32 -> 32, 16384 / 24000: 140 / 137, 230 / 202
//  - FP64 from order 20 on: 24 -> 24, 24000 / 32768: 214 / 210, 290 / 261
template <typename T>
long analysis_line(int p0, int p1) {
  const bool f64 = sizeof(T) == 8;
  long line = kAlways;
  if (p0 > 24 && p1 > 24)
    line = f64 ? (analysis_lds(p0, p1, 2, sizeof(T)) > kLdsMost ? 1280 : 5120) : 20480;
  else if (f64 && p0 >= 20)
    line = 24576;
  if (2 * p1 <= p0 && (f64 || p0 <= 20)) line = std::min(line, f64 ? 12288L : 16384L);
  if (p0 <= 4)
    line = std::min(line, f64 ? 10240L : 12288L);
  else if (p0 <= 6 || (p0 <= 12 && p1 <= p0))
    line = std::min(line, 24576L);
  return line;
}

}  // namespace

template <typename T>
bool synth_fused(const T *S, long N, int p0, int p1, int nvar, const ShMatsHost &h, const T *mats,
                 const int *dleg, const int *dfour, T *const *X, T alpha, hipStream_t st,
                 int *status) {
  if (N >= synth_line<T>(p0, p1, nvar)) return false;
  const int fg = functions_per_group(N, nvar, synth_lds, p0, p1, sizeof(T));
  if (fg == 0) return false;
  for (int v = 0; v < nvar; ++v)
    if (overlap(S, N * sh_ncoef(p0), X[v], N * sh_ngrid(p1))) return false;
  SynthArgs<T> a{};
  a.S = S;
  a.N = N;
  a.p0 = p0;
  a.p1 = p1;
  a.alpha = alpha;
  a.leg = mats + h.Ml[0];
  for (int v = 0; v < nvar; ++v) {
    a.kind[v] = dleg[v];
    a.frag[v] = frag_table<T>(p0, p1, dfour[v], h);
    a.X[v] = X[v];
    if (!a.frag[v]) {
      *status = VES3D_MEMORY_ERROR;
      return true;
    }
  }
  *status = launch_groups<T>(a, fg, nvar, st);
  return true;
}

template <typename T>
bool analysis_fused(const T *X, long N, int p0, int p1, bool transpose, const ShMatsHost &h,
                    const T *mats, T *S, hipStream_t st, int *status) {
  if (N >= analysis_line<T>(p0, p1)) return false;
  const int fg = functions_per_group(N, 1, analysis_lds, p0, p1, sizeof(T));
  if (fg == 0 || overlap(X, N * sh_ngrid(p0), S, N * sh_ncoef(p1))) return false;
  const T *frag = frag_table<T>(p0, p1, transpose ? 4 : 3, h);
  const T *leg = transpose ? frag_table<T>(p0, p1, 5, h) : mats + h.Mlinv[0];
  if (!frag || !leg) {
    *status = VES3D_MEMORY_ERROR;
    return true;
  }
  const AnalysisArgs<T> a{X, N, p0, p1, frag, leg, S};
  *status = launch_groups<T>(a, fg, 1, st);
  return true;
}

#define V3D_INST(T)                                                                       \
  template bool synth_fused<T>(const T *, long, int, int, int, const ShMatsHost &,        \
                               const T *, const int *, const int *, T *const *, T,        \
                               hipStream_t, int *);                                       \
  template bool analysis_fused<T>(const T *, long, int, int, bool, const ShMatsHost &,    \
                                  const T *, T *, hipStream_t, int *);
V3D_INST(double)
V3D_INST(float)
#undef V3D_INST

}  // namespace v3d
