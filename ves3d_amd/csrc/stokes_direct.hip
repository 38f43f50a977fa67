// stokes_direct.hip -- direct Stokes single/double-layer sums on gfx950.
//
// Two kernel families:
//
//  1. k_pairs_* and k_far_groups_*: the all-pairs / far-field sum that stands
//     in for the FMM (StokesAlltoAll, src/CPUKernels.cc:966-1054, and the
//     PVFMM pair kernels src/PVFMMInterface.cc:161-238, :284-369).  One target
//     per lane, 256 targets per workgroup.  Every lane of a wave meets the
//     same source at the same time, so the sources are read with uniform
//     addresses (s_load into SGPRs, which the VALU takes as operands): no LDS
//     staging, no barriers.  The source range is cut into `nsplit` slices of
//     whole groups or, where a slice per group would leave the chip idle, of
//     parts of groups; the slice index is the fastest-varying part of the
//     block index, so with nsplit a multiple of 8 every XCD (blocks are dealt
//     round-robin over the 8 XCDs) streams only its own slices of sources
//     through its L2.  Each slice writes an FP64 partial, and k_sum_slices
//     adds the partials in a fixed order (deterministic, no atomics).
//     The FP64 kernels read the caller's arrays as they lie.  The FP32
//     ("f32c") form packs each source relative to an FP64 anchor near it and
//     shifts the lane's target by the same anchor in FP64 before rounding, so
//     coordinate differences keep FP32 relative accuracy independent of the
//     box size; pair terms are summed in FP32 over 64 sources and merged into
//     an FP32 (hi, lo) TwoSum pair.  Few sources, and most single layers, take
//     the same FP32 terms from LDS tiles (k_tiles_f32c).
//
//  2. k_vesicle_*: the per-vesicle Device<>::DirectStokes /
//     DirectStokesDoubleLayer sums (src/CPUKernels.cc:8-118, :1059-1136) on
//     AxisMajor [ves][xyz][stride] data: 64 targets of one vesicle per
//     workgroup, its sources split over the workgroup's waves and read through
//     the scalar cache, or staged through LDS by one wave where they are few or
//     come from memory.
#include <algorithm>
#include <atomic>
#include <type_traits>
#include "common.hpp"
#include "implicit.hpp"
#include "runtime.hpp"

namespace v3d {

constexpr int FF_BLOCK = 256;
constexpr int FF_TILE = 256;  // sources that share an anchor in k_pairs_f32c
constexpr int FF_SUB = 64;    // FP32 form: TwoSum merge period (sources)
constexpr int FF_PART = 32;   // fewest sources of a part of a group

// 1/sqrt(x) for x > 0: the hardware estimate (v_rsq_f64, about 2^-20
// relative) refined by one third-order step y (1 + e/2 + 3e^2/8),
// e = 1 - x y^2, which leaves a rounding-level error.  x = 0 gives NaN here
// (callers select it away); no special-value fix-ups in the pair loop.
__device__ __forceinline__ double rsqrt_pair(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(y * -x, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}
__device__ __forceinline__ float rsqrt_pair(float x) { return __frsqrt_rn(x); }

// The r^2 bias that removes a target's own group from a sum without making
// control flow divergent.  FP32: 1/sqrt(inf) = 0 and every term is an exact
// zero.  FP64: infinity would turn the refinement step into a NaN; with 1e200
// an own-group source adds 1e-100 |f|, nothing at 53 bits.  Both hold for finite
// densities; the public sums (k_pairs_*), whose groups may hold anything, also
// take a lane's sums from before its own group, and the bias keeps its
// coincident points from repeating runs.
constexpr double kOwnGroupBias64 = 1e200;
constexpr float kOwnGroupBias = __builtin_inff();

// Slices over parts of groups: unit u = (group u / nsub, part u % nsub), and
// slice k holds units k per .. (k + 1) per - 1 (the last slice what is left).
// share (1 or 4): waves of a workgroup that take the same targets, each a
// slice of its own, and add their sums in LDS.
struct SliceMap {
  unsigned units, per, nsub, share;
};
struct Slice {
  unsigned u, u1;  // units
  unsigned g, j;   // group and part of unit u
};
__device__ __forceinline__ Slice slice_of(const SliceMap &m, unsigned block_slice) {
  const unsigned wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned k = m.share == 1 ? block_slice : block_slice * m.share + wv;
  Slice s;
  s.u = min(k * m.per, m.units);
  s.u1 = min(s.u + m.per, m.units);
  s.g = s.u / m.nsub;
  s.j = s.u % m.nsub;
  return s;
}
// a / b with the short 32-bit division wherever the operands allow it
__device__ __forceinline__ long quot(long a, long b) {
  return ((a | b) >> 32) ? a / b : (long)((unsigned)a / (unsigned)b);
}

// The targets of a wave: 64 consecutive ones, one per lane.  A lane past the
// last target computes for the last one and stores nothing, so that control
// flow inside the source loops stays uniform.
struct WaveTargets {
  long row;    // wave index over the targets
  bool live;   // the wave has a target
  long t, tc;  // the lane's target, clamped to the last one
  long group;  // the lane's group (grouped sums)
  long own;    // the group that holds all the wave's targets, or -1
};
__device__ __forceinline__ WaveTargets wave_targets(long tb, unsigned share, long n_trg, long tpg) {
  const long wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  WaveTargets w;
  w.row = share == 1 ? tb * (FF_BLOCK / 64) + wv : tb;
  const long first = w.row * 64, last = min(first + 64, n_trg) - 1;
  w.live = first < n_trg;
  w.t = first + (threadIdx.x & 63);
  w.tc = min(w.t, n_trg - 1);
  w.group = w.own = -1;
  if (tpg > 0 && w.live) {
    const long gf = quot(first, tpg);
    w.own = gf == quot(last, tpg) ? gf : -1;
    w.group = w.own >= 0 ? gf : quot(w.tc, tpg);
  }
  return w;
}

// Writes the wave's sums (N per target) to o[N t ..]: where the workgroup's
// waves share their targets, those of all four added in wave order.
template <int N>
__device__ __forceinline__ void store_sums(const WaveTargets &w, unsigned share, long n_trg,
                                           const double (&v)[N], double *__restrict__ o) {
  double s[N];
#pragma unroll
  for (int c = 0; c < N; ++c) s[c] = v[c];
  if (share > 1) {
    __shared__ double red[FF_BLOCK / 64 - 1][N][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (wv > 0) {
#pragma unroll
      for (int c = 0; c < N; ++c) red[wv - 1][c][lane] = s[c];
    }
    __syncthreads();
    if (wv > 0) return;
#pragma unroll
    for (int k = 0; k < FF_BLOCK / 64 - 1; ++k)
#pragma unroll
      for (int c = 0; c < N; ++c) s[c] += red[k][c][lane];
  }
  if (w.t < n_trg) {
#pragma unroll
    for (int c = 0; c < N; ++c) o[3 * w.t + c] = s[c];
  }
}

// One pair's contribution: f / r + (f.d) d / r^3 and k (n.d)(g.d) d / r^5,
// with ri = 1 / r, f at `f`, (g, n) at `q`.  With both layers the terms along
// d share one coefficient.
template <bool SL, bool DL, typename T>
__device__ __forceinline__ void add_pair(T dx, T dy, T dz, T ri, const T *__restrict__ f,
                                         const T *__restrict__ q, T k, T (&S)[3]) {
  const T ri2 = ri * ri;
  if constexpr (!DL) {
    const T ip = (f[0] * dx + f[1] * dy + f[2] * dz) * ri2;
    S[0] = fma(ri, fma(dx, ip, f[0]), S[0]);
    S[1] = fma(ri, fma(dy, ip, f[1]), S[1]);
    S[2] = fma(ri, fma(dz, ip, f[2]), S[2]);
  } else {
    const T t = (q[3] * dx + q[4] * dy + q[5] * dz) * (q[0] * dx + q[1] * dy + q[2] * dz) * ri2;
    if constexpr (SL) {
      const T w = fma(k, t, f[0] * dx + f[1] * dy + f[2] * dz) * (ri * ri2);
      S[0] = fma(dx, w, fma(ri, f[0], S[0]));
      S[1] = fma(dy, w, fma(ri, f[1], S[1]));
      S[2] = fma(dz, w, fma(ri, f[2], S[2]));
    } else {
      const T w = t * (ri * ri2);
      S[0] = fma(dx, w, S[0]);
      S[1] = fma(dy, w, S[1]);
      S[2] = fma(dz, w, S[2]);
    }
  }
}

// r^2 >= 0 ordered as an unsigned integer (FP64: by its high word).
__device__ __forceinline__ unsigned order_key(double x) { return (unsigned)__double2hiint(x); }
__device__ __forceinline__ unsigned order_key(float x) { return __float_as_uint(x); }

// GUARD: pairs with r^2 <= eps2 contribute nothing.  Such pairs are rare (a
// point meeting itself), so runs of FF_RUN sources are summed without a test
// while the smallest r^2 is kept (half an integer instruction per pair); a
// wave that met one repeats the run with a selection per pair.
constexpr int FF_RUN = 32;

// n consecutive FP64 sources (positions p, densities f, (g, n) at q) at one
// target, U at a time.  A lane with a bias keeps its sums (spans: the wave has
// such lanes).
template <int U, bool SL, bool DL, bool GUARD>
__device__ __forceinline__ void add_sources64(double tx, double ty, double tz, double bias,
                                              bool spans, int n, const double *__restrict__ p,
                                              const double *__restrict__ f,
                                              const double *__restrict__ q, double k, double eps2,
                                              double (&S)[3]) {
  unsigned m = ~0u;
  auto block = [&](int i, auto uc, bool select) {
    constexpr int V = decltype(uc)::value;
    double dx[V], dy[V], dz[V], r2[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const double *__restrict__ x = p + (i + u) * 3;
      dx[u] = tx - x[0];
      dy[u] = ty - x[1];
      dz[u] = tz - x[2];
      r2[u] = fma(dz[u], dz[u], fma(dy[u], dy[u], fma(dx[u], dx[u], bias)));
    }
    if (GUARD && !select) {
#pragma unroll
      for (int u = 0; u < V; ++u) m = min(m, order_key(r2[u]));
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
      double ri = rsqrt_pair(r2[u]);
      if (GUARD && select) ri = r2[u] > eps2 ? ri : 0.0;
      add_pair<SL, DL>(dx[u], dy[u], dz[u], ri, f + (i + u) * 3, q + (i + u) * 6, k, S);
    }
  };
  using One = std::integral_constant<int, 1>;
  const int run = GUARD ? FF_RUN : n;
  for (int i0 = 0; i0 < n; i0 += run) {
    const int i1 = min(n, i0 + run);
    const double S0[3] = {S[0], S[1], S[2]};
    m = ~0u;
    int i = i0;
    for (; i + U <= i1; i += U) block(i, std::integral_constant<int, U>(), false);
    for (; i < i1; ++i) block(i, One(), false);
    if (GUARD && __any(m <= order_key(eps2))) {
#pragma unroll
      for (int c = 0; c < 3; ++c) S[c] = S0[c];
#pragma unroll 1
      for (i = i0; i < i1; ++i) block(i, One(), true);
    }
    if (spans) {
#pragma unroll
      for (int c = 0; c < 3; ++c) S[c] = bias != 0.0 ? S0[c] : S[c];
    }
  }
}

// One step of U pairs' arithmetic, kept together by the scheduler: a SIMD
// issues runs of one independent FP32 instruction faster than the same
// instructions pair by pair (18 instructions per single-layer pair: 62 against
// 71 cycles measured on registers alone, whatever file the operands are in).
template <int U, typename F>
__device__ __forceinline__ void stage(F f) {
#pragma unroll
  for (int u = 0; u < U; ++u) f(u);
  __builtin_amdgcn_sched_barrier(0);
}

// U consecutive FP32 records at one target (lx, ly, lz): NS single-layer
// densities, into S (and T), and with DL the double layer, into S:
// (x, y, z[, f[, h]][, g, n]).  KEY: m keeps the smallest r^2.
template <int U, int NS, bool DL, bool KEY>
__device__ __forceinline__ void add_block32(const float *__restrict__ rec, float lx, float ly,
                                            float lz, float bias, float k, float (&S)[3],
                                            float (&T)[3], unsigned &m) {
  constexpr int R = 3 + 3 * NS + (DL ? 6 : 0);
  static_assert(!DL || NS <= 1, "one density beside a double layer");
  float s[U * R];
#pragma unroll
  for (int i = 0; i < U * R; ++i) s[i] = rec[i];
  float d[U][3], ri[U], t[U];
  stage<U>([&](int u) { d[u][0] = lx - s[u * R]; });
  stage<U>([&](int u) { d[u][1] = ly - s[u * R + 1]; });
  stage<U>([&](int u) { d[u][2] = lz - s[u * R + 2]; });
  stage<U>([&](int u) { ri[u] = fmaf(d[u][0], d[u][0], bias); });
  stage<U>([&](int u) { ri[u] = fmaf(d[u][1], d[u][1], ri[u]); });
  stage<U>([&](int u) { ri[u] = fmaf(d[u][2], d[u][2], ri[u]); });
  if constexpr (KEY) stage<U>([&](int u) { m = min(m, order_key(ri[u])); });
  stage<U>([&](int u) { ri[u] = rsqrt_pair(ri[u]); });
  auto dot = [&](float (&o)[U], int c) {  // record entries c .. c + 2 times d
    stage<U>([&](int u) { o[u] = s[u * R + c] * d[u][0]; });
    stage<U>([&](int u) { o[u] = fmaf(s[u * R + c + 1], d[u][1], o[u]); });
    stage<U>([&](int u) { o[u] = fmaf(s[u * R + c + 2], d[u][2], o[u]); });
  };
  if constexpr (!DL) {
#pragma unroll
    for (int e = 0; e < NS; ++e) {
      const int c0 = 3 + 3 * e;
      float (&Z)[3] = e ? T : S;
      float a[U][3];
      dot(t, c0);
      stage<U>([&](int u) { t[u] *= ri[u]; });
      stage<U>([&](int u) { t[u] *= ri[u]; });
#pragma unroll
      for (int c = 0; c < 3; ++c)
        stage<U>([&](int u) { a[u][c] = fmaf(d[u][c], t[u], s[u * R + c0 + c]); });
      stage<U>([&](int u) {
#pragma unroll
        for (int c = 0; c < 3; ++c) Z[c] = fmaf(ri[u], a[u][c], Z[c]);
      });
    }
  } else {
    float w[U], q[U];
    dot(t, R - 3);
    dot(w, R - 6);
    stage<U>([&](int u) { q[u] = ri[u] * ri[u]; });
    stage<U>([&](int u) { t[u] *= w[u]; });
    stage<U>([&](int u) { t[u] *= q[u]; });
    stage<U>([&](int u) { q[u] *= ri[u]; });
    if constexpr (NS == 1) {
      dot(w, 3);
      stage<U>([&](int u) { t[u] = fmaf(k, t[u], w[u]); });
      stage<U>([&](int u) {
#pragma unroll
        for (int c = 0; c < 3; ++c) S[c] = fmaf(ri[u], s[u * R + 3 + c], S[c]);
      });
    }
    stage<U>([&](int u) { t[u] *= q[u]; });
    stage<U>([&](int u) {
#pragma unroll
      for (int c = 0; c < 3; ++c) S[c] = fmaf(d[u][c], t[u], S[c]);
    });
  }
}

// FP64 sums of n_groups groups of spg sources (ungrouped: one group, tpg = 0),
// part j of a group its sources j plen .. (j + 1) plen - 1.
// Bound: FP64 VALU issue, 23 instructions per single-layer pair, 33 with both
// layers (4.0-4.5 cycles each on a SIMD, 16 for v_rsq_f64).  Measured with
// both layers between 320 vesicles of 544 points (3.0e10 pairs): 32.9 ms;
// sources staged through LDS as 128-byte records, read back as broadcasts,
// took 42.9 ms.
template <bool SL, bool DL, bool GUARD>
__global__ __launch_bounds__(FF_BLOCK) void k_pairs_f64(
    const double *__restrict__ spos, const double *__restrict__ sld,
    const double *__restrict__ dld, long spg, const double *__restrict__ tpos, long n_trg, long tpg,
    SliceMap map, long plen, unsigned nsplit, double eps2, double scale, double ratio,
    double *__restrict__ part) {
  const unsigned slice = blockIdx.x % nsplit;
  const WaveTargets w = wave_targets(blockIdx.x / nsplit, map.share, n_trg, tpg);
  if (!w.live) return;
  const double tx = tpos[3 * w.tc], ty = tpos[3 * w.tc + 1], tz = tpos[3 * w.tc + 2];
  double S[3] = {0, 0, 0};
  Slice k = slice_of(map, slice);
  constexpr int U = DL ? 2 : 4;
  while (k.u < k.u1) {
    // the slice's parts of group k.g, in one run
    const unsigned take = min(map.nsub - k.j, k.u1 - k.u);
    const long g = k.g, r0 = k.j * plen, n = min(take * plen, spg - r0), s0 = g * spg + r0;
    if (g != w.own) {  // wave-uniform skip
      const double bias = w.group == g ? kOwnGroupBias64 : 0.0;
      const bool spans = __any(w.group == g);
      const double *__restrict__ p = spos + 3 * s0;
      const double *__restrict__ f = SL ? sld + 3 * s0 : p;
      const double *__restrict__ q = DL ? dld + 6 * s0 : p;
      for (long i = 0; i < n; i += 1 << 24)
        add_sources64<U, SL, DL, GUARD>(tx, ty, tz, bias, spans, (int)min(n - i, 1L << 24),
                                        p + 3 * i, f + 3 * i, q + 6 * i, ratio, eps2, S);
    }
    k.u += take;
    k.j = 0;
    ++k.g;
  }
  const double v[3] = {scale * S[0], scale * S[1], scale * S[2]};
  store_sums(w, map.share, n_trg, v, part + (long)slice * n_trg * 3);
}

// FP32 partial sums merged into a TwoSum (hi, lo) pair.
struct Acc32 {
  float h[3], l[3];
};
__device__ __forceinline__ void acc_merge(Acc32 &a, const float (&x)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float s_, e_;
    two_sum(a.h[c], x[c], s_, e_);
    a.h[c] = s_;
    a.l[c] += e_;
  }
}

// FP32 records (x, y, z[, f][, g, n]) relative to the anchor of their tile of
// FF_TILE sources (the tile's first point; tiles restart with every group).
template <bool SL, bool DL>
__global__ void k_pack_pairs32(const double *__restrict__ spos, const double *__restrict__ sld,
                               const double *__restrict__ dld, long n, long spg,
                               float *__restrict__ rec) {
  constexpr int R = 3 + (SL ? 3 : 0) + (DL ? 6 : 0);
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long g0 = spg > 0 ? quot(i, spg) * spg : 0;
  const double *a = spos + 3 * (g0 + (i - g0) / FF_TILE * FF_TILE);
  float *r = rec + i * R;
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = (float)(spos[3 * i + c] - a[c]);
  if (SL) {
#pragma unroll
    for (int c = 0; c < 3; ++c) r[3 + c] = (float)sld[3 * i + c];
  }
  if (DL) {
#pragma unroll
    for (int c = 0; c < 6; ++c) r[R - 6 + c] = (float)dld[6 * i + c];
  }
}

// The FP32 form over such records: cell c is tile c % ntile of group
// c / ntile (ungrouped: one group of n_src sources), cut into nsub parts of
// plen sources.  Bound: FP32 VALU issue, 18 instructions per single-layer
// pair and 28 with both layers, 3.5 cycles each on average.  Measured, single
// layer from 59,803 sources to 7,001 targets: 214 us with its packing and
// sum (217 us from LDS tiles).
template <bool SL, bool DL, bool GUARD>
__global__ __launch_bounds__(FF_BLOCK, DL ? 8 : (GUARD ? 6 : 7)) void k_pairs_f32c(
    const float *__restrict__ rec, const double *__restrict__ spos, long spg, unsigned ntile,
    const double *__restrict__ tpos, long n_trg, long tpg, SliceMap map, int plen, unsigned nsplit,
    float eps2, double scale, float ratio, double *__restrict__ part) {
  constexpr int R = 3 + (SL ? 3 : 0) + (DL ? 6 : 0), U = DL ? 4 : 8;
  constexpr int FO = 3, QO = R - 6;
  const unsigned slice = blockIdx.x % nsplit;
  const WaveTargets w = wave_targets(blockIdx.x / nsplit, map.share, n_trg, tpg);
  if (!w.live) return;
  const double tx = tpos[3 * w.tc], ty = tpos[3 * w.tc + 1], tz = tpos[3 * w.tc + 2];
  Acc32 A = {{0, 0, 0}, {0, 0, 0}};
  Slice k = slice_of(map, slice);
  unsigned tile = k.g % ntile;
  long g = k.g / ntile;
  while (k.u < k.u1) {
    // the slice's parts of cell k.g, in one run
    const unsigned take = min(map.nsub - k.j, k.u1 - k.u);
    if (g != w.own) {  // wave-uniform skip
      const long c0 = g * spg + (long)tile * FF_TILE;
      const int cnt = (int)min((long)FF_TILE, spg - (long)tile * FF_TILE);
      const int r0 = (int)k.j * plen, r1 = min(cnt, r0 + (int)take * plen);
      const bool mine = w.group == g;
      const float bias = mine ? kOwnGroupBias : 0.0f;
      const double *a = spos + 3 * c0;
      const float lx = (float)(tx - a[0]), ly = (float)(ty - a[1]), lz = (float)(tz - a[2]);
      for (int i0 = r0; i0 < r1; i0 += FF_SUB) {
        const float *__restrict__ r = rec + (c0 + i0) * R;
        const int n = min(FF_SUB, r1 - i0);
        float S[3] = {0, 0, 0};
        constexpr int run = GUARD ? FF_RUN : FF_SUB;
        for (int k0 = 0; k0 < n; k0 += run) {
          const int k1 = min(n, k0 + run);
          const float S0[3] = {S[0], S[1], S[2]};
          unsigned m = ~0u;
          int i = k0;
          for (; i + U <= k1; i += U)
            add_block32<U, SL ? 1 : 0, DL, GUARD>(r + i * R, lx, ly, lz, bias, ratio, S, S, m);
          for (; i < k1; ++i)
            add_block32<1, SL ? 1 : 0, DL, GUARD>(r + i * R, lx, ly, lz, bias, ratio, S, S, m);
          if (GUARD && __any(m <= order_key(eps2))) {
#pragma unroll
            for (int c = 0; c < 3; ++c) S[c] = S0[c];
#pragma unroll 1
            for (i = k0; i < k1; ++i) {
              const float *__restrict__ s = r + i * R;
              const float dx = lx - s[0], dy = ly - s[1], dz = lz - s[2];
              const float r2 = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, bias)));
              add_pair<SL, DL>(dx, dy, dz, r2 > eps2 ? rsqrt_pair(r2) : 0.0f, s + FO, s + QO,
                               ratio, S);
            }
          }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) S[c] = mine ? 0.0f : S[c];
        acc_merge(A, S);
      }
    }
    k.u += take;
    k.j = 0;
    if (++tile == ntile) {
      tile = 0;
      ++g;
    }
  }
  double v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = scale * ((double)A.h[c] + (double)A.l[c]);
  store_sums(w, map.share, n_trg, v, part + (long)slice * n_trg * 3);
}

// The FP32 form with its sources converted into LDS tile by tile, a workgroup's
// 256 targets on one slice: whole groups, or (spg = 0) an even part of the
// sources.  A lane leaves its own group out.
template <bool SL, bool DL, bool GUARD>
__global__ __launch_bounds__(FF_BLOCK) void k_tiles_f32c(
    const double *__restrict__ spos, const double *__restrict__ sld,
    const double *__restrict__ dld, long n_src, long spg, long n_groups,
    const double *__restrict__ tpos, long n_trg, long tpg, int nsplit, float eps2, double scale,
    float ratio, double *__restrict__ part) {
  struct __align__(16) Rec {
    float x[4], f[SL ? 4 : 1], q[DL ? 8 : 1];
  };
  __shared__ Rec sh[FF_TILE];
  const long slice = blockIdx.x % nsplit, tb = blockIdx.x / nsplit;
  const long t = tb * FF_BLOCK + threadIdx.x;
  const bool tvalid = t < n_trg, grouped = spg > 0;
  double tx = 0, ty = 0, tz = 0;
  if (tvalid) {
    tx = tpos[3 * t];
    ty = tpos[3 * t + 1];
    tz = tpos[3 * t + 2];
  }
  const long my_g = grouped && tvalid ? t / tpg : -1;
  const long tfirst = tb * FF_BLOCK, tlast = min(tfirst + FF_BLOCK, n_trg) - 1;
  // the group holding all the block's targets (or -1)
  const long own_b = grouped && tfirst / tpg == tlast / tpg ? tfirst / tpg : -1;
  Acc32 A = {{0, 0, 0}, {0, 0, 0}};
  const long g0 = grouped ? slice * n_groups / nsplit : 0;
  const long g1 = grouped ? (slice + 1) * n_groups / nsplit : 1;
  for (long g = g0; g < g1; ++g) {
    if (g == own_b) continue;  // block-uniform skip
    const long sb = grouped ? g * spg : slice * n_src / nsplit;
    const long se = grouped ? sb + spg : (slice + 1) * n_src / nsplit;
    const bool lane_on = tvalid && my_g != g;
    for (long c0 = sb; c0 < se; c0 += FF_TILE) {
      const int cnt = (int)min((long)FF_TILE, se - c0);
      __syncthreads();
      const double *a = spos + 3 * c0;
      if ((int)threadIdx.x < cnt) {
        const long s = c0 + threadIdx.x;
        Rec r;
#pragma unroll
        for (int c = 0; c < 3; ++c) r.x[c] = (float)(spos[3 * s + c] - a[c]);
        if constexpr (SL) {
#pragma unroll
          for (int c = 0; c < 3; ++c) r.f[c] = (float)sld[3 * s + c];
        }
        if constexpr (DL) {
#pragma unroll
          for (int c = 0; c < 6; ++c) r.q[c] = (float)dld[6 * s + c];
        }
        sh[threadIdx.x] = r;
      }
      __syncthreads();
      if (!lane_on) continue;
      const float lx = (float)(tx - a[0]), ly = (float)(ty - a[1]), lz = (float)(tz - a[2]);
      for (int j0 = 0; j0 < cnt; j0 += FF_SUB) {
        const int j1 = min(cnt, j0 + FF_SUB);
        float S[3] = {0, 0, 0};
#pragma unroll 4
        for (int j = j0; j < j1; ++j) {
          const float dx = lx - sh[j].x[0], dy = ly - sh[j].x[1], dz = lz - sh[j].x[2];
          const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
          const float rq = rsqrt_pair(r2);
          add_pair<SL, DL>(dx, dy, dz, GUARD ? (r2 > eps2 ? rq : 0.0f) : rq, sh[j].f, sh[j].q,
                           ratio, S);
        }
        acc_merge(A, S);
      }
    }
  }
  if (tvalid) {
    double *o = part + (slice * n_trg + t) * 3;
#pragma unroll
    for (int c = 0; c < 3; ++c) o[c] = scale * ((double)A.h[c] + (double)A.l[c]);
  }
}

// out[i] = the sum of the slices' partials: G threads per output add every
// G-th slice, and their sums are added in order.
template <int G>
__global__ __launch_bounds__(256) void k_sum_slices(const double *__restrict__ part, int nsplit,
                                                    long n, double *__restrict__ out) {
  constexpr int W = 256 / G;
  __shared__ double sh[G][W];
  const int c = threadIdx.x % W, q = threadIdx.x / W;
  const long i = (long)blockIdx.x * W + c;
  double s = 0;
  if (i < n) {
#pragma unroll 4
    for (int k = q; k < nsplit; k += G) s += part[(long)k * n + i];
  }
  sh[q][c] = s;
  __syncthreads();
  if (q == 0 && i < n) {
    for (int k = 1; k < G; ++k) s += sh[k][c];
    out[i] = s;
  }
}
static int sum_slices(const double *part, int nsplit, long n, double *out, hipStream_t st) {
  // one or two slices (few sources): a thread per output; few: one coalesced
  // 512-byte read per wave; many (few targets): 16 threads share an output's
  // chain of loads
  if (nsplit < 3)
    k_sum_slices<1><<<cdiv(n, 256), 256, 0, st>>>(part, nsplit, n, out);
  else if (nsplit >= 64)
    k_sum_slices<16><<<cdiv(n, 16), 256, 0, st>>>(part, nsplit, n, out);
  else
    k_sum_slices<4><<<cdiv(n, 64), 256, 0, st>>>(part, nsplit, n, out);
  return launch_status();
}

// How the sources are cut.  A wave's life must be short against the launch,
// or its last round leaves SIMDs idle: 32 waves per SIMD of the 256-CU part
// (32 * 1024), as long as a slice keeps 128 sources (the partial sums are 48
// bytes of traffic per slice and target); else 16 per SIMD in slices of at
// least FF_PART sources.  Where the targets alone give less than 2048 waves
// (1024 where the sources make fewer than four parts), the waves of a workgroup
// share their targets, which quarters the partial sums; 1024 slices bound them
// where the targets are few.  Otherwise the slices come in multiples of 8, one
// per XCD, where there are sources for 8 (300 sources to 1,000,000 targets in
// FP64: 251 us in two, 290 in eight); with shared targets they do on demand
// (per_xcd), for sources past an L2 (both layers from 100,000 points, 9.6 MB, to
// 10,000 in FP64: 1063 us, 1514 in 53 slices), if the last slice is filled too (48
// groups of 1202 sources, 5.5 MB: 1058 us in 36 slices, 1206 in 36 of 40).  Parts of
// groups even out the slices (about eight units each) unless there are many groups
// per slice.
// Measured: the far field of two vesicles (624 targets, 2404 sources) 10 us,
// 348 us with whole groups per slice; 2400 points to themselves 14.5 us with
// the sum, 22.7 us in slices of 256 sources.
struct Split {
  int nsplit;
  SliceMap map;
};
static Split choose_split(long n_trg, long n_groups, long spg, long max_slices = 1024,
                          bool per_xcd = false) {
  const long waves = (n_trg + 63) / 64, total = n_groups * spg;
  const unsigned share = waves < (total < 128 ? 1024 : 2048) ? 4 : 1;
  const long w16 = (16 * 1024 + waves - 1) / waves, w32 = 2 * w16;
  long want = total / 128 >= w16 ? std::min(w32, total / 128) : std::min(w16, total / FF_PART);
  if (share == 1) want = total / 128 >= 8 ? std::max(8L, (want + 7) / 8 * 8) : total / 128;
  want = std::max(1L, std::min(want, max_slices * share));
  const long finest = (spg + FF_PART - 1) / FF_PART;
  // units of `want` slices, about eight each
  auto parts = [&](long want) {
    return n_groups >= 8 * want ? 1 : std::min((8 * want + n_groups - 1) / n_groups, finest);
  };
  long nsub = parts(want), units = n_groups * nsub;
  long per = std::max(1L, units / want);
  if ((units + per - 1) / per > max_slices * share) per = (units + want - 1) / want;
  if (per_xcd && share > 1 && want >= 8 * share) {
    // a multiple of 8 workgroup slices, if the units fill the last one too (an
    // XCD with a slice less than the others waits for them)
    const long w = std::min((want + 8 * share - 1) / (8 * share), max_slices / 8) * 8 * share;
    const long s = parts(w), u = n_groups * s, p = (u + w - 1) / w;
    if (w > 0 && u >= 8 * w && (u + p - 1) / p > w - share) {
      nsub = s;
      units = u;
      per = p;
    }
  }
  const long slices = (units + per - 1) / per;
  Split s;
  s.nsplit = (int)((slices + share - 1) / share);
  s.map = SliceMap{(unsigned)units, (unsigned)per, (unsigned)nsub, share};
  return s;
}
// Slices of k_tiles_f32c, at most one per group or tile (cells): a multiple of 8
// (one per XCD), raised until the grid holds about 16 waves per SIMD.
static Split tile_split(long n_trg, long cells, long max_slices) {
  const long tblocks = (n_trg + FF_BLOCK - 1) / FF_BLOCK;
  long ns = 8;
  while (ns < 64 && tblocks * ns * (FF_BLOCK / 64) < 16 * 1024) ns *= 2;
  ns = std::min({ns, cells, max_slices});
  return Split{(int)ns, SliceMap{0, 0, 1, 1}};
}
// Where the FP32 form takes its sources through LDS tiles (k_tiles_f32c): no
// packing launch for few sources, and in the single layer, whose guarded record
// loop waits for scalar loads and the smallest distance, also where the targets
// alone fill the chip or groups are short.  Us, tiles / records: single layer, 64
// sources and 1000 targets 11.8 / 15.1; 300 and 10,000: 13.7 / 14.8, 1,000,000: 164 /
// 247; 2400 and 130,000: 152 / 165; 20,000 and 100,000: 897 / 931; but 1000 and 1000
// 18.7 / 14.6; groups of 12, 60,000 points 1839 / 2235, of 84, 21,000: 229 / 231, but of
// 312, 31,200: 567 / 491; both layers, 64 and 1000: 12.0 / 15.0, 300 and 130,000: 38 /
// 58, but 1000 and 1000 24.7 / 15.1, 20,000 and 100,000 1358 / 1253.
static bool tiles32(size_t n_src, size_t n_trg, size_t spg, bool dl) {
  if (spg > 0) return (!dl && spg <= 100) || (spg <= 64 && n_src * n_trg <= 2000000);
  if (!dl) return n_src <= 512 || n_trg >= 20000;
  return n_src <= 128 || (n_src <= 512 && n_trg >= (n_src > FF_TILE ? 24000 : 65536));
}
// Workgroups of a launch over n_trg targets.
static dim3 split_grid(const Split &s, long n_trg) {
  const long waves = (n_trg + 63) / 64;
  const long tblocks = s.map.share == 1 ? (waves + FF_BLOCK / 64 - 1) / (FF_BLOCK / 64) : waves;
  return dim3((unsigned)(tblocks * s.nsplit));
}
// Part length of a group of cnt sources cut into nsub parts, a multiple of q.
static long part_length(long cnt, unsigned nsub, long q) {
  const long l = (cnt + nsub - 1) / nsub;
  return std::max(q, (l + q - 1) / q * q);
}

template <bool SL, bool DL, bool GUARD>
static int launch_pairs64(dim3 grid, hipStream_t st, const double *spos, const double *sld,
                          const double *dld, long spg, const double *tpos, long n_trg, long tpg,
                          const Split &sp, double eps2, double csl, double cdl, double *part) {
  k_pairs_f64<SL, DL, GUARD><<<grid, FF_BLOCK, 0, st>>>(
      spos, sld, dld, spg, tpos, n_trg, tpg, sp.map, part_length(spg, sp.map.nsub, 4),
      (unsigned)sp.nsplit, eps2, SL ? csl : cdl, SL ? cdl / csl : 1.0, part);
  return launch_status();
}
// (rec null: through LDS tiles)
template <bool SL, bool DL, bool GUARD>
static int launch_pairs32(dim3 grid, hipStream_t st, const double *spos, const double *sld,
                          const double *dld, long n_src, long spg, unsigned ntile,
                          const double *tpos, long n_trg, long tpg, const Split &sp, double eps2,
                          double csl, double cdl, double *part, float *rec) {
  if (!rec) {
    k_tiles_f32c<SL, DL, GUARD><<<grid, FF_BLOCK, 0, st>>>(
        spos, sld, dld, n_src, tpg > 0 ? spg : 0, tpg > 0 ? n_src / spg : 0, tpos, n_trg, tpg,
        sp.nsplit, (float)eps2, SL ? csl : cdl, (float)(SL ? cdl / csl : 1.0), part);
    return launch_status();
  }
  k_pack_pairs32<SL, DL><<<cdiv(n_src, 256), 256, 0, st>>>(spos, sld, dld, n_src,
                                                           tpg > 0 ? spg : 0, rec);
  V3D_CHECK(launch_status());
  k_pairs_f32c<SL, DL, GUARD><<<grid, FF_BLOCK, 0, st>>>(
      rec, spos, spg, ntile, tpos, n_trg, tpg, sp.map, (int)part_length(std::min(spg, (long)FF_TILE), sp.map.nsub, 8),
      (unsigned)sp.nsplit, (float)eps2, SL ? csl : cdl, (float)(SL ? cdl / csl : 1.0), part);
  return launch_status();
}

// Shared driver of the all-pairs and far-field entry points.
// part_fixed (optional): caller-provided scratch of part_cap bytes for the
// per-slice partial sums instead of the library's workspace; the slice count
// is then held to what fits.
template <bool F32>
static int far_eval(const double *spos, const double *sld, const double *dld,
                    size_t n_src, const double *tpos, double *tvel, size_t n_trg,
                    size_t spg, size_t tpg, double eps2, double csl, double cdl,
                    hipStream_t st, bool guard = true, double *part_fixed = nullptr,
                    size_t part_cap = 0) {
  if (n_trg == 0) return VES3D_SUCCESS;
  if (!tpos || !tvel) return VES3D_INVALID_PARAMETER;
  if (n_src == 0 || (!sld && !dld)) {
    V3D_HIP(hipMemsetAsync(tvel, 0, n_trg * 3 * sizeof(double), st));
    return VES3D_SUCCESS;
  }
  if (!spos) return VES3D_INVALID_PARAMETER;
  const bool grouped = spg > 0 && tpg > 0;
  if (grouped && (n_src % spg || n_trg % tpg || n_src / spg != n_trg / tpg))
    return VES3D_INVALID_PARAMETER;
  const long n_groups = grouped ? (long)(n_src / spg) : 1;
  const long sp = grouped ? (long)spg : (long)n_src, tp = grouped ? (long)tpg : 0;
  const size_t per_slice = n_trg * 3 * sizeof(double);
  long max_slices = 1024;
  if (part_fixed) {
    if (per_slice > part_cap) return VES3D_INVALID_PARAMETER;
    max_slices = std::min(max_slices, (long)(part_cap / per_slice));
  }
  const size_t rec_n = 3 + (sld ? 3 : 0) + (dld ? 6 : 0);
  const bool tiles = F32 && tiles32(n_src, n_trg, grouped ? spg : 0, dld != nullptr);
  const bool per_xcd = !F32 && n_src * rec_n * sizeof(double) > (4u << 20);  // an L2
  const unsigned ntile = (unsigned)((sp + FF_TILE - 1) / FF_TILE);
  const Split split = tiles ? tile_split((long)n_trg, grouped ? n_groups : ntile, max_slices)
                      : F32 ? choose_split((long)n_trg, n_groups * ntile,
                                           std::min(sp, (long)FF_TILE), max_slices)
                            : choose_split((long)n_trg, n_groups, sp, max_slices, per_xcd);
  double *part =
      part_fixed ? part_fixed : (double *)workspace(kWsFarPartial, split.nsplit * per_slice);
  if (!part) return VES3D_MEMORY_ERROR;
  const bool packs = F32 && !tiles;
  float *rec = packs ? (float *)workspace(kWsFarRecords, n_src * rec_n * sizeof(float)) : nullptr;
  if (packs && !rec) return VES3D_MEMORY_ERROR;
  const dim3 grid = split_grid(split, (long)n_trg);
#define V3D_PAIRS(SL, DL, G)                                                                     \
  V3D_CHECK(F32 ? (launch_pairs32<SL, DL, G>(grid, st, spos, sld, dld, (long)n_src, sp, ntile,   \
                                             tpos, (long)n_trg, tp, split, eps2, csl, cdl, part, \
                                             rec))                                               \
                : (launch_pairs64<SL, DL, G>(grid, st, spos, sld, dld, sp, tpos, (long)n_trg,    \
                                             tp, split, eps2, csl, cdl, part)))
  if (sld && dld) {
    if (guard) V3D_PAIRS(true, true, true);
    else V3D_PAIRS(true, true, false);
  } else if (sld) {
    if (guard) V3D_PAIRS(true, false, true);
    else V3D_PAIRS(true, false, false);
  } else {
    if (guard) V3D_PAIRS(false, true, true);
    else V3D_PAIRS(false, true, false);
  }
#undef V3D_PAIRS
  return sum_slices(part, split.nsplit, (long)n_trg * 3, tvel, st);
}

// ---------------------------------------------------------------------------
// Far field between groups, with several source levels.  Every group
// (vesicle) carries its fine sources (the upsampled surface) and, optionally,
// coarser ones: level 1 the surface at its own order with its own quadrature
// weights, level 2 a lower order still.  flags[w][g] names the level wave w
// (targets 64 w .. 64 w + 63) reads group g at: level l where every target of
// the wave is at least kappa_l times g's radius from g's centre, so that the
// coarser quadrature is as accurate as the fine one there (null: the fine
// level everywhere; the flags never name an absent level).  The level, the
// record base and the count are wave-uniform (SGPRs).  A wave whose targets
// all belong to group g skips g.
constexpr int kMaxLevels = 3;
struct LevelSizes {
  int cnt[kMaxLevels];   // sources per group
  int plen[kMaxLevels];  // sources per part of a group
};
// The wave's level flags, 64 groups at a time in one register across the
// lanes: a flag in the source loop is then a v_readlane, not a load that
// everything after it waits for.
struct WaveFlags {
  const unsigned char *row;  // null: level 0 everywhere
  unsigned n_groups, base;
  int v;
  __device__ __forceinline__ void load(unsigned g) {
    base = g;
    const unsigned i = g + (threadIdx.x & 63);
    v = i < n_groups ? row[i] : 0;
  }
  __device__ __forceinline__ int level(unsigned g) {
    if (!row) return 0;
    if (g - base >= 64) load(g);
    return __builtin_amdgcn_readlane(v, (int)(g - base));
  }
};
__device__ __forceinline__ WaveFlags wave_flags(const unsigned char *flags, long row,
                                                unsigned n_groups, unsigned g0) {
  WaveFlags f{flags ? flags + row * n_groups : nullptr, n_groups, 0, 0};
  if (flags) f.load(g0);
  return f;
}

template <int ND>
__device__ __forceinline__ void store_pass(const WaveTargets &w, unsigned share, unsigned slice,
                                           long n_trg, const double (&v)[3 * ND], double *part1,
                                           double *part2) {
  const long o = (long)slice * n_trg * 3;
  const double a[3] = {v[0], v[1], v[2]};
  store_sums(w, share, n_trg, a, part1 + o);
  if constexpr (ND == 2) {
    const double b[3] = {v[3], v[4], v[5]};
    if (share > 1) __syncthreads();  // the first sums have left LDS
    store_sums(w, share, n_trg, b, part2 + o);
  }
}

// FP64 levels: point-major positions and densities as they lie.  ND: number
// of densities on the same sources (the step's right-hand side and its first
// matvec): the pair geometry (d, r^2, 1/r, 1/r^2) is computed once and serves
// both Stokeslet sums.
struct FarLevels64 {
  const double *pos[kMaxLevels], *den[2][kMaxLevels];
  LevelSizes n;
  const unsigned char *flags;
};
template <int ND>
__global__ __launch_bounds__(FF_BLOCK) void k_far_groups_f64(
    const FarLevels64 L, unsigned n_groups, const double *__restrict__ tpos, long n_trg, long tpg,
    SliceMap map, unsigned nsplit, double csl, double *__restrict__ part1,
    double *__restrict__ part2) {
  const unsigned slice = blockIdx.x % nsplit;
  const WaveTargets w = wave_targets(blockIdx.x / nsplit, map.share, n_trg, tpg);
  if (!w.live) return;
  const double tx = tpos[3 * w.tc], ty = tpos[3 * w.tc + 1], tz = tpos[3 * w.tc + 2];
  const int own = (int)w.own, group = (int)w.group;
  double S[ND][3] = {};
  Slice k = slice_of(map, slice);
  WaveFlags fl = wave_flags(L.flags, w.row, n_groups, k.g);
  while (k.u < k.u1) {
    const unsigned take = min(map.nsub - k.j, k.u1 - k.u);
    const int g = (int)k.g;
    if (g != own) {  // wave-uniform skip
      const double bias = group == g ? kOwnGroupBias64 : 0.0;
      const int lv = fl.level(g);
      const int cnt = L.n.cnt[lv], r0 = (int)k.j * L.n.plen[lv];
      const int n = min((int)take * L.n.plen[lv], cnt - r0);
      const long s0 = 3 * ((long)g * cnt + r0);
      const double *__restrict__ p = L.pos[lv] + s0;
      const double *__restrict__ f = L.den[0][lv] + s0;
      const double *__restrict__ h = L.den[ND - 1][lv] + s0;
      auto block = [&](int i, auto uc) {
        constexpr int U = decltype(uc)::value;
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const int e = 3 * (i + k);
          const double dx = tx - p[e], dy = ty - p[e + 1], dz = tz - p[e + 2];
          const double ri = rsqrt_pair(fma(dz, dz, fma(dy, dy, fma(dx, dx, bias))));
          add_pair<true, false>(dx, dy, dz, ri, f + e, f, 0.0, S[0]);
          if constexpr (ND == 2) add_pair<true, false>(dx, dy, dz, ri, h + e, h, 0.0, S[1]);
        }
      };
      constexpr int U = ND == 2 ? 2 : 4;
      int i = 0;
      for (; i + U <= n; i += U) block(i, std::integral_constant<int, U>());
      for (; i < n; ++i) block(i, std::integral_constant<int, 1>());
    }
    k.u += take;
    k.j = 0;
    ++k.g;
  }
  double v[3 * ND];
#pragma unroll
  for (int c = 0; c < 3 * ND; ++c) v[c] = csl * S[c / 3][c % 3];
  store_pass<ND>(w, map.share, slice, n_trg, v, part1, part2);
}

// FP32 levels: records (x, y, z, f[, h]) of 3 + 3 ND floats, relative to the
// group's anchor (its first fine source, for every level).  Measured, three
// levels of 512 vesicles at p = 16 (3.3e10 pairs): 13.5 ms with one density
// (15.1 ms with the pairs one after the other in program order, a flag load
// per group and the counts' remainders one source at a time); 65 VGPRs would
// cost the eighth wave per SIMD.
struct FarLevels32 {
  const float *rec[kMaxLevels];
  LevelSizes n;
  const unsigned char *flags;
};
template <int ND>
__global__ void k_pack_far32(const double *__restrict__ spos, const double *__restrict__ s1,
                             const double *__restrict__ s2, long n, long spg,
                             const double *__restrict__ anc, long apg, float *__restrict__ rec) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *a = anc + 3 * quot(i, spg) * apg;
  float *r = rec + i * (3 + 3 * ND);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    r[c] = (float)(spos[3 * i + c] - a[c]);
    r[3 + c] = (float)s1[3 * i + c];
    if constexpr (ND == 2) r[6 + c] = (float)s2[3 * i + c];
  }
}
template <int ND>
__global__ __launch_bounds__(FF_BLOCK, 8) void k_far_groups_f32c(
    const FarLevels32 L, const double *__restrict__ spos, unsigned n_groups,
    const double *__restrict__ tpos, long n_trg, long tpg, SliceMap map, unsigned nsplit,
    double csl, double *__restrict__ part1, double *__restrict__ part2) {
  constexpr int R = 3 + 3 * ND;
  const unsigned slice = blockIdx.x % nsplit;
  const WaveTargets w = wave_targets(blockIdx.x / nsplit, map.share, n_trg, tpg);
  if (!w.live) return;
  const double tx = tpos[3 * w.tc], ty = tpos[3 * w.tc + 1], tz = tpos[3 * w.tc + 2];
  const int own = (int)w.own, group = (int)w.group;
  Acc32 A = {{0, 0, 0}, {0, 0, 0}}, B = {{0, 0, 0}, {0, 0, 0}};
  Slice k = slice_of(map, slice);
  WaveFlags fl = wave_flags(L.flags, w.row, n_groups, k.g);
  while (k.u < k.u1) {
    const unsigned take = min(map.nsub - k.j, k.u1 - k.u);
    const int g = (int)k.g;
    if (g != own) {  // wave-uniform skip
      const float bias = group == g ? kOwnGroupBias : 0.0f;
      const double *a = spos + 3 * (long)g * L.n.cnt[0];  // the group's anchor
      const float lx = (float)(tx - a[0]), ly = (float)(ty - a[1]), lz = (float)(tz - a[2]);
      const int lv = fl.level(g);
      const int cnt = L.n.cnt[lv], r0 = (int)k.j * L.n.plen[lv];
      const int r1 = min(cnt, r0 + (int)take * L.n.plen[lv]);
      const float *__restrict__ r = L.rec[lv] + (long)g * cnt * R;
      for (int i0 = r0; i0 < r1; i0 += FF_SUB) {
        const float *__restrict__ rr = r + (long)i0 * R;
        const int n = min(FF_SUB, r1 - i0);
        float S[3] = {0, 0, 0}, T[3] = {0, 0, 0};
        constexpr int U = ND == 2 ? 4 : 8;
        unsigned m = 0;
        int i = 0;
        for (; i + U <= n; i += U)
          add_block32<U, ND, false, false>(rr + i * R, lx, ly, lz, bias, 0.0f, S, T, m);
        for (; i < n; ++i)
          add_block32<1, ND, false, false>(rr + i * R, lx, ly, lz, bias, 0.0f, S, T, m);
        acc_merge(A, S);
        if constexpr (ND == 2) acc_merge(B, T);
      }
    }
    k.u += take;
    k.j = 0;
    ++k.g;
  }
  double v[3 * ND];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    v[c] = csl * ((double)A.h[c] + (double)A.l[c]);
    if constexpr (ND == 2) v[3 + c] = csl * ((double)B.h[c] + (double)B.l[c]);
  }
  store_pass<ND>(w, map.share, slice, n_trg, v, part1, part2);
}

// 0: the all-pairs entry points' kernels (k_pairs_*), otherwise
// k_far_groups_*; selects the far field between groups without coarser levels.
static std::atomic<int> g_far_kind{1};

// ---------------------------------------------------------------------------
// Per-vesicle Device<>::DirectStokes / DirectStokesDoubleLayer.

// U consecutive sources of one vesicle (AxisMajor, stride ss) at one target.
// DLK=false: single layer, w [d / r + (d . r) r / r^3]
// DLK=true : double layer, w (r.n)(r.d) r / r^5                (r = src - trg)
// HASW: quadrature weights w (else 1).  m keeps the smallest r^2; SELECT: pairs
// with r = 0 contribute nothing, any other r^2 is taken as it is (see FF_RUN).
template <int U, bool DLK, bool HASW, bool SELECT, typename T>
__device__ __forceinline__ void add_surface(const T *__restrict__ src, const T *__restrict__ nrm,
                                            const T *__restrict__ den, const T *__restrict__ qw,
                                            long ss, T tx, T ty, T tz, T (&S)[3], unsigned &m) {
  T x[3][U], f[3][U], n[3][U], w[U];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[c][u] = src[c * ss + u];
      f[c][u] = den[c * ss + u];
      if constexpr (DLK) n[c][u] = nrm[c * ss + u];
    }
  if constexpr (HASW) {
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = qw[u];
  }
  T d[3][U], ri[U], t[U], q[U];
  stage<U>([&](int u) { d[0][u] = x[0][u] - tx; });
  stage<U>([&](int u) { d[1][u] = x[1][u] - ty; });
  stage<U>([&](int u) { d[2][u] = x[2][u] - tz; });
  stage<U>([&](int u) { ri[u] = d[0][u] * d[0][u]; });
  stage<U>([&](int u) { ri[u] = fma(d[1][u], d[1][u], ri[u]); });
  stage<U>([&](int u) { ri[u] = fma(d[2][u], d[2][u], ri[u]); });
  if constexpr (SELECT) {
    stage<U>([&](int u) { ri[u] = ri[u] != T(0) ? T(1) / sqrt(ri[u]) : T(0); });
  } else {
    stage<U>([&](int u) { m = min(m, order_key(ri[u])); });
    stage<U>([&](int u) { ri[u] = rsqrt_pair(ri[u]); });
  }
  auto dot = [&](T (&o)[U], const T (&v)[3][U]) {
    stage<U>([&](int u) { o[u] = v[0][u] * d[0][u]; });
    stage<U>([&](int u) { o[u] = fma(v[1][u], d[1][u], o[u]); });
    stage<U>([&](int u) { o[u] = fma(v[2][u], d[2][u], o[u]); });
  };
  dot(t, f);
  stage<U>([&](int u) { q[u] = ri[u] * ri[u]; });
  if constexpr (SELECT) {  // (1/r^2 may overflow)
    stage<U>([&](int u) { t[u] = t[u] * ri[u] * ri[u]; });
  } else {
    stage<U>([&](int u) { t[u] *= q[u]; });
  }
  if constexpr (HASW) stage<U>([&](int u) { ri[u] *= w[u]; });
  if constexpr (DLK) {
    T g[U];
    dot(g, n);
    stage<U>([&](int u) { t[u] *= g[u]; });
    stage<U>([&](int u) { q[u] *= ri[u]; });
    stage<U>([&](int u) { t[u] *= q[u]; });
    stage<U>([&](int u) {
#pragma unroll
      for (int c = 0; c < 3; ++c) S[c] = fma(d[c][u], t[u], S[c]);
    });
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      stage<U>([&](int u) { d[c][u] = fma(d[c][u], t[u], f[c][u]); });
    stage<U>([&](int u) {
#pragma unroll
      for (int c = 0; c < 3; ++c) S[c] = fma(ri[u], d[c][u], S[c]);
    });
  }
}

// r^2 below the normal numbers, where the hardware's 1/sqrt estimate fails.
template <typename T>
constexpr unsigned kTinyKey = sizeof(T) == 8 ? 0x00100000u : 0x00800000u;

// A workgroup takes 64 targets of one vesicle; wave k the sources
// k chunk .. (k + 1) chunk - 1, and the waves' sums are added in order
// through LDS.  Runs with a vanishing r^2, or one past the largest number
// (where the estimate's refinement gives no number), are summed again with the
// division.  Workgroups reach the XCDs in turn, so the groups (vesicle, target
// block) are dealt out in consecutive ranges: a vesicle's groups run together
// and find its sources in one L2 (in launch order 822 us instead of 632 for the
// single, 2068 instead of 1030 for the double layer below).
// Bound: VALU issue (25 instructions per FP64 single-layer pair with weights)
// and the scalar loads of 7 (10) numbers per source.  One wave per 64 targets
// with the sources staged through LDS left most of the chip idle and divided for
// every pair.  FP64, 512 vesicles of 2112 sources and 544 targets: 1430 -> 632
// us, double layer 1420 -> 1030; 40 vesicles of 544 and 544: 108 -> 25 us; FP32:
// 696 -> 276, 815 -> 409, 98 -> 18 us.
template <typename Real, bool DLK, bool HASW>
__global__ __launch_bounds__(1024) void k_vesicle_stokes(
    const Real *__restrict__ src, const Real *__restrict__ nrm, const Real *__restrict__ den,
    const Real *__restrict__ qw, long ss, long ts, long head, long tail, long chunk,
    unsigned nblocks, const Real *__restrict__ trg, Real *__restrict__ pot, Real scal) {
  __shared__ Real red[15][3][64];
  const unsigned per = gridDim.x / 8, more = gridDim.x % 8, xcd = blockIdx.x % 8;
  const unsigned id = xcd * per + min(xcd, more) + blockIdx.x / 8;
  const long vt = id / nblocks;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long t = head + (long)(id % nblocks) * 64 + lane;
  const Real *T = trg + 3 * ts * vt + min(t, tail - 1);
  const Real tx = T[0], ty = T[ts], tz = T[2 * ts];
  const long s0 = wv * chunk, n = min(chunk, ss - s0);
  const Real *__restrict__ X = src + 3 * ss * vt + s0;
  const Real *__restrict__ D = den + 3 * ss * vt + s0;
  const Real *__restrict__ N = DLK ? nrm + 3 * ss * vt + s0 : X;
  const Real *__restrict__ W = HASW ? qw + s0 : X;
  Real S[3] = {0, 0, 0};
  // as many as the SGPRs hold: 7 (SL) or 10 (DL) streams of U values
  constexpr int U = sizeof(Real) == 8 ? (DLK ? 2 : 4) : (DLK ? 4 : 8);
  for (long i0 = 0; i0 < n; i0 += FF_RUN) {
    const long i1 = min(n, i0 + FF_RUN);
    const Real S0[3] = {S[0], S[1], S[2]};
    unsigned m = ~0u;
    long i = i0;
    for (; i + U <= i1; i += U)
      add_surface<U, DLK, HASW, false>(X + i, N + i, D + i, W + i, ss, tx, ty, tz, S, m);
    for (; i < i1; ++i)
      add_surface<1, DLK, HASW, false>(X + i, N + i, D + i, W + i, ss, tx, ty, tz, S, m);
    const Real sum = S[0] + S[1] + S[2];
    if (__any(m < kTinyKey<Real> || sum != sum)) {
#pragma unroll
      for (int c = 0; c < 3; ++c) S[c] = S0[c];
#pragma unroll 1
      for (i = i0; i < i1; ++i)
        add_surface<1, DLK, HASW, true>(X + i, N + i, D + i, W + i, ss, tx, ty, tz, S, m);
    }
  }
  const int nw = blockDim.x >> 6;
  if (wv > 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) red[wv - 1][c][lane] = S[c];
  }
  __syncthreads();
  if (wv > 0 || t >= tail) return;
  Real *P = pot + 3 * ts * vt + t;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    for (int k = 0; k < nw - 1; ++k) S[c] += red[k][c][lane];
    P[c * ts] = S[c] * scal;
  }
}

// One wave per 64 targets of a vesicle, whose sources go through LDS.
constexpr int VS_TILE = 256;
template <typename Real, bool DLK>
__global__ __launch_bounds__(64) void k_vesicle_staged(
    const Real *__restrict__ src, const Real *__restrict__ nrm, const Real *__restrict__ den,
    const Real *__restrict__ qw, long ss, long ts, long head, long tail,
    const Real *__restrict__ trg, Real *__restrict__ pot, Real scal) {
  __shared__ Real sh[VS_TILE][DLK ? 10 : 6];
  const long vt = blockIdx.y;
  const long t = head + (long)blockIdx.x * 64 + threadIdx.x;
  const bool tvalid = t < tail;
  const Real *S = src + 3 * ss * vt;
  const Real *D = den + 3 * ss * vt;
  const Real *N = DLK ? nrm + 3 * ss * vt : nullptr;
  Real tx = 0, ty = 0, tz = 0;
  if (tvalid) {
    const Real *T = trg + 3 * ts * vt;
    tx = T[t];
    ty = T[ts + t];
    tz = T[2 * ts + t];
  }
  Real px = 0, py = 0, pz = 0;
  for (long c0 = 0; c0 < ss; c0 += VS_TILE) {
    const int cnt = (int)min((long)VS_TILE, ss - c0);
    __syncthreads();
    for (int i = threadIdx.x; i < cnt; i += 64) {
      const long s = c0 + i;
      const Real w = qw ? qw[s] : Real(1);
      sh[i][0] = S[s];
      sh[i][1] = S[ss + s];
      sh[i][2] = S[2 * ss + s];
      if (DLK) {
        sh[i][3] = D[s];
        sh[i][4] = D[ss + s];
        sh[i][5] = D[2 * ss + s];
        sh[i][6] = N[s];
        sh[i][7] = N[ss + s];
        sh[i][8] = N[2 * ss + s];
        sh[i][9] = w;
      } else {
        sh[i][3] = D[s] * w;
        sh[i][4] = D[ss + s] * w;
        sh[i][5] = D[2 * ss + s] * w;
      }
    }
    __syncthreads();
    if (tvalid) {
#pragma unroll 4
      for (int j = 0; j < cnt; ++j) {
        const Real dx = sh[j][0] - tx, dy = sh[j][1] - ty, dz = sh[j][2] - tz;
        const Real r2 = dx * dx + dy * dy + dz * dz;
        const Real ri = (r2 != Real(0)) ? Real(1) / sqrt(r2) : Real(0);
        if (DLK) {
          const Real ri2 = ri * ri;
          const Real rn = sh[j][6] * dx + sh[j][7] * dy + sh[j][8] * dz;
          const Real rf = sh[j][3] * dx + sh[j][4] * dy + sh[j][5] * dz;
          const Real c = rn * rf * (ri2 * ri2 * ri) * sh[j][9];
          px += dx * c;
          py += dy * c;
          pz += dz * c;
        } else {
          const Real cc = (dx * sh[j][3] + dy * sh[j][4] + dz * sh[j][5]) * ri * ri;
          px += (sh[j][3] + cc * dx) * ri;
          py += (sh[j][4] + cc * dy) * ri;
          pz += (sh[j][5] + cc * dz) * ri;
        }
      }
    }
  }
  if (tvalid) {
    Real *P = pot + 3 * ts * vt;
    P[t] = px * scal;
    P[ts + t] = py * scal;
    P[2 * ts + t] = pz * scal;
  }
}

template <typename Real, bool DLK>
static int vesicle_stokes(const Real *src, const Real *nrm, const Real *den,
                          const Real *qw, size_t ss, size_t ts, size_t nv,
                          const Real *trg, size_t head, size_t tail, Real *pot,
                          hipStream_t st) {
  if (tail < head || tail > ts) return VES3D_INVALID_PARAMETER;
  if (nv == 0 || tail == head) return VES3D_SUCCESS;
  if (!src || !den || !trg || !pot || (DLK && !nrm)) return VES3D_INVALID_PARAMETER;
  if (nv > 65535) return VES3D_INVALID_PARAMETER;
  const Real scal = DLK ? Real(-3.0 / (4.0 * kPi)) : Real(1.0 / kPi / 8.0);
  const size_t nblocks = cdiv(tail - head, 64), groups = nblocks * nv;
  if (groups > 0x7fffffff) return VES3D_INVALID_PARAMETER;
  // Staged through LDS by one wave where a group has too few sources for the
  // start and end of a wave that splits them (FP64 double layer, 16 sources, 1500
  // vesicles of 544 targets 37 us, 40 to 96 split; single layer, 8, 4000 vesicles 44,
  // 50 to 194), and in the double layer where at most two groups share a vesicle's
  // sources and all vesicles' are too many for the caches, so that the scalar
  // loads of ten streams wait for memory (2112 sources, 20 targets, 4000 vesicles:
  // FP64 1142 us, 2757 split, FP32 623, 917; 512 sources, FP64 283, 337; but 1104
  // sources of 1500 vesicles 324, 292, four groups per vesicle 1002, 717, 8 targets
  // of 1500 vesicles with 2112 sources 928, 764, and in FP32 5000 sources 1055, 703).
  const size_t src_bytes = nv * ss * 9 * sizeof(Real);
  const bool many = groups >= 3000, large = src_bytes >= 200000000;
  const bool waits = sizeof(Real) == 8 ? (many && ss >= 128) || (large && tail - head >= 16)
                                       : many && large;
  const bool staged = ss <= 16 || (DLK && nblocks <= 2 && waits);
  if (staged) {
    k_vesicle_staged<Real, DLK><<<dim3((unsigned)nblocks, (unsigned)nv), 64, 0, st>>>(
        src, nrm, den, qw, (long)ss, (long)ts, (long)head, (long)tail, trg, pot, scal);
    return launch_status();
  }
  // Four waves per group from 1024 groups on, 16 below, and no more than give each
  // at least 8 (FP32: 16) sources: 4 / 16 waves for 1500 vesicles of 64 sources and
  // 544 targets in FP32 43 / 164 us, two 36; 40 vesicles of 512 and 544 in FP64 22 / 21.
  int nw = groups >= 1024 ? 4 : 16;
  while (nw > 1 && (size_t)nw * (sizeof(Real) == 8 ? 8 : 16) > ss) nw /= 2;
  const long chunk = (long)((ss + nw - 1) / nw + 3) / 4 * 4;
  if (qw)
    k_vesicle_stokes<Real, DLK, true><<<(unsigned)groups, 64 * nw, 0, st>>>(
        src, nrm, den, qw, (long)ss, (long)ts, (long)head, (long)tail, chunk, (unsigned)nblocks,
        trg, pot, scal);
  else
    k_vesicle_stokes<Real, DLK, false><<<(unsigned)groups, 64 * nw, 0, st>>>(
        src, nrm, den, qw, (long)ss, (long)ts, (long)head, (long)tail, chunk, (unsigned)nblocks,
        trg, pot, scal);
  return launch_status();
}

// Coincident-point guard of the PVFMMEval stand-in (r^2 <= 128 eps is skipped).
static const double kEvalEps2 = 128.0 * 2.220446049250313e-16;

// Bounding sphere of every group's fine sources: bnd[g] = (centre, radius),
// the centre the mean of the sources.  One workgroup per group.
__global__ __launch_bounds__(256) void k_group_bounds(const double *__restrict__ spos, long spg,
                                                      double4 *__restrict__ bnd) {
  const long g = blockIdx.x;
  const double *P = spos + 3 * g * spg;
  __shared__ double red[4][4];
  __shared__ double cen[3];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  double c[3] = {0, 0, 0};
  for (long j = threadIdx.x; j < spg; j += 256)
    for (int d = 0; d < 3; ++d) c[d] += P[3 * j + d];
  for (int d = 0; d < 3; ++d) {
    const double t = wave_sum(c[d]);
    if (lane == 0) red[wv][d] = t;
  }
  __syncthreads();
  if (threadIdx.x < 3)
    cen[threadIdx.x] =
        (((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x]) /
        (double)spg;
  __syncthreads();
  double m = 0;
  for (long j = threadIdx.x; j < spg; j += 256) {
    const double dx = P[3 * j] - cen[0], dy = P[3 * j + 1] - cen[1], dz = P[3 * j + 2] - cen[2];
    m = fmax(m, dx * dx + dy * dy + dz * dz);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  if (lane == 0) red[wv][3] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    bnd[g] = make_double4(cen[0], cen[1], cen[2],
                          sqrt(fmax(fmax(red[0][3], red[1][3]), fmax(red[2][3], red[3][3]))));
}

// flags[w][g] = 2 where every target of wave w is at least kappa2 R_g from
// c_g (kappa2 > 0), else 1 where at least kappa R_g, else 0.  One workgroup
// per wave: its 64 targets in LDS, the threads over the groups.
// counts[0] += the wave's level-1 (wave, group) pairs, counts[1] += its fine
// ones (groups the wave does not skip as its own), counts[2] += its level-2
// ones.
__global__ __launch_bounds__(256) void k_coarse_flags(const double *__restrict__ tpos, long n_trg,
                                                      long tpg, const double4 *__restrict__ bnd,
                                                      long n_groups, double kappa, double kappa2,
                                                      unsigned char *__restrict__ flags,
                                                      unsigned long long *__restrict__ counts) {
  const long w = blockIdx.x;
  __shared__ double T[64][3];
  __shared__ unsigned cnt[3];
  if (threadIdx.x < 64) {
    const long t = min(w * 64 + threadIdx.x, n_trg - 1);
    for (int d = 0; d < 3; ++d) T[threadIdx.x][d] = tpos[3 * t + d];
  }
  if (threadIdx.x < 3) cnt[threadIdx.x] = 0;
  __syncthreads();
  const long gf = (w * 64) / tpg, gl = min(w * 64 + 63, n_trg - 1) / tpg;
  unsigned nc = 0, nf = 0, nc2 = 0;
  for (long g = threadIdx.x; g < n_groups; g += 256) {
    const double4 b = bnd[g];
    double m = 1e300;
    for (int k = 0; k < 64; ++k) {
      const double dx = T[k][0] - b.x, dy = T[k][1] - b.y, dz = T[k][2] - b.z;
      m = fmin(m, dx * dx + dy * dy + dz * dz);
    }
    const double lim = kappa * b.w, lim2 = kappa2 * b.w;
    const int lv = (kappa2 > 0.0 && m >= lim2 * lim2) ? 2 : (m >= lim * lim ? 1 : 0);
    flags[w * n_groups + g] = (unsigned char)lv;
    if (lv == 2) ++nc2;
    else if (lv == 1) ++nc;
    else if (!(gf == g && gl == g)) ++nf;
  }
  atomicAdd(&cnt[0], nc);
  atomicAdd(&cnt[1], nf);
  atomicAdd(&cnt[2], nc2);
  __syncthreads();
  if (threadIdx.x < 3) atomicAdd(&counts[threadIdx.x], (unsigned long long)cnt[threadIdx.x]);
}

__global__ void k_zero_u64(unsigned long long *p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

int far_field_sl_dl(bool f32c, const double *spos, const double *sld, const double *dld,
                    size_t n_src, const double *tpos, double *tvel, size_t n_trg, size_t spg,
                    size_t tpg, bool guard, hipStream_t st) {
  const double csl = 1.0 / (8.0 * kPi), cdl = 3.0 / (4.0 * kPi);
  const double eps2 = guard ? kEvalEps2 : 0.0;
  if (f32c)
    return far_eval<true>(spos, sld, dld, n_src, tpos, tvel, n_trg, spg, tpg, eps2, csl, cdl, st,
                          guard);
  return far_eval<false>(spos, sld, dld, n_src, tpos, tvel, n_trg, spg, tpg, eps2, csl, cdl, st,
                         guard);
}

int direct_eval_f64_fixed(const double *src_pos, const double *sl_den, const double *dl_den,
                          size_t n_src, const double *trg_pos, double *trg_vel, size_t n_trg,
                          size_t spg, size_t tpg, double *part, size_t part_bytes,
                          hipStream_t st) {
  if (!part) return VES3D_INVALID_PARAMETER;
  return far_eval<false>(src_pos, sl_den, dl_den, n_src, trg_pos, trg_vel, n_trg, spg, tpg,
                         kEvalEps2, 1.0 / (8.0 * kPi), 3.0 / (4.0 * kPi), st, true, part,
                         part_bytes);
}

// A level-2 set needs a level-1 set; two densities need both of each set.
static bool coarse_valid(const FarCoarse &c, bool two) {
  if (!c.pos || !c.den1 || !c.flags || c.cpg == 0 || (two && !c.den2)) return false;
  if (c.cpg2 == 0) return true;
  return c.pos2 && c.l2den1 && (!two || c.l2den2);
}

int far_coarse_flags(const double *spos, size_t n_src, size_t spg, const double *tpos,
                     size_t n_trg, size_t tpg, double kappa, double kappa2, unsigned char *flags,
                     unsigned long long *counts, hipStream_t st) {
  if (!spos || !tpos || !flags || !counts || spg == 0 || tpg == 0 || n_src % spg || n_trg == 0 ||
      !(kappa > 1.0) || !(kappa2 == 0.0 || kappa2 > kappa))
    return VES3D_INVALID_PARAMETER;
  const long n_groups = (long)(n_src / spg);
  double4 *bnd = (double4 *)workspace(kWsFarBounds, sizeof(double4) * n_groups);
  if (!bnd) return VES3D_MEMORY_ERROR;
  k_group_bounds<<<(unsigned)n_groups, 256, 0, st>>>(spos, (long)spg, bnd);
  V3D_CHECK(launch_status());
  k_zero_u64<<<1, 64, 0, st>>>(counts, 3);
  V3D_CHECK(launch_status());
  const long n_waves = ((long)n_trg + 63) / 64;
  k_coarse_flags<<<(unsigned)n_waves, 256, 0, st>>>(tpos, (long)n_trg, (long)tpg, bnd, n_groups,
                                                    kappa, kappa2, flags, counts);
  return launch_status();
}

// Packed FP32 records of every level (ND densities), or null on failure.
template <int ND>
static int pack_levels32(const double *spos, const double *s1, const double *s2, long n_src,
                         long spg, const FarCoarse *c, long n_groups, hipStream_t st,
                         FarLevels32 *L) {
  constexpr size_t rsz = (3 + 3 * ND) * sizeof(float);
  const long n_c = c ? (long)c->cpg * n_groups : 0, n_c2 = c ? (long)c->cpg2 * n_groups : 0;
  float *rec = (float *)workspace(kWsFarRecords, n_src * rsz);
  float *crec = n_c ? (float *)workspace(kWsFarCoarse, n_c * rsz) : nullptr;
  float *crec2 = n_c2 ? (float *)workspace(kWsFarCoarse2, n_c2 * rsz) : nullptr;
  if (!rec || (n_c && !crec) || (n_c2 && !crec2)) return VES3D_MEMORY_ERROR;
  k_pack_far32<ND><<<cdiv(n_src, 256), 256, 0, st>>>(spos, s1, s2, n_src, spg, spos, spg, rec);
  V3D_CHECK(launch_status());
  if (n_c) {
    k_pack_far32<ND><<<cdiv(n_c, 256), 256, 0, st>>>(c->pos, c->den1, c->den2, n_c, (long)c->cpg,
                                                     spos, spg, crec);
    V3D_CHECK(launch_status());
  }
  if (n_c2) {
    k_pack_far32<ND><<<cdiv(n_c2, 256), 256, 0, st>>>(c->pos2, c->l2den1, c->l2den2, n_c2,
                                                      (long)c->cpg2, spos, spg, crec2);
    V3D_CHECK(launch_status());
  }
  L->rec[0] = rec;
  L->rec[1] = crec;
  L->rec[2] = crec2;
  return VES3D_SUCCESS;
}

// ND densities s1 (and s2) on the same sources, one pass.
template <int ND>
static int far_groups(bool f32c, const double *spos, const double *s1, const double *s2,
                      size_t n_src, const double *tpos, double *tvel1, double *tvel2,
                      size_t n_trg, size_t spg, size_t tpg, hipStream_t st,
                      const FarCoarse *coarse) {
  if (n_trg == 0) return VES3D_SUCCESS;
  if (!spos || !s1 || !tpos || !tvel1 || (ND == 2 && (!s2 || !tvel2)))
    return VES3D_INVALID_PARAMETER;
  if (n_src % spg || n_trg % tpg || n_src / spg != n_trg / tpg) return VES3D_INVALID_PARAMETER;
  if (coarse && !coarse_valid(*coarse, ND == 2)) return VES3D_INVALID_PARAMETER;
  const double csl = 1.0 / (8.0 * kPi);
  const long n_groups = (long)(n_src / spg);
  if (n_groups > 0x7fffffffL || spg > 0x7fffffffUL) return VES3D_INVALID_PARAMETER;
  const Split split = choose_split((long)n_trg, n_groups, (long)spg);
  const size_t per_pass = (size_t)split.nsplit * n_trg * 3;
  double *part = (double *)workspace(kWsFarPartial, ND * per_pass * sizeof(double));
  if (!part) return VES3D_MEMORY_ERROR;
  double *part2 = part + (ND - 1) * per_pass;
  LevelSizes n;
  const long cnt[kMaxLevels] = {(long)spg, coarse ? (long)coarse->cpg : 0,
                                coarse ? (long)coarse->cpg2 : 0};
  for (int l = 0; l < kMaxLevels; ++l) {
    n.cnt[l] = (int)cnt[l];
    n.plen[l] = (int)part_length(cnt[l], split.map.nsub, f32c ? 8 : 4);
  }
  const unsigned char *flags = coarse ? coarse->flags : nullptr;
  const dim3 grid = split_grid(split, (long)n_trg);
  if (f32c) {
    FarLevels32 L{};
    V3D_CHECK(pack_levels32<ND>(spos, s1, s2, (long)n_src, (long)spg, coarse, n_groups, st, &L));
    L.n = n;
    L.flags = flags;
    k_far_groups_f32c<ND><<<grid, FF_BLOCK, 0, st>>>(L, spos, (unsigned)n_groups, tpos, (long)n_trg,
                                                     (long)tpg, split.map, (unsigned)split.nsplit,
                                                     csl, part, part2);
  } else {
    FarLevels64 L{};
    L.pos[0] = spos;
    L.den[0][0] = s1;
    L.den[1][0] = s2;
    if (coarse) {
      L.pos[1] = coarse->pos;
      L.den[0][1] = coarse->den1;
      L.den[1][1] = coarse->den2;
      L.pos[2] = coarse->pos2;
      L.den[0][2] = coarse->l2den1;
      L.den[1][2] = coarse->l2den2;
    }
    L.n = n;
    L.flags = flags;
    k_far_groups_f64<ND><<<grid, FF_BLOCK, 0, st>>>(L, (unsigned)n_groups, tpos, (long)n_trg,
                                                    (long)tpg, split.map, (unsigned)split.nsplit,
                                                    csl, part, part2);
  }
  V3D_CHECK(launch_status());
  V3D_CHECK(sum_slices(part, split.nsplit, (long)n_trg * 3, tvel1, st));
  return ND == 2 ? sum_slices(part2, split.nsplit, (long)n_trg * 3, tvel2, st) : VES3D_SUCCESS;
}

int far_field_between_groups(bool f32c, const double *spos, const double *sld, size_t n_src,
                             const double *tpos, double *tvel, size_t n_trg, size_t spg,
                             size_t tpg, hipStream_t st, const FarCoarse *coarse) {
  if (spg == 0 || tpg == 0) return VES3D_INVALID_PARAMETER;
  if (!coarse && g_far_kind.load() == 0)
    return far_field_sl_dl(f32c, spos, sld, nullptr, n_src, tpos, tvel, n_trg, spg, tpg, false, st);
  return far_groups<1>(f32c, spos, sld, nullptr, n_src, tpos, tvel, nullptr, n_trg, spg, tpg, st,
                       coarse);
}

int far_field_between_groups2(bool f32c, const double *spos, const double *sld1,
                              const double *sld2, size_t n_src, const double *tpos, double *tvel1,
                              double *tvel2, size_t n_trg, size_t spg, size_t tpg,
                              hipStream_t st, const FarCoarse *coarse) {
  if (spg == 0 || tpg == 0) return VES3D_INVALID_PARAMETER;
  if (!coarse && g_far_kind.load() == 0) {  // one density at a time
    V3D_CHECK(far_field_between_groups(f32c, spos, sld1, n_src, tpos, tvel1, n_trg, spg, tpg, st));
    return far_field_between_groups(f32c, spos, sld2, n_src, tpos, tvel2, n_trg, spg, tpg, st);
  }
  return far_groups<2>(f32c, spos, sld1, sld2, n_src, tpos, tvel1, tvel2, n_trg, spg, tpg, st,
                       coarse);
}

}  // namespace v3d

// ---------------------------------------------------------------------------
// C ABI
using namespace v3d;

extern "C" {

int ves3d_hip_direct_stokes_f64(const double *src, const double *den,
                                const double *qw, size_t src_stride,
                                size_t trg_stride, size_t n_surfs,
                                const double *trg, size_t head, size_t tail,
                                double *pot, ves3d_stream_t stream) {
  return vesicle_stokes<double, false>(src, nullptr, den, qw, src_stride, trg_stride,
                                       n_surfs, trg, head, tail, pot, (hipStream_t)stream);
}
int ves3d_hip_direct_stokes_f32(const float *src, const float *den,
                                const float *qw, size_t src_stride,
                                size_t trg_stride, size_t n_surfs,
                                const float *trg, size_t head, size_t tail,
                                float *pot, ves3d_stream_t stream) {
  return vesicle_stokes<float, false>(src, nullptr, den, qw, src_stride, trg_stride,
                                      n_surfs, trg, head, tail, pot, (hipStream_t)stream);
}
int ves3d_hip_direct_stokes_dl_f64(const double *src, const double *norm,
                                   const double *den, const double *qw,
                                   size_t src_stride, size_t trg_stride,
                                   size_t n_surfs, const double *trg,
                                   size_t head, size_t tail, double *pot,
                                   ves3d_stream_t stream) {
  return vesicle_stokes<double, true>(src, norm, den, qw, src_stride, trg_stride,
                                      n_surfs, trg, head, tail, pot, (hipStream_t)stream);
}
int ves3d_hip_direct_stokes_dl_f32(const float *src, const float *norm,
                                   const float *den, const float *qw,
                                   size_t src_stride, size_t trg_stride,
                                   size_t n_surfs, const float *trg,
                                   size_t head, size_t tail, float *pot,
                                   ves3d_stream_t stream) {
  return vesicle_stokes<float, true>(src, norm, den, qw, src_stride, trg_stride,
                                     n_surfs, trg, head, tail, pot, (hipStream_t)stream);
}

int ves3d_hip_stokes_all2all_f64(const double *src, const double *den,
                                 size_t np, double *pot, ves3d_stream_t stream) {
  return far_eval<false>(src, den, nullptr, np, src, pot, np, 0, 0, 0.0,
                         1.0 / kPi / 8.0, 0.0, (hipStream_t)stream);
}
int ves3d_hip_stokes_all2all_f32c(const double *src, const double *den,
                                  size_t np, double *pot, ves3d_stream_t stream) {
  return far_eval<true>(src, den, nullptr, np, src, pot, np, 0, 0, 0.0,
                        1.0 / kPi / 8.0, 0.0, (hipStream_t)stream);
}

int ves3d_hip_set_far_kernel(int kind) {
  if (kind < 0 || kind > 2) return VES3D_INVALID_PARAMETER;
  g_far_kind.store(kind);
  return VES3D_SUCCESS;
}


int ves3d_hip_direct_eval_f64(const double *src_pos, const double *sl_den,
                              const double *dl_den, size_t n_src,
                              const double *trg_pos, double *trg_vel,
                              size_t n_trg, size_t spg, size_t tpg,
                              ves3d_stream_t stream) {
  return far_eval<false>(src_pos, sl_den, dl_den, n_src, trg_pos, trg_vel, n_trg,
                         spg, tpg, kEvalEps2, 1.0 / (8.0 * kPi),
                         3.0 / (4.0 * kPi), (hipStream_t)stream);
}
int ves3d_hip_direct_eval_f32c(const double *src_pos, const double *sl_den,
                               const double *dl_den, size_t n_src,
                               const double *trg_pos, double *trg_vel,
                               size_t n_trg, size_t spg, size_t tpg,
                               ves3d_stream_t stream) {
  return far_eval<true>(src_pos, sl_den, dl_den, n_src, trg_pos, trg_vel, n_trg,
                        spg, tpg, kEvalEps2, 1.0 / (8.0 * kPi),
                        3.0 / (4.0 * kPi), (hipStream_t)stream);
}

}  // extern "C"
