// singular.hip -- rotations of SH coefficients to every grid point
// (RotateAll / RotateTranspose, src/SphericalHarmonics.cc:362-541), the
// singular self-interaction operator build (StokesSingularInteg_,
// :952-1180) and its per-vesicle application (the self term of
// StokesVelocity::operator(), src/StokesVelocity.cc:385-447).
//
// Rotation: the per-degree block products Bo[l] = Bi[l] * Mr[t][l] run as one
// grouped GEMM launch (descriptor per (t, l), batch over vesicles) on a
// degree-major copy of the coefficients; the longitude phase and the
// degree-major gather/scatter are separate elementwise kernels.
//
// Singular build, per chunk of vesicles:
//   Grid2SHC -> RotateAll -> SHC2Grid(p0 -> p1, +derivatives) & SHC2Pole
//   -> pole kernel (FP64) -> SHC2GridTranspose(p1 -> p0) -> RotateTranspose
//   -> rearrange -> Grid2SHC = [Nves][3 Ncoef][3 Ncoef]
// The FP64 build of 12 <= p1 <= 32 fuses the pole kernel with
// SHC2GridTranspose and RotateTranspose (k_pole_transpose), and the
// rearrangement with the last Grid2SHC (k_rearrange_g2s).  The FP32 form runs
// every GEMM stage in FP32 and keeps the pole kernel (singular weights, 1/r
// near the rotated pole) in FP64.  Both write the operator's (a, b) and
// (b, a) blocks equal (the rows of one symmetric tensor component), which
// the step's self apply relies on (k_self_apply_sym, k_self_apply_split).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "runtime.hpp"
#include "sht.hpp"

namespace v3d {

namespace {

std::mutex g_mu;
// The build's scratch (kWsSing0) is one per device: each build waits on its
// stream for the device's previous build, wherever that ran
struct BuildOrder {
  hipEvent_t done = nullptr;
  bool recorded = false;
};
std::map<int, BuildOrder> g_build_order;
// 1: the singular build's pole kernel runs fused with the transposed synthesis
// and rotation (k_pole_transpose) where its shapes allow; 0: as separate
// kernels (ves3d_hip_set_pole_kernel)
std::atomic<int> g_pole_fused{1};
struct RotPlan {
  GemmDesc *d;
  int n, tile;
};
std::map<std::tuple<int, int, int, int, long>, RotPlan> g_rplans;

// Grouped GEMM plan of the per-degree rotation products.
// transpose=false: RotateAll, rows (j, d) of vesicle v, output slab t.
// transpose=true : RotateTranspose, rows (j, d) of (v, t), Mr read transposed.
const RotPlan *rot_plan(int p, int dof, bool transpose,
                                           const RotMatsHost &h) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_mu);
  auto key = std::make_tuple(dev, p, dof, (int)transpose, 0L);
  auto it = g_rplans.find(key);
  if (it != g_rplans.end()) return &it->second;
  const long Ncoef = sh_ncoef(p);
  const long slab = (long)p * dof * Ncoef;  // one (v, t) slab
  std::vector<GemmDesc> v;
  for (int t = 0; t <= p; ++t)
    for (int l = 0; l <= p; ++l) {
      GemmDesc d{};
      const int len = h.len[l];
      d.M = p * dof;
      d.N = len;
      d.K = len;
      d.a_rs = Ncoef;
      d.a_cs = 1;
      d.b_off = h.off[t * (p + 1) + l];
      d.b_rs = transpose ? 1 : len;
      d.b_cs = transpose ? len : 1;
      d.b_bs = 0;
      d.c_rs = Ncoef;
      d.c_cs = 1;
      if (!transpose) {
        d.a_off = h.doff[l];
        d.a_bs = slab;
        d.c_off = t * slab + h.doff[l];
        d.c_bs = (p + 1) * slab;
      } else {
        d.a_off = t * slab + h.doff[l];
        d.a_bs = (p + 1) * slab;
        d.c_off = t * slab + h.doff[l];
        d.c_bs = (p + 1) * slab;
      }
      v.push_back(d);
    }
  GemmDesc *dd = upload_descs(v.data(), (int)v.size());
  if (!dd) return nullptr;
  return &(g_rplans[key] = RotPlan{dd, (int)v.size(), gemm_pick_tile(v.data(), (int)v.size())});
}

template <typename T>
const T *rot_ptr(const RotMatsDev *r);
template <>
const double *rot_ptr<double>(const RotMatsDev *r) { return r->d64; }
template <>
const float *rot_ptr<float>(const RotMatsDev *r) { return r->d32; }

// The four coefficient permutation kernels below run one wavefront per row
// of Ncoef coefficients (four rows per 256-thread block): the row's indices
// are decomposed once per wavefront, lanes stride over the row, and the
// permuted reads stay inside one row (L1-resident).

// B0p[v][j][d][pos] = phase_j(S0[v][d])[perm[pos]] with exp(-i k j pi / p)
// (src/SphericalHarmonics.cc:398-418); phase[j][k] = (cos, sin)(k j pi / p).
// Rows: (v, j, d).
template <typename T>
__global__ __launch_bounds__(256) void k_rot_phase_gather(
    const T *__restrict__ S0, long rows, int p, int dof, int ncoef,
    const int *__restrict__ perm, const int *__restrict__ partner,
    const int *__restrict__ order, const int *__restrict__ is_sin,
    const double *__restrict__ phase, T *__restrict__ out) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int d = (int)(row % dof);
  const long r = row / dof;
  const int j = (int)(r % p);
  const long v = r / p;
  const T *s = S0 + (v * dof + d) * ncoef;
  T *o = out + row * ncoef;
  for (int pos = threadIdx.x & 63; pos < ncoef; pos += 64) {
    const int c = perm[pos];
    const int k = order[c];
    T val;
    if (k == 0 || k == p) {
      val = s[c];
    } else {
      const bool sn = is_sin[c];
      const T x0 = s[sn ? partner[c] : c], x1 = s[sn ? c : partner[c]];
      const double cv = phase[2 * (j * (p + 1) + k)], sv = phase[2 * (j * (p + 1) + k) + 1];
      const T r0 = (T)cv, r1 = (T)(-sv);
      val = sn ? x0 * r1 + x1 * r0 : x0 * r0 - x1 * r1;
    }
    o[pos] = val;
  }
}

// out[row][c] = in[row][iperm[c]]  (degree-major -> coefficient order)
template <typename T>
__global__ __launch_bounds__(256) void k_scatter_coef(const T *__restrict__ in, long rows,
                                                      int ncoef, const int *__restrict__ iperm,
                                                      T *__restrict__ out) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T *s = in + row * ncoef;
  T *o = out + row * ncoef;
  for (int c = threadIdx.x & 63; c < ncoef; c += 64) o[c] = s[iperm[c]];
}

// out[row][pos] = in[row][perm[pos]]  (coefficient order -> degree-major)
template <typename T>
__global__ __launch_bounds__(256) void k_gather_coef(const T *__restrict__ in, long rows,
                                                     int ncoef, const int *__restrict__ perm,
                                                     T *__restrict__ out) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T *s = in + row * ncoef;
  T *o = out + row * ncoef;
  for (int pos = threadIdx.x & 63; pos < ncoef; pos += 64) o[pos] = s[perm[pos]];
}

// out[v][t][j][d][c] = phase_j^+(in)[c] reading the degree-major input
// (src/SphericalHarmonics.cc:511-537).  Rows: (v, t, j, d).  tab[c] holds
// c's two degree-major sources, its order and its kind (copy, cos, sin), so
// each output takes one 16-byte table read before its data reads.
template <typename T, bool STAGED>
__global__ __launch_bounds__(256) void k_rot_scatter_phase(const T *__restrict__ in, long rows,
                                                           int p, int dof, int ncoef,
                                                           const int4 *__restrict__ tab,
                                                           const double *__restrict__ phase,
                                                           T *__restrict__ out) {
  // STAGED: the block's four input rows go through LDS with contiguous
  // reads, and the permuted reads hit LDS (rows up to kScatterStageBytes)
  extern __shared__ unsigned char rsp_smem[];
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const bool live = row < rows;
  const T *s = in + row * ncoef;
  if constexpr (STAGED) {
    T *srow = (T *)rsp_smem + (threadIdx.x >> 6) * ncoef;
    if (live)
      for (int c = threadIdx.x & 63; c < ncoef; c += 64) srow[c] = s[c];
    __syncthreads();
    s = srow;
  }
  if (!live) return;
  const int j = (int)((row / dof) % p);
  const double *ph = phase + 2L * j * (p + 1);
  T *o = out + row * ncoef;
  for (int c = threadIdx.x & 63; c < ncoef; c += 64) {
    const int4 e = tab[c];
    T val;
    if (e.w == 0) {
      val = s[e.x];
    } else {
      const T x0 = s[e.x], x1 = s[e.y];
      const T r0 = (T)ph[2 * e.z], r1 = (T)ph[2 * e.z + 1];
      val = e.w == 2 ? x0 * r1 + x1 * r0 : x0 * r0 - x1 * r1;
    }
    o[c] = val;
  }
}

// Largest LDS staging of four rows (the rotation scatter at p <= 31 in FP64).
constexpr size_t kScatterStageBytes = 32768;

// Blocks of four rows.
inline unsigned row_blocks(long rows) { return (unsigned)((rows + 3) / 4); }

inline unsigned grid_for(long n) {
  long b = (n + 255) / 256;
  if (b > 65536L * 16) b = 65536L * 16;
  return (unsigned)(b < 1 ? 1 : b);
}

}  // namespace

// RotateAll: S [Nv*dof][Ncoef] -> out [Nv][p+1][p][dof][Ncoef]; work: Nv*p*dof*Ncoef
// + Nv*(p+1)*p*dof*Ncoef elements.
template <typename T>
int rotate_all(const T *S, long Nv, int p, int dof, T *out, T *work, hipStream_t st) {
  const RotMatsDev *r = rot_mats(p);
  if (!r) return VES3D_MEMORY_ERROR;
  const auto *pl = rot_plan(p, dof, false, *r->h);
  if (!pl) return VES3D_MEMORY_ERROR;
  const int nc = sh_ncoef(p);
  T *B0p = work;
  T *S1p = work + Nv * p * dof * (long)nc;
  const long rows0 = Nv * p * (long)dof;
  const long rows = Nv * (p + 1) * (long)p * dof;
  if (rows / 4 >= 0x7fffffffL) return VES3D_INVALID_PARAMETER;
  k_rot_phase_gather<T><<<row_blocks(rows0), 256, 0, st>>>(
      S, rows0, p, dof, nc, r->perm, r->partner, r->order, r->is_sin, r->phase, B0p);
  V3D_CHECK(launch_status());
  V3D_CHECK(gemm_grouped<T>(pl->d, pl->n, (int)Nv, p * dof, 2 * p, B0p,
                            rot_ptr<T>(r), S1p, T(1), T(0), st, pl->tile));
  k_scatter_coef<T><<<row_blocks(rows), 256, 0, st>>>(S1p, rows, nc, r->iperm, out);
  return launch_status();
}

// RotateTranspose: in/out [Nv][p+1][p][dof][Ncoef]; work: 2 * that size.
template <typename T>
int rotate_transpose(const T *in, long Nv, int p, int dof, T *out, T *work, hipStream_t st) {
  const RotMatsDev *r = rot_mats(p);
  if (!r) return VES3D_MEMORY_ERROR;
  const auto *pl = rot_plan(p, dof, true, *r->h);
  if (!pl) return VES3D_MEMORY_ERROR;
  const int nc = sh_ncoef(p);
  const long rows = Nv * (p + 1) * (long)p * dof;
  if (rows / 4 >= 0x7fffffffL) return VES3D_INVALID_PARAMETER;
  T *Bp = work + rows * nc;
  k_gather_coef<T><<<row_blocks(rows), 256, 0, st>>>(in, rows, nc, r->perm, work);
  V3D_CHECK(launch_status());
  V3D_CHECK(gemm_grouped<T>(pl->d, pl->n, (int)Nv, p * dof, 2 * p, work,
                            rot_ptr<T>(r), Bp, T(1), T(0), st, pl->tile));
  const size_t stage = 4 * nc * sizeof(T);
  if (stage <= kScatterStageBytes)
    k_rot_scatter_phase<T, true><<<row_blocks(rows), 256, stage, st>>>(
        Bp, rows, p, dof, nc, (const int4 *)r->scatter, r->phase, out);
  else
    k_rot_scatter_phase<T, false><<<row_blocks(rows), 256, 0, st>>>(
        Bp, rows, p, dof, nc, (const int4 *)r->scatter, r->phase, out);
  return launch_status();
}

// ------------------------------------------------------------- pole kernel
// For each rotation r, pole t (0: x=-1, 1: x=+1) and upsampled source s:
// the 6 symmetric tensor components of the SL (and/or DL) kernel times the
// singular quadrature weight (src/SphericalHarmonics.cc:970-1073).  One
// thread per (r, s) serves both poles, so the rotated geometry (X, X_theta,
// X_phi: 72 bytes in FP64) is read once for the two 48-byte outputs.
template <typename T>
__global__ void k_pole_kernel(const T *__restrict__ X, const T *__restrict__ Xt,
                              const T *__restrict__ Xp, const T *__restrict__ trg,
                              const double *__restrict__ qw, long nrot, int p1,
                              T *__restrict__ SL0, T *__restrict__ DL0) {
  const int M1 = 2 * p1 * (p1 + 1);
  const long total = nrot * (long)M1;
  const double eps = 2.220446049250313e-16;
  const double csl = 1.0 / (8.0 * kPi), cdl = 3.0 / (4.0 * kPi);
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long)gridDim.x * blockDim.x) {
    const int s = (int)(i % M1);
    const long r = i / M1;
    const int j0 = s / (2 * p1);
    const long b = r * 3 * (long)M1 + s;
    const double x0 = X[b], y0 = X[b + M1], z0 = X[b + 2 * M1];
    const double xt = Xt[b], yt = Xt[b + M1], zt = Xt[b + 2 * M1];
    const double xp = Xp[b], yp = Xp[b + M1], zp = Xp[b + 2 * M1];
    const double nx = yt * zp - zt * yp, ny = zt * xp - xt * zp, nz = xt * yp - yt * xp;
    const double area = SL0 ? sqrt(nx * nx + ny * ny + nz * nz) : 0.0;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const double w = qw[t ? j0 : p1 - j0];
      const double dx = trg[(r * 3 + 0) * 2 + t] - x0, dy = trg[(r * 3 + 1) * 2 + t] - y0,
                   dz = trg[(r * 3 + 2) * 2 + t] - z0;
      const double r2 = dx * dx + dy * dy + dz * dz;
      double rinv = 1.0 / sqrt(r2);
      if (r2 <= eps) rinv = 0;
      const double rinv2 = rinv * rinv;
      const double dd[6] = {dx * dx, dx * dy, dx * dz, dy * dy, dy * dz, dz * dz};
      const long o = ((2 * r + t) * 6) * (long)M1 + s;
      if (DL0) {
        const double rn5 = cdl * w * (nx * dx + ny * dy + nz * dz) * rinv2 * rinv2 * rinv;
#pragma unroll
        for (int c = 0; c < 6; ++c) DL0[o + c * (long)M1] = (T)(dd[c] * rn5);
      }
      if (SL0) {
        const double ar = csl * w * area * rinv;
        const double ar2 = ar * rinv2;
#pragma unroll
        for (int c = 0; c < 6; ++c)
          SL0[o + c * (long)M1] = (T)(dd[c] * ar2 + ((c == 0 || c == 3 || c == 5) ? ar : 0.0));
      }
    }
  }
}

// 1/sqrt(x), x > 0: the hardware estimate and one third-order step (as
// rsqrt_pair of the direct sums).
__device__ __forceinline__ double rsqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(y * -x, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// The pole kernel fused with SHC2GridTranspose(p1 -> p0) of its values:
// K1[r][t*6+c][k] = sum over the grid (lat, lon) of the kernel value of
// rotation r, pole t, tensor component c at (lat, lon), times MatFourier(p0,
// p1)[jj][lon] (the Fourier stage) and MatLegendre(p0, p1)[m][n][lat] (the
// Legendre stage), k = blockoff(p0, jj) + n, m = (jj + 1) / 2 -- the products
// the two grouped GEMMs of sht_shc2grid_transpose form, without the kernel
// values (12 functions on the upsampled grid per rotation) or the Fourier
// stage's output passing through HBM -- and K2 = RotateTranspose of the rows
// (src/SphericalHarmonics.cc:451-541), which is what leaves.
// Both tables have a mirror symmetry: MatFourier of order m at lon + pi is
// (-1)^m of that at lon, and MatLegendre of degree n and order m at the
// latitude P1 - lat is (-1)^(n-m) of that at lat.  So the sums and differences
// of the values at the four mirror points (lat or P1 - lat, lon or lon + pi)
// serve one parity of m and of n - m each, with a quarter of the products.
// Persistent workgroups walk the rotations r = blockIdx.x + i gridDim.x and,
// within a rotation, the latitude pairs (lat, P1 - lat), two per pass up to P1 =
// 16 (331 vesicles of order 7, single layer, the whole build: 982 -> 901 us):
//   1. four lanes evaluate pole t's 6 kernel values at the four mirror points
//      of (lat, lon < P1), form the four combinations by lane swaps and store
//      them in Kv[n - m parity][m parity][lon][t * 6 + q] (kPtKs doubles per
//      point, an odd stride, the four parts kPtPad further apart);
//   2. wave (n - m parity, m parity) forms T[n - m parity][c][jj] = sum_lon
//      Kv[..][lon][c] Mf[lon][jj] over its P0 columns jj on
//      v_mfma_f64_16x16x4f64 (lane l: A(l % 16, l / 16), B(l / 16, l % 16),
//      results at rows l / 16 + 4 i, column l % 16; rows c >= 12 are not used),
//      its columns of MatFourier in registers for the whole kernel;
//   3. thread (6 components, 3 degrees of one parity of a frequency jj) adds
//      T[parity][c][jj] times the pair's Legendre values into its 6 x 3
//      accumulators (FP64 registers).
// One barrier per pass: Kv and T have two buffers, and stage 3 runs a pass
// late, beside stage 2's matrix products.  Each thread loads the geometry and
// the Legendre values (which lie by latitude, degree and triple: consecutive
// words for the lanes of a wave) of its next pass while the current one runs.
// At a rotation's end the accumulators go to LDS (over Kv and T) as 12
// degree-major rows (dpos: the place of each coefficient), the waves form the
// per-degree products with the rotation's blocks on v_mfma_f64_16x16x4f64 (12
// of 16 rows used, the others are whatever follows; the blocks lie in `frag` in operand order, 512 contiguous
// bytes per load), and a thread per coefficient applies the longitude phase to
// the 12 rows and stores them.
// Bound: the geometry's reads (72 bytes per point, 2.7 TB/s at p0 = 16) beside
// FP64 issue, matrix and vector, where three workgroups of one wave per SIMD
// each run at a time: 1.9 ms per 104 vesicles and layer at p0 = 16, 1.3 ms
// without the reads; leaving out any of the other stages changes little.
// Workgroups of 384 threads on three latitudes, without the mirror sums, took
// 3.7 ms: at 168 VGPRs two of them per CU would have needed 3 waves on every
// SIMD, the dispatcher places 2, 2, 1, 1 of each, so one ran at a time.
// With rotation products and phases as passes of their own 1.55 GB per 104
// vesicles were written and read again, 0.8 ms.
constexpr int kPtKs = 13;
constexpr int kPtPad = 4;
constexpr int kPtThreads = 256;
// Latitude pairs per pass: half a circle of at most 16 longitudes leaves half the
// lanes of one pair's waves without a point.
__host__ __device__ constexpr int pole_pairs(int p1) { return p1 <= 16 ? 2 : 1; }
// Doubles of one mirror combination's values.
__host__ __device__ constexpr int pole_kv_part(int p1) { return p1 * kPtKs + kPtPad; }
// Degree l's rotation block in operand order: 4 loads of 64 doubles (one tile
// of 16 columns, 16 entries) for the nsmall degrees of at most 16 entries, 16
// loads (two tiles of 16 columns, 32 entries) for the others.
__host__ __device__ inline int rot_frag_off(int l, int nsmall) {
  return l < nsmall ? 256 * l : 256 * nsmall + 1024 * (l - nsmall);
}

// Degrees of a block of len degrees with parity par of n - m, and its triples.
__host__ __device__ inline int pole_degrees(int len, int par) { return (len + 1 - par) / 2; }
__host__ __device__ inline int pole_block_triples(int len) {
  return (pole_degrees(len, 0) + 2) / 3 + (pole_degrees(len, 1) + 2) / 3;
}
// Degree triples of the orders before m (blocks of p0 + 1 - m degrees).
__host__ __device__ inline int pole_triples(int p0, int m) {
  int n = 0;
  for (int i = 0; i < m; ++i) n += pole_block_triples(p0 + 1 - i);
  return n;
}
// Threads of the Legendre role: two component halves of every frequency's
// triples (two frequencies for the orders 1 .. p0 - 1).
inline int pole_legendre_threads(int p0) {
  return 2 * (2 * pole_triples(p0, p0 + 1) - pole_triples(p0, 1) - 1);
}

// LDS doubles of k_pole_transpose: Kv and T, which the rotation's rows share.
__host__ __device__ inline long pole_lds_doubles(int p0, int p1) {
  const int kt = 2 * pole_pairs(p1) * (4 * pole_kv_part(p1) + 2 * 12 * p1), st = 12 * (p0 * (p0 + 2) + 1);
  return kt > st ? kt : st;
}

// a and b become a + b and a - b after the odd rows of 16 lanes (kRows == 16)
// or the upper half wave (32) of a have changed places with the even rows or
// the lower half of b: the even lanes hold the sum and the difference of a's
// mirror values, the odd ones of b's.
template <int kRows>
__device__ __forceinline__ void mirror_sums(double &a, double &b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto swap = [](unsigned u, unsigned v) {
    if constexpr (kRows == 16)
      return __builtin_amdgcn_permlane16_swap(u, v, false, false);
    else
      return __builtin_amdgcn_permlane32_swap(u, v, false, false);
  };
  const auto lo = swap((unsigned)x, (unsigned)y);
  const auto hi = swap((unsigned)(x >> 32), (unsigned)(y >> 32));
  const double u = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
  const double v = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
  a = u + v;
  b = u - v;
}

template <int P1>
__global__ __launch_bounds__(kPtThreads, 3) void k_pole_transpose(
    const double *__restrict__ X, const double *__restrict__ Xt, const double *__restrict__ Xp,
    const double *__restrict__ trg, const double *__restrict__ qw, long nrot, int p0,
    const double *__restrict__ mft, const double *__restrict__ mlt, int layer,
    const int *__restrict__ dpos, const double *__restrict__ frag, long frag_t,
    int nsmall, const int4 *__restrict__ sources,
    const double *__restrict__ phase, double *__restrict__ K2) {
  typedef double v4d __attribute__((ext_vector_type(4)));
  static_assert(P1 % 2 == 0 && 8 * P1 <= kPtThreads);
  constexpr int L = 2 * P1, Nlat = P1 + 1, NP = P1 / 2 + 1, M1 = L * Nlat, KS = (P1 + 3) / 4;
  constexpr int kPart = pole_kv_part(P1), PP = pole_pairs(P1), NS = (NP + PP - 1) / PP;
  extern __shared__ double lds[];
  const int F = 2 * p0, Nc = p0 * (p0 + 2);
  const int ntri = pole_triples(p0, p0 + 1);
  double *Kv = lds;                                // [buffer][pair][2][2][P1][kPtKs]
  double *Ts = Kv + 8 * PP * kPart;                // [buffer][pair][2][12][P1]
  double *St = lds;                                // [12][Nc + 1], over Kv and Ts
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  // kernel-value role: pole t (the wave's) at longitude j + half P1 of the
  // pair's row; 16 lanes read 16 consecutive longitudes.  (With the four mirror
  // points in a lane quad every four lanes of a load touch four lines: 2.7 ms
  // instead of 1.9.)
  constexpr int kBlocks = (P1 + 15) / 16;  // longitude blocks of half a circle
  const int uwv = __builtin_amdgcn_readfirstlane(wv);
  const int row = (tid >> 4) & 1, half = (tid >> 5) & 1;
  const int t = (uwv / kBlocks) & 1, j = 16 * (uwv % kBlocks) + (tid & 15);
  const int pr = PP == 2 ? uwv >> 1 : 0;  // the pass's pair
  const bool kvt = j < P1;
  // Fourier role: the columns of order parity tile from the row combination frow
  const int frow = wv >> 1, tile = wv & 1;
  const int li = lane & 15, lk = lane >> 4;
  // the wave's output column for lane li (-1: a padding column)
  int fcol = -1;
  for (int cc = 0, seen = 0; cc < F; ++cc)
    if ((((cc + 1) / 2) & 1) == tile) {
      if (seen == li) fcol = cc;
      ++seen;
    }
  double mf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    mf[s] = fcol >= 0 && 4 * s + lk < P1 ? mft[(long)fcol * L + 4 * s + lk] : 0.0;
  // Legendre role: components c .. c + 5 and the degrees m + par + 2 (3 q + n)
  // of frequency row jj of the order-p0 layout, whose block starts at off
  // (after block 0 of length p0 + 1, the blocks of order m' = 1 .. p0 come in
  // pairs of length p0 + 1 - m').  Lanes take the triples of all cosine rows,
  // then those of the sine rows (m = 1 .. p0 - 1).
  const int ntri1 = pole_triples(p0, 1);
  const int nrow = 2 * ntri - ntri1 - 1;
  const bool lt = tid < 2 * nrow;
  const int c = lt ? tid / nrow * 6 : 0;
  const int tr = lt ? tid % nrow : 0;
  const bool sine = tr >= ntri;
  const int tm = sine ? tr - ntri + ntri1 : tr;  // triple within the table
  int m = 0, q = tm;
  while (q >= pole_block_triples(p0 + 1 - m)) q -= pole_block_triples(p0 + 1 - m++);
  const int len = p0 + 1 - m, even = (pole_degrees(len, 0) + 2) / 3;
  const int par = q >= even ? 1 : 0;
  const int d0 = par + 6 * (q - par * even);  // first degree less m
  const int jj = m == 0 ? 0 : 2 * m - (sine ? 0 : 1);
  const int off = jj == 0 ? 0 : (p0 + 1) + 2 * ((m - 1) * (p0 + 1) - (m - 1) * m / 2) +
                                    (sine ? p0 + 1 - m : 0);
  int dp[3];  // the places of the thread's coefficients
#pragma unroll
  for (int n = 0; n < 3; ++n) dp[n] = lt && d0 + 2 * n < len ? dpos[off + d0 + 2 * n] : -1;
  const double eps = 2.220446049250313e-16;
  // geometry, pole and Legendre values of the next (rotation, pass), loaded by
  // every thread at indices in range: unconditional loads leave no value to
  // merge after a branch, so nothing waits for them before their use.  The
  // rotation's base is uniform, the place in it 32 bits.
  double g[9], tg[3], w, ml[PP][3];
  const unsigned place = 8 * ((row ? P1 * L : 0) + half * P1 + min(j, P1 - 1)),
                 wplace = 8 * (2 * row + t);
  const int step = row ? -8 * L : 8 * L;
  auto at = [](const double *base, unsigned bytes) {
    typedef const char __attribute__((address_space(1))) gchar;
    typedef const double __attribute__((address_space(1))) gdouble;
    gchar *b = (gchar *)base;
    asm("" : "+s"(b));  // a scalar base and a 32-bit place, not 64-bit vector sums
    return *(gdouble *)(b + bytes);
  };
  auto load = [&](long r_, int g_) {
    const long rc = r_ < nrot ? r_ : nrot - 1;
    const int lp = min(g_ * PP + pr, NP - 1);
    const unsigned o = place + lp * step;
    const double *x = X + rc * 3 * M1, *xt = Xt + rc * 3 * M1, *xp = Xp + rc * 3 * M1;
    g[0] = at(x, o); g[1] = at(x + M1, o); g[2] = at(x + 2 * M1, o);
    g[3] = at(xt, o); g[4] = at(xt + M1, o); g[5] = at(xt + 2 * M1, o);
    g[6] = at(xp, o); g[7] = at(xp + M1, o); g[8] = at(xp + 2 * M1, o);
    w = at(qw + 4 * lp, wplace);
    if (PP > 1 && g_ * PP + pr >= NP) w = 0.0;  // past the last pair
  };
  auto load_pole = [&](long r_) {
    const long rc = r_ < nrot ? r_ : nrot - 1;
    for (int d = 0; d < 3; ++d) tg[d] = at(trg + (rc * 3 + d) * 2 + t, 0);
  };
  const unsigned mplace = 8 * tm;
  auto load_ml = [&](int g_) {
#pragma unroll
    for (int u = 0; u < PP; ++u)
      for (int n = 0; n < 3; ++n)
        ml[u][n] = at(mlt + (min(g_ * PP + u, NP - 1) * 3 + n) * ntri, mplace);
  };
  load(blockIdx.x, 0);
  load_pole(blockIdx.x);
  for (long r = blockIdx.x; r < nrot; r += gridDim.x) {
    double acc[6][3] = {};
    double f[PP][6];
    auto load_t = [&](int g_) {
#pragma unroll
      for (int u = 0; u < PP; ++u) {
        const double *tc = Ts + (((g_ & 1) * PP + u) * 24 + par * 12 + c) * P1 + jj;
#pragma unroll
        for (int i = 0; i < 6; ++i) f[u][i] = tc[i * P1];
      }
    };
    auto legendre = [&] {
#pragma unroll
      for (int u = 0; u < PP; ++u)
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
          for (int n = 0; n < 3; ++n) acc[i][n] = fma(f[u][i], ml[u][n], acc[i][n]);
    };
#pragma unroll 1
    for (int gi = 0; gi < NS; ++gi) {
      {
        const double yt = g[4], zt = g[5], xt = g[3], xp = g[6], yp = g[7], zp = g[8];
        const double nx = yt * zp - zt * yp, ny = zt * xp - xt * zp, nz = xt * yp - yt * xp;
        const double dx = tg[0] - g[0], dy = tg[1] - g[1], dz = tg[2] - g[2];
        const double wt = w;
        const bool more = gi + 1 < NS;
        load(more ? r : r + gridDim.x, more ? gi + 1 : 0);
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double rinv = r2 <= eps ? 0.0 : rsqrt_refined(r2);
        const double rinv2 = rinv * rinv;
        const double dd[6] = {dx * dx, dx * dy, dx * dz, dy * dy, dy * dz, dz * dz};
        double val, diag = 0.0;
        if (layer == 1) {
          val = wt * (nx * dx + ny * dy + nz * dz) * rinv2 * rinv2 * rinv;
        } else {
          const double n2 = nx * nx + ny * ny + nz * nz;
          const double area = n2 > 0.0 ? n2 * rsqrt_refined(n2) : 0.0;
          diag = wt * area * rinv;
          val = diag * rinv2;
        }
        double v[6];
#pragma unroll
        for (int i = 0; i < 6; ++i)
          v[i] = (i == 0 || i == 3 || i == 5) ? fma(dd[i], val, diag) : dd[i] * val;
        // v[2 q], v[2 q + 1]: first the rows' sum and difference of component
        // 2 q + row, then the sums and differences over the half circles of
        // the rows' combination half
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          mirror_sums<16>(v[2 * q], v[2 * q + 1]);
          mirror_sums<32>(v[2 * q], v[2 * q + 1]);
        }
        if (kvt) {
          double *kv = Kv + (((gi & 1) * PP + pr) * 4 + 2 * half) * kPart + j * kPtKs + t * 6 + row;
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            kv[2 * q] = v[2 * q];
            kv[kPart + 2 * q] = v[2 * q + 1];
          }
        }
      }
      __syncthreads();  // Kv and the previous pass's T are in
      {
        // (the rows c >= 12 of A are other values; what they give is not read)
        const double *kv = Kv + ((gi & 1) * PP * 4 + wv) * kPart + li;
        v4d d[2] = {};  // two accumulation chains: the pairs', or the steps' halves
        double a[PP][KS];
#pragma unroll
        for (int u = 0; u < PP; ++u)
#pragma unroll
          for (int s = 0; s < KS; ++s)
            a[u][s] = kv[u * 4 * kPart + min(4 * s + lk, P1 - 1) * kPtKs];
        if (gi > 0) load_t(gi - 1);
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int u = 0; u < PP; ++u) {
            v4d &e = d[PP == 2 ? u : s & 1];
            e = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][s], mf[s], e, 0, 0, 0);
          }
        if (gi > 0) legendre();
        load_ml(gi);
        if (PP == 1) d[0] += d[1];
        if (fcol >= 0) {
#pragma unroll
          for (int u = 0; u < PP; ++u) {
            double *o = Ts + (((gi & 1) * PP + u) * 24 + frow * 12 + lk) * P1 + fcol;
#pragma unroll
            for (int i = 0; i < 3; ++i) o[4 * i * P1] = d[u][i];
          }
        }
      }
    }
    __syncthreads();  // the last T is in
    load_t(NS - 1);
    legendre();
    // the rotation's 12 rows, degree-major.  (The thread's index is opaque from
    // here on: what is derived from it is not kept in registers over the passes.)
    int id = tid, cc = c;
    asm("" : "+v"(id), "+v"(cc));
    const int lane = id & 63, li = lane & 15, lk = lane >> 4;
    const unsigned v_rot = (unsigned)r / p0;  // rotations of a launch fit 32 bits
    const double *fr = frag + v_rot % (p0 + 1) * frag_t + lane;
    double op[16];
    auto operand = [&](int l) {
      const double *f = fr + rot_frag_off(l, nsmall);
      if (l < nsmall) {
#pragma unroll
        for (int k = 0; k < 4; ++k) op[k] = f[64 * k];
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) op[k] = f[64 * k];
      }
    };
    load_pole(r + gridDim.x);
    __syncthreads();  // T is read
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      if (dp[n] < 0) continue;
      double *o = St + cc * (Nc + 1) + dp[n];
#pragma unroll
      for (int i = 0; i < 6; ++i) o[i * (Nc + 1)] = acc[i][n];
    }
    int l = p0 - wv;
    if (l >= 0) operand(l);
    __syncthreads();
    // per-degree products, in place: a degree's columns depend on its own
    // entries only, and one wave forms them all.  The waves take the degrees
    // from the longest down, back and forth; the next degree's operand is
    // loaded while the current one's results are stored.
#pragma unroll 1
    for (int i = 0; l >= 0; ++i) {
      const int n = min(2 * l + 1, 2 * p0);
      double *ro = St + l * l;  // the degree's first entry
      const double *av = ro + li * (Nc + 1);
      v4d e0 = {0.0, 0.0, 0.0, 0.0}, e1 = {0.0, 0.0, 0.0, 0.0};
      double a[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) a[k] = av[min(4 * k + lk, n - 1)];  // the operand's zeros past n
      if (l < nsmall) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          e0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], op[k], e0, 0, 0, 0);
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          e0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], op[k], e0, 0, 0, 0);
          e1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], op[8 + k], e1, 0, 0, 0);
        }
      }
      constexpr int nw = kPtThreads / 64;
      l = p0 - (i + 1) * nw - (i & 1 ? wv : nw - 1 - wv);
      if (l >= 0) operand(l);
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        double *o = ro + (lk + 4 * u) * (Nc + 1) + li;
        if (li < n) o[0] = e0[u];
        if (16 + li < n) o[16] = e1[u];
      }
    }
    __syncthreads();
    // longitude phases, in coefficient order
    for (int k = id; k < Nc; k += kPtThreads) {
      const int4 src = sources[k];
      const double *ph = phase + 2 * (((unsigned)r % p0) * (p0 + 1) + src.z);
      // a copy, cosine: x0 r0 - x1 r1, sine: x0 r1 + x1 r0
      const double r0 = ph[0], r1 = ph[1];
      const double w0 = src.w == 0 ? 1.0 : (src.w == 2 ? r1 : r0);
      const double w1 = src.w == 0 ? 0.0 : (src.w == 2 ? r0 : -r1);
      double *o = K2 + r * 12 * (long)Nc + k;
#pragma unroll 4
      for (int i = 0; i < 12; ++i)
        o[i * Nc] = St[i * (Nc + 1) + src.x] * w0 + St[i * (Nc + 1) + src.y] * w1;
    }
    __syncthreads();  // St read before the next rotation's kernel values
  }
}

// M1arr[v][a*Ncoef+k][b][lat][lon] from K2[v][j1][j2][t2*6+c][k]
// (src/SphericalHarmonics.cc:1090-1131): t2=0 pole -> grid (j1, j2),
// t2=1 pole -> grid (p0-j1, p0+j2); c = sym(a, b).  For fixed (v, a, b) this
// is a transpose between k (contiguous in K2) and the grid point g
// (contiguous in M1arr): a block moves a 32 (k) x 64 (g) tile through LDS so
// that both the reads and the writes are whole contiguous runs.
constexpr int kRaK = 32, kRaG = 64;
template <typename T>
__global__ __launch_bounds__(256) void k_singular_rearrange(const T *__restrict__ K2, long Nv,
                                                            int p0, T *__restrict__ M1) {
  __shared__ T tile[kRaG][kRaK + 1];
  const int Ncoef = p0 * (p0 + 2), Ngrid = 2 * p0 * (p0 + 1);
  const int tk = (Ncoef + kRaK - 1) / kRaK, tg = (Ngrid + kRaG - 1) / kRaG;
  long bid = blockIdx.x;
  const int gt = (int)(bid % tg);
  bid /= tg;
  const int kt = (int)(bid % tk);
  bid /= tk;
  const int ab = (int)(bid % 9);
  const long v = bid / 9;
  if (v >= Nv) return;
  const int a = ab / 3, b = ab % 3;
  const int lo = a < b ? a : b, hi = a < b ? b : a;
  const int c = lo == 0 ? hi : (lo == 1 ? 2 + hi : 5);
  const int k0 = kt * kRaK, g0 = gt * kRaG;
  const int t = threadIdx.x;
#pragma unroll
  for (int q = 0; q < (kRaK * kRaG) / 256; ++q) {
    const int kk = t % kRaK, gg = t / kRaK + q * (256 / kRaK);
    const int g = g0 + gg, k = k0 + kk;
    T val = T(0);
    if (g < Ngrid && k < Ncoef) {
      const int lat = g / (2 * p0), lon = g % (2 * p0);
      int j1, j2, t2;
      if (lon < p0) {
        j1 = lat; j2 = lon; t2 = 0;
      } else {
        j1 = p0 - lat; j2 = lon - p0; t2 = 1;
      }
      val = K2[((((v * (p0 + 1) + j1) * (long)p0 + j2) * 12 + t2 * 6 + c) * (long)Ncoef) + k];
    }
    tile[gg][kk] = val;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < (kRaK * kRaG) / 256; ++q) {
    const int gg = t % kRaG, kk = t / kRaG + q * (256 / kRaG);
    const int g = g0 + gg, k = k0 + kk;
    if (g < Ngrid && k < Ncoef)
      M1[(((v * 3 + a) * (long)Ncoef + k) * 3 + b) * Ngrid + g] = tile[gg][kk];
  }
}

// The rearrangement above and Grid2SHC(p0 -> p0) of its rows in one pass
// (FP64, p0 <= 16): out[v][a Nc + k][b Nc + c] = Grid2SHC of the grid function
// M1(v, a, k, b)[lat][lon] that k_singular_rearrange writes (the same K2
// element per grid point), then the Fourier and Legendre stages of
// sht_grid2shc (src/SphericalHarmonics.cc:151-235).  M1(v, a, k, b) depends on
// (a, b) only through the symmetric tensor component c6(a, b), so a workgroup
// takes (v, c6) and kRgK consecutive k and writes the rows of (a, b) and
// (b, a).  In rounds of four latitudes, wave w forms
//   Fs[w][k][j] = sum_lon M1(k)[lat][lon] MatFourierInv[lon][j],  lat = l0 + w,
// on v_mfma_f64_16x16x4f64 (lane l: A(l % 16, l / 16), B(l / 16, l % 16),
// results at rows l / 16 + 4 i, column l % 16), its A operand read from K2
// (16 consecutive k of one grid point: a 128-byte run per 16 lanes, the next
// round's loaded during this one) and MatFourierInv in registers; after a
// barrier every thread adds the round's Legendre terms
//   Fs[u][k][j_c] MatLegendreInv[m_c][lat][n_c]
// to its outputs (k, c), k = k0 + wave + 4 r, c = lane + 64 q.  Neither the
// rearranged grid values nor the Fourier sums pass through HBM.
constexpr int kRgK = 16;
constexpr int kRgMl = 17 * 153;  // MatLegendreInv doubles at p0 = 16
__global__ __launch_bounds__(256, 3) void k_rearrange_g2s(const double *__restrict__ K2,
                                                          long Nv, int p0,
                                                          const double *__restrict__ mfinv,
                                                          const double *__restrict__ mlinv,
                                                          double *__restrict__ out) {
  typedef double v4d __attribute__((ext_vector_type(4)));
  __shared__ double Fs[4][kRgK][33];
  __shared__ double Ml[kRgMl];
  const int Nc = p0 * (p0 + 2), Nlat = p0 + 1, L = 2 * p0;
  const int nml = Nlat * (p0 + 1) * (p0 + 2) / 2;
  const int nkt = (Nc + kRgK - 1) / kRgK;
  long bid = blockIdx.x;
  const int kt = (int)(bid % nkt);
  bid /= nkt;
  const int c6 = (int)(bid % 6);  // xx, xy, xz, yy, yz, zz
  const long v = bid / 6;
  if (v >= Nv) return;
  const int a = c6 < 3 ? 0 : (c6 < 5 ? 1 : 2), b = c6 < 3 ? c6 : (c6 < 5 ? c6 - 2 : 2);
  const int k0 = kt * kRgK;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  for (int i = tid; i < nml; i += 256) Ml[i] = mlinv[i];
  // B operand: MatFourierInv[lon = 4 s + lk][j = 16 ct + li]
  double bf[2][8];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int lon = 4 * s + lk, j = 16 * ct + li;
      bf[ct][s] = (lon < L && j < L) ? mfinv[lon * L + j] : 0.0;
    }
  // outputs c = lane + 64 q: block column j, MatLegendreInv offset of (m, n)
  // at latitude 0, and the block's row length (degrees)
  int cj[5], cb[5], cl[5];
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const int c = lane + 64 * q;
    cj[q] = -1;
    cb[q] = 0;
    cl[q] = 0;
    for (int jj = 0, off = 0; jj < L && c < Nc; ++jj) {
      const int m = (jj + 1) / 2, len = p0 + 1 - m;
      if (c < off + len) {
        cj[q] = jj;
        cl[q] = len;
        cb[q] = Nlat * (m * (p0 + 1) - m * (m - 1) / 2) + (c - off);
        break;
      }
      off += len;
    }
  }
  double acc[4][5];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int q = 0; q < 5; ++q) acc[r][q] = 0.0;
  const double *kv2 = K2 + v * (long)(p0 + 1) * p0 * 12 * Nc;
  const int kk = k0 + li;
  const bool kvalid = kk < Nc;
  // A operand of latitude lat: M1(kk)[lat][4 s + lk]
  double xa[8];
  auto load = [&](int lat) {
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int lon = 4 * s + lk;
      double x = 0.0;
      if (kvalid && lon < L && lat < Nlat) {
        const bool t2 = lon >= p0;
        const int j1 = t2 ? p0 - lat : lat, j2 = t2 ? lon - p0 : lon;
        x = kv2[(((long)j1 * p0 + j2) * 12 + (t2 ? 6 : 0) + c6) * Nc + kk];
      }
      xa[s] = x;
    }
  };
  load(w);
  __syncthreads();  // Ml in
  for (int l0 = 0; l0 < Nlat; l0 += 4) {
    if (l0 + w < Nlat) {
      v4d d0 = {0.0, 0.0, 0.0, 0.0}, d1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[s], bf[0][s], d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[s], bf[1][s], d1, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        Fs[w][lk + 4 * i][li] = d0[i];
        Fs[w][lk + 4 * i][16 + li] = d1[i];
      }
    }
    load(l0 + 4 + w);
    __syncthreads();  // the round's Fourier sums are in
    const int nu = min(4, Nlat - l0);
    for (int u = 0; u < nu; ++u) {
      const int lat = l0 + u;
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        if (cj[q] < 0) continue;
        const double ml = Ml[cb[q] + lat * cl[q]];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r][q] += Fs[u][w + 4 * r][cj[q]] * ml;
      }
    }
    __syncthreads();  // Fs read before the next round writes it
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = k0 + w + 4 * r;
    if (k >= Nc) continue;
    double *o = out + ((((v * 3 + a) * (long)Nc + k) * 3 + b) * Nc);
    double *o2 = out + ((((v * 3 + b) * (long)Nc + k) * 3 + a) * Nc);
#pragma unroll
    for (int q = 0; q < 5; ++q)
      if (cj[q] >= 0) {
        o[lane + 64 * q] = acc[r][q];
        if (a != b) o2[lane + 64 * q] = acc[r][q];
      }
  }
}

template <typename T>
__global__ void k_copy_cast_grid(const double *__restrict__ in, long n, T *__restrict__ out) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    out[i] = (T)in[i];
}

namespace {
std::map<std::pair<int, int>, double *> g_sw;  // singular weights per (device, p1)
const double *sing_weights_dev(int p1) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_mu);
  auto key = std::make_pair(dev, p1);
  auto it = g_sw.find(key);
  if (it != g_sw.end()) return it->second;
  std::vector<double> w;
  singular_weights(p1, w);
  double *d = nullptr;
  if (hipMalloc(&d, sizeof(double) * w.size()) != hipSuccess) return nullptr;
  if (hipMemcpy(d, w.data(), sizeof(double) * w.size(), hipMemcpyHostToDevice) != hipSuccess)
    return nullptr;
  g_sw[key] = d;
  return d;
}
}  // namespace

// Elements of scratch the build needs per vesicle of a chunk; the fused
// pole stage needs neither the kernel values K0 nor the transposed
// synthesis's scratch.
static long singular_elems_per_ves(int p0, int p1, bool fused) {
  const long Nc = sh_ncoef(p0), Ng = sh_ngrid(p0), M1 = sh_ngrid(p1);
  const long nr = (long)(p0 + 1) * p0;  // rotations per vesicle
  long e = 0;
  e += 3 * Ng;                          // X0 in T
  e += 3 * Nc;                          // S0
  e += nr * 3 * Nc;                     // S (rotated)
  e += 3 * nr * 3 * M1;                 // X, Xt, Xp
  e += nr * 3 * 2;                      // poles
  if (!fused) e += nr * 12 * M1;        // K0
  e += nr * 12 * Nc;                    // K2
  long w1 = shc2grid_work(nr * 3, p0, p1);
  if (fused) {
    w1 = std::max(w1, 3 * (p0 + nr) * Nc);  // rotation scratch
  } else {
    e += nr * 12 * Nc;                  // K1
    e += 3 * Nc * 3 * Ng;               // M1 rearranged
    w1 = std::max(w1, grid2shc_work(nr * 12, p1, p0));
    w1 = std::max(w1, grid2shc_work(9 * Nc, p0, p0));
    w1 = std::max(w1, 3 * nr * 12 * Nc);  // rotation scratch
  }
  e += w1;
  return e;
}

// k_pole_transpose's tables: RotateTranspose's per-degree blocks Mr[t][l] in
// operand order (rot_frag_off: tile ct, step s, lane: column 16 ct + lane % 16,
// entry 4 s + lane / 16, zero past the degree's entries), MatLegendre(p0, p1)
// by latitude, degree of a triple and triple (zero past a block), and for the
// single and the double layer SingularWeights(p1) times the kernel's factor by
// latitude pair, row of the pair and pole (zero where the equator is its own
// mirror row).
struct PoleTables {
  double *frag = nullptr, *ml = nullptr, *qw = nullptr;
  int nsmall = 0;
  long per_t = 0;  // doubles per latitude
};
std::map<std::tuple<int, int, int>, PoleTables> g_pole_tables;  // (device, p0, p1)

const PoleTables *pole_tables(int p0, int p1) {
  const RotMatsDev *rm = rot_mats(p0);
  const ShMatsDev *sm = sh_mats(p1, p0);
  int dev = 0;
  if (!rm || !sm || hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_mu);
  const auto key = std::make_tuple(dev, p0, p1);
  auto it = g_pole_tables.find(key);
  if (it != g_pole_tables.end()) return &it->second;
  const RotMatsHost &h = *rm->h;
  PoleTables r;
  while (r.nsmall <= p0 && h.len[r.nsmall] <= 16) ++r.nsmall;
  r.per_t = rot_frag_off(p0 + 1, r.nsmall);
  const size_t nfrag = (size_t)(p0 + 1) * r.per_t;
  const int ntri = pole_triples(p0, p0 + 1), NP = p1 / 2 + 1;
  const size_t nml = (size_t)NP * 3 * ntri;
  std::vector<double> f(nfrag + nml + 2 * 4 * NP, 0.0), qw;
  singular_weights(p1, qw);
  for (int t = 0; t <= p0; ++t)
    for (int l = 0; l <= p0; ++l) {
      const int len = h.len[l], steps = l < r.nsmall ? 4 : 8;
      const double *M = &h.data[h.off[t * (p0 + 1) + l]];
      double *o = &f[(size_t)t * r.per_t + rot_frag_off(l, r.nsmall)];
      for (int col = 0; col < len; ++col)
        for (int k = 0; k < len; ++k)
          o[((col / 16) * steps + k / 4) * 64 + (k % 4) * 16 + col % 16] = M[(size_t)col * len + k];
    }
  for (int m = 0, t0 = 0; m <= p0; ++m)
    for (int par = 0; par < 2; ++par) {
      const int cnt = pole_degrees(p0 + 1 - m, par);
      const double *src = &sm->h->data[sm->h->MlT[m]];
      for (int n = 0; n < cnt; ++n)
        for (int lat = 0; lat < NP; ++lat)
          f[nfrag + (size_t)(lat * 3 + n % 3) * ntri + t0 + n / 3] =
              src[(par + 2 * n) * (p1 + 1) + lat];
      t0 += (cnt + 2) / 3;
    }
  for (int layer = 0; layer < 2; ++layer)
    for (int i = 0; i < 4 * NP; ++i) {
      const int row = i / 2 % 2, lat = row ? p1 - i / 4 : i / 4;
      if (row && lat == i / 4) continue;
      f[nfrag + nml + layer * 4 * NP + i] =
          qw[i % 2 ? lat : p1 - lat] * (layer ? 3.0 / (4.0 * kPi) : 1.0 / (8.0 * kPi));
    }
  if (hipMalloc(&r.frag, sizeof(double) * f.size()) != hipSuccess) return nullptr;
  r.ml = r.frag + nfrag;
  r.qw = r.ml + nml;
  if (hipMemcpy(r.frag, f.data(), sizeof(double) * f.size(), hipMemcpyHostToDevice) !=
      hipSuccess) {
    (void)hipFree(r.frag);
    return nullptr;
  }
  return &(g_pole_tables[key] = r);
}

// k_pole_transpose's instance of the upsampled order p1; null where there is
// none.
const void *pole_instance(int p1) {
  switch (p1) {
    case 12: return (const void *)k_pole_transpose<12>;
    case 14: return (const void *)k_pole_transpose<14>;
    case 16: return (const void *)k_pole_transpose<16>;
    case 18: return (const void *)k_pole_transpose<18>;
    case 20: return (const void *)k_pole_transpose<20>;
    case 22: return (const void *)k_pole_transpose<22>;
    case 24: return (const void *)k_pole_transpose<24>;
    case 26: return (const void *)k_pole_transpose<26>;
    case 28: return (const void *)k_pole_transpose<28>;
    case 30: return (const void *)k_pole_transpose<30>;
    case 32: return (const void *)k_pole_transpose<32>;
    default: return nullptr;
  }
}

// Launch shape of k_pole_transpose for (p0, p1) on the current device: the
// persistent grid's workgroups; kern == nullptr where the fused stage does not
// apply.
struct PoleShape {
  const void *kern = nullptr;
  int blocks = 0;
  size_t lds = 0;
};

PoleShape pole_fused_shape(int p0, int p1) {
  PoleShape sh;
  // The build's upsampled orders 2 p0 for p0 = 6 .. 16: 16 columns per parity
  // and 256 threads hold the roles up to p0 = 16, p1 = 32.
  const void *kern = 2 * p0 <= p1 ? pole_instance(p1) : nullptr;
  if (!kern || pole_legendre_threads(p0) > kPtThreads) return sh;
  int dev = 0, maxlds = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) !=
          hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    (void)hipGetLastError();
    return sh;
  }
  const size_t lds = sizeof(double) * (size_t)pole_lds_doubles(p0, p1);
  if (lds > (size_t)maxlds) return sh;
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, kPtThreads, lds) != hipSuccess) {
    (void)hipGetLastError();
    return sh;
  }
  if (nb < 1) return sh;
  sh.kern = kern;
  sh.blocks = nb * cus;
  sh.lds = lds;
  return sh;
}

template <typename T>
int singular_build(const double *X0, long Nv, int p0, int p1, T *SL, T *DL, hipStream_t st) {
  if (p0 < 1 || p1 < 1 || p0 > 128 || p1 > 255 || Nv < 0) return VES3D_INVALID_PARAMETER;
  if (Nv == 0 || (!SL && !DL)) return VES3D_SUCCESS;
  if (!X0) return VES3D_INVALID_PARAMETER;
  const long Nc = sh_ncoef(p0), Ng = sh_ngrid(p0), M1 = sh_ngrid(p1);
  const long nr = (long)(p0 + 1) * p0;
  const double *qw = sing_weights_dev(p1);
  if (!qw) return VES3D_MEMORY_ERROR;
  // the fused stage serves the FP64 build: with FP32 transforms the
  // separate kernels' FP32 GEMMs are faster than its FP64 arithmetic
  const PoleShape ps = std::is_same<T, double>::value && g_pole_fused.load(std::memory_order_relaxed)
                           ? pole_fused_shape(p0, p1)
                           : PoleShape();
  const bool fused = ps.kern != nullptr;
  // The FP32 form's transforms stay grouped GEMMs: the pole kernel subtracts
  // FP32 positions and raises the difference to r^-5, so that another order of
  // their sums moves the operators by far more than it rounds (2.6e-4 between
  // the two at order 24, 40 vesicles).  With the one-kernel forms the distance to
  // the FP64 build went either way: the single layer's up at orders 12, 20 and 24
  // (3.3e-6, 5.0e-6, 6.8e-6 -> 3.5e-6, 5.6e-6, 7.4e-6) and down at 6, 8 and 16
  // (1.3e-6, 1.8e-6, 3.0e-6 -> 1.1e-6, 1.7e-6, 2.8e-6), the double layer's by 0.90
  // to 1.05.  The price: one-kernel transforms took 0.7 of the time for a few
  // vesicles (order 16, two: 196 -> 148 us), 0.94 for 30 at order 24, 1.1 for 300
  // at order 10.
  const ShtForm form = std::is_same<T, float>::value ? ShtForm::kGrouped : ShtForm::kAuto;
  const long per = singular_elems_per_ves(p0, p1, fused);
  const long budget = (6L << 30) / (long)sizeof(T);
  long chunk = std::max(1L, std::min(Nv, budget / per));
  T *ws = (T *)workspace(kWsSing0, sizeof(T) * per * chunk);
  if (!ws) return VES3D_MEMORY_ERROR;
  hipEvent_t done = nullptr;
  {
    int dev = 0;
    V3D_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_mu);
    BuildOrder &o = g_build_order[dev];
    if (!o.done) V3D_HIP(hipEventCreateWithFlags(&o.done, hipEventDisableTiming));
    if (o.recorded) V3D_HIP(hipStreamWaitEvent(st, o.done, 0));
    done = o.done;
    o.recorded = true;
  }
  for (long v0 = 0; v0 < Nv; v0 += chunk) {
    const long cv = std::min(chunk, Nv - v0);
    const long rot = cv * nr;
    T *p = ws;
    T *x0 = p; p += cv * 3 * Ng;
    T *S0 = p; p += cv * 3 * Nc;
    T *S = p; p += rot * 3 * Nc;
    T *X = p; p += rot * 3 * M1;
    T *Xt = p; p += rot * 3 * M1;
    T *Xp = p; p += rot * 3 * M1;
    T *P = p; p += rot * 3 * 2;
    T *K0 = p; if (!fused) p += rot * 12 * M1;
    T *K1 = p; if (!fused) p += rot * 12 * Nc;
    T *K2 = p; p += rot * 12 * Nc;
    T *M1a = p; if (!fused) p += cv * 3 * Nc * 3 * Ng;
    T *w = p;
    const long nx0 = cv * 3 * Ng;
    k_copy_cast_grid<T><<<grid_for(nx0), 256, 0, st>>>(X0 + v0 * 3 * Ng, nx0, x0);
    V3D_CHECK(launch_status());
    V3D_CHECK(sht_grid2shc<T>(x0, cv * 3, p0, p0, S0, w, st, form));
    V3D_CHECK(rotate_all<T>(S0, cv, p0, 3, S, w, st));
    V3D_CHECK(sht_shc2grid<T>(S, rot * 3, p0, p1, X, Xt, Xp, w, st, form));
    V3D_CHECK(sht_shc2pole<T>(S, rot * 3, p0, P, st));
    for (int layer = 0; layer < 2; ++layer) {
      T *dst = layer == 0 ? SL : DL;
      if (!dst) continue;
      if constexpr (std::is_same<T, double>::value) {
        if (fused) {
          const double *mft = sht_mft<double>(p1, p0);
          const RotMatsDev *rm = rot_mats(p0);
          const PoleTables *pt = pole_tables(p0, p1);
          if (!mft || !rm || !pt) return VES3D_MEMORY_ERROR;
          const unsigned nb = (unsigned)std::min<long>(rot, ps.blocks);
          const int *dpos = rm->iperm;
          const double *pqw = pt->qw + layer * 4 * (p1 / 2 + 1);
          const int4 *sources = (const int4 *)rm->scatter;
          long nrot = rot, frag_t = pt->per_t;
          int order = p0, lay = layer, nsmall = pt->nsmall;
          void *args[] = {&X,   &Xt,   &Xp,       &P,      &pqw,     &nrot,
                          &order, &mft,  (void *)&pt->ml,     &lay,    &dpos,    (void *)&pt->frag,
                          &frag_t, &nsmall, &sources, (void *)&rm->phase, &K2};
          V3D_HIP(hipLaunchKernel(ps.kern, dim3(nb), dim3(kPtThreads), args, ps.lds, st));
          V3D_CHECK(launch_status());
        }
      }
      if (!fused) {
        k_pole_kernel<T><<<grid_for(rot * M1), 256, 0, st>>>(
            X, Xt, Xp, P, qw, rot, p1, layer == 0 ? K0 : nullptr, layer == 1 ? K0 : nullptr);
        V3D_CHECK(launch_status());
        V3D_CHECK(sht_shc2grid_transpose<T>(K0, rot * 12, p1, p0, K1, w, st, form));
        V3D_CHECK(rotate_transpose<T>(K1, cv, p0, 12, K2, w, st));
      }
      if constexpr (std::is_same<T, double>::value) {
        if (fused) {  // rearrangement and Grid2SHC in one pass
          const ShMatsDev *sm = sh_mats(p0, p0);
          if (!sm) return VES3D_MEMORY_ERROR;
          const long g_blocks = cv * 6L * cdiv(Nc, kRgK);
          if (g_blocks > 0x7fffffffL) return VES3D_INVALID_PARAMETER;
          k_rearrange_g2s<<<(unsigned)g_blocks, 256, 0, st>>>(
              K2, cv, p0, sm->d64 + sm->h->Mfinv, sm->d64 + sm->h->Mlinv[0],
              dst + v0 * 9 * Nc * Nc);
          V3D_CHECK(launch_status());
          continue;
        }
      }
      const long ra_blocks = cv * 9L * cdiv(Nc, kRaK) * cdiv(Ng, kRaG);
      if (ra_blocks > 0x7fffffffL) return VES3D_INVALID_PARAMETER;
      k_singular_rearrange<T><<<(unsigned)ra_blocks, 256, 0, st>>>(K2, cv, p0, M1a);
      V3D_CHECK(launch_status());
      V3D_CHECK(sht_grid2shc<T>(M1a, cv * 9 * Nc, p0, p0, dst + v0 * 9 * Nc * Nc, w, st, form));
    }
  }
  return hip_status(hipEventRecord(done, st));
}

// ------------------------------------------------------------- self apply
// V[v][c] = sum_r F[v][r] SL[v][r][c] (+ G[v][r] DL[v][r][c]), r, c < 3 Ncoef
// (src/StokesVelocity.cc:397-447).  One workgroup per (vesicle, 256 columns);
// matrix rows stream through coalesced, the density vector sits in LDS.
template <typename TM>
__global__ __launch_bounds__(256) void k_self_apply(const TM *__restrict__ SL,
                                                     const double *__restrict__ F,
                                                     const TM *__restrict__ DL,
                                                     const double *__restrict__ G, int n,
                                                     double *__restrict__ V) {
  extern __shared__ double sh[];
  const long v = blockIdx.y;
  const int c = blockIdx.x * 256 + threadIdx.x;
  double *f = sh, *g = sh + n;
  for (int i = threadIdx.x; i < n; i += 256) {
    f[i] = SL ? F[v * n + i] : 0.0;
    g[i] = DL ? G[v * n + i] : 0.0;
  }
  __syncthreads();
  if (c >= n) return;
  double acc0 = 0, acc1 = 0, acc2 = 0, acc3 = 0;
  if (SL) {
    const TM *M = SL + v * (long)n * n + c;
    int r = 0;
    for (; r + 3 < n; r += 4) {
      acc0 += f[r] * (double)M[(long)r * n];
      acc1 += f[r + 1] * (double)M[(long)(r + 1) * n];
      acc2 += f[r + 2] * (double)M[(long)(r + 2) * n];
      acc3 += f[r + 3] * (double)M[(long)(r + 3) * n];
    }
    for (; r < n; ++r) acc0 += f[r] * (double)M[(long)r * n];
  }
  if (DL) {
    const TM *M = DL + v * (long)n * n + c;
    int r = 0;
    for (; r + 3 < n; r += 4) {
      acc0 += g[r] * (double)M[(long)r * n];
      acc1 += g[r + 1] * (double)M[(long)(r + 1) * n];
      acc2 += g[r + 2] * (double)M[(long)(r + 2) * n];
      acc3 += g[r + 3] * (double)M[(long)(r + 3) * n];
    }
    for (; r < n; ++r) acc0 += g[r] * (double)M[(long)r * n];
  }
  V[v * n + c] = (acc0 + acc1) + (acc2 + acc3);
}

// As k_self_apply for the singular build's operators, whose 3 x 3 blocks of
// Ncoef x Ncoef satisfy B_ab = B_ba (block (a, b) holds the rows of the
// symmetric tensor component c(a, b), formed once and written to both):
// thread cc reads the six blocks a <= b at column cc once and forms
// V[b Nc + cc] = sum_a sum_k F[a Nc + k] B_ab[k][cc] for b = 0, 1, 2 -- two
// thirds of the general kernel's matrix reads.  One workgroup per vesicle.
template <typename TM>
__global__ __launch_bounds__(256) void k_self_apply_sym(const TM *__restrict__ SL,
                                                         const double *__restrict__ F,
                                                         const TM *__restrict__ DL,
                                                         const double *__restrict__ G, int nc,
                                                         double *__restrict__ V) {
  extern __shared__ double sh[];
  const int n = 3 * nc;
  const long v = blockIdx.y;
  const int cc = threadIdx.x;
  double *f = sh, *g = sh + n;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    f[i] = SL ? F[v * n + i] : 0.0;
    g[i] = DL ? G[v * n + i] : 0.0;
  }
  __syncthreads();
  if (cc >= nc) return;
  double v0 = 0, v1 = 0, v2 = 0;
  auto run = [&](const TM *M, const double *x) {
    const TM *m = M + v * (long)n * n + cc;  // element (row, b nc + cc) at row n + b nc
#pragma unroll 2
    for (int k = 0; k < nc; ++k) {
      const TM *r0 = m + (long)k * n, *r1 = m + (long)(nc + k) * n,
               *r2 = m + (long)(2 * nc + k) * n;
      const double b00 = (double)r0[0], b01 = (double)r0[nc], b02 = (double)r0[2 * nc];
      const double b11 = (double)r1[nc], b12 = (double)r1[2 * nc], b22 = (double)r2[2 * nc];
      const double x0 = x[k], x1 = x[nc + k], x2 = x[2 * nc + k];
      v0 += x0 * b00 + x1 * b01 + x2 * b02;
      v1 += x0 * b01 + x1 * b11 + x2 * b12;
      v2 += x0 * b02 + x1 * b12 + x2 * b22;
    }
  };
  if (SL) run(SL, f);
  if (DL) run(DL, g);
  V[v * n + cc] = v0;
  V[v * n + nc + cc] = v1;
  V[v * n + 2 * nc + cc] = v2;
}

// Both with a workgroup's 16 waves on parts of the rows of 64 columns (SYM: lane
// cc as the thread above), the parts added in order through LDS.
// Bound: the matrix reads (5.9 TB/s for 512 vesicles at order 16) or, with few
// vesicles, their latency.  A thread per column down all rows, before -> after
// in us (FP64, order 12, symmetric): 2 vesicles 23 -> 9, 48: 39 -> 13; order 16:
// 66 -> 14, 72 -> 29; general: 37 -> 9, 116 -> 45.
template <typename TM, bool SYM>
__global__ __launch_bounds__(1024) void k_self_apply_split(const TM *__restrict__ SL,
                                                           const double *__restrict__ F,
                                                           const TM *__restrict__ DL,
                                                           const double *__restrict__ G, int nc,
                                                           double *__restrict__ V) {
  constexpr int kSums = SYM ? 3 : 1;
  __shared__ double part[15][kSums][64];
  const int n = 3 * nc, lines = SYM ? nc : n;  // rows and columns of a block
  const long v = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int col = blockIdx.x * 64 + lane, per = (lines + 15) / 16;
  const int k0 = min(wv * per, lines), k1 = min(k0 + per, lines);
  double s[kSums] = {};
  auto run = [&](const TM *M, const double *x) {
    const TM *m = M + v * (long)n * n + min(col, lines - 1);
    x += v * n;
#pragma unroll 4
    for (int k = k0; k < k1; ++k) {
      const TM *r0 = m + (long)k * n;
      if constexpr (SYM) {
        const TM *r1 = r0 + (long)nc * n, *r2 = r1 + (long)nc * n;
        const double b00 = (double)r0[0], b01 = (double)r0[nc], b02 = (double)r0[2 * nc];
        const double b11 = (double)r1[nc], b12 = (double)r1[2 * nc], b22 = (double)r2[2 * nc];
        const double x0 = x[k], x1 = x[nc + k], x2 = x[2 * nc + k];
        s[0] += x0 * b00 + x1 * b01 + x2 * b02;
        s[1] += x0 * b01 + x1 * b11 + x2 * b12;
        s[2] += x0 * b02 + x1 * b12 + x2 * b22;
      } else {
        s[0] += x[k] * (double)r0[0];
      }
    }
  };
  if (SL) run(SL, F);
  if (DL) run(DL, G);
  if (wv > 0) {
#pragma unroll
    for (int b = 0; b < kSums; ++b) part[wv - 1][b][lane] = s[b];
  }
  __syncthreads();
  if (wv > 0 || col >= lines) return;
#pragma unroll
  for (int b = 0; b < kSums; ++b) {
    for (int w = 0; w < 15; ++w) s[b] += part[w][b][lane];
    V[v * n + b * nc + col] = s[b];
  }
}

template <typename TM>
int self_apply(const TM *SL, const double *F, const TM *DL, const double *G, long Nv, int p,
               double *V, hipStream_t st, bool sym) {
  if (p < 1 || Nv < 0 || Nv > 65535) return VES3D_INVALID_PARAMETER;
  if (Nv == 0) return VES3D_SUCCESS;
  if (!V || (SL && !F) || (DL && !G)) return VES3D_INVALID_PARAMETER;
  const int n = 3 * sh_ncoef(p);
  if (!SL && !DL) return hip_status(hipMemsetAsync(V, 0, sizeof(double) * n * Nv, st));
  const int nc = sh_ncoef(p);
  const int lines = sym ? nc : n;  // columns with a sum of their own
  const dim3 gs(cdiv(lines, 64), (unsigned)Nv);
  const long waves = (long)gs.x * Nv;
  const bool f64 = sizeof(TM) == 8;
  // From about two workgroups per CU on a thread per column reads longer runs
  // and needs no sums over waves, unless a vesicle's block of 256 threads is
  // large enough to leave the last CUs waiting.  Us, thread per column / split,
  // matrices of 512 vesicles (1024: *):
  //   symmetric, FP64: orders 5* 12 / 15, 8 24 / 29, 12 119 / 124, 13 161 / 178,
  //     16 (288 coefficients) 355 / 341; FP32: 8* 26 / 39, 11* 94 / 115, 13 93 / 112;
  //     but order 6 14 / 12 and 320 vesicles of order 14 155 / 131
  //   general, FP32: orders 5* 12 / 15, 8* 34 / 45, 11* 140 / 158, 13 124 / 144, but
  //     16 259 / 248; FP64: 5* 14 / 19, 7 22 / 27, 7* 43 / 52, 12 168 / 174, but from
  //     256 columns on 10 93 / 89, 10* 202 / 175, and where the matrices outgrow the
  //     256 MB last-level cache, 2000 vesicles of order 6: 66 / 58
  // FP64 of order 12 nearly fills its blocks of 256: 108 / 114 for 320 vesicles,
  // 86 / 66 for 192.
  bool wide;
  if (sym)
    wide = nc < 256 && Nv >= 512 && waves >= 1024;
  else if (f64)
    wide = (Nv >= 512 && waves >= 1536 && n < 256 &&
            (n < 128 || Nv * n * n <= (300L << 20) / 8)) ||
           (waves >= 2560 && (int)cdiv(n, 256) * 256 - n <= n / 32 && n <= 4096);
  else
    wide = Nv >= 512 && waves >= 2048 && n < 640;
  // V over F or G: one workgroup per vesicle, which has read both before it
  // writes (up to order 8; the blocks of more columns read what others write)
  const bool over = !sym && n <= 256 && ((SL && V == F) || (DL && V == G));
  const size_t lds = 2 * n * sizeof(double);
  if (sym && wide)
    k_self_apply_sym<TM><<<dim3(1, (unsigned)Nv), 64 * gs.x, lds, st>>>(SL, F, DL, G, nc, V);
  else if (sym)
    k_self_apply_split<TM, true><<<gs, 1024, 0, st>>>(SL, F, DL, G, nc, V);
  else if (wide || over)
    k_self_apply<TM><<<dim3(cdiv(n, 256), (unsigned)Nv), 256, lds, st>>>(SL, F, DL, G, n, V);
  else
    k_self_apply_split<TM, false><<<gs, 1024, 0, st>>>(SL, F, DL, G, nc, V);
  return launch_status();
}

template int rotate_all<double>(const double *, long, int, int, double *, double *, hipStream_t);
template int rotate_transpose<double>(const double *, long, int, int, double *, double *,
                                      hipStream_t);
template int singular_build<double>(const double *, long, int, int, double *, double *, hipStream_t);
template int singular_build<float>(const double *, long, int, int, float *, float *, hipStream_t);
template int self_apply<double>(const double *, const double *, const double *, const double *,
                                long, int, double *, hipStream_t, bool);
template int self_apply<float>(const float *, const double *, const float *, const double *,
                               long, int, double *, hipStream_t, bool);

}  // namespace v3d

using namespace v3d;

extern "C" {
int ves3d_hip_rotate_all_f64(const double *S, size_t N, int p, int dof, double *S_out,
                             ves3d_stream_t stream) {
  if (!S || !S_out || dof < 1 || p < 1) return VES3D_INVALID_PARAMETER;
  const long nc = sh_ncoef(p);
  double *w = (double *)workspace(kWsSing1, sizeof(double) * (long)N * p * dof * nc * (p + 2));
  if (!w) return VES3D_MEMORY_ERROR;
  return rotate_all<double>(S, (long)N, p, dof, S_out, w, (hipStream_t)stream);
}
int ves3d_hip_rotate_transpose_f64(const double *S_in, size_t N, int p, int dof, double *S_out,
                                   ves3d_stream_t stream) {
  if (!S_in || !S_out || dof < 1 || p < 1) return VES3D_INVALID_PARAMETER;
  const long nc = sh_ncoef(p);
  double *w = (double *)workspace(kWsSing1, sizeof(double) * 2L * N * (p + 1) * p * dof * nc);
  if (!w) return VES3D_MEMORY_ERROR;
  return rotate_transpose<double>(S_in, (long)N, p, dof, S_out, w, (hipStream_t)stream);
}
int ves3d_hip_pole_kernel_shape(int p0, int p1, int *rows_host, int *threads_host,
                                int *workgroups_host) {
  if (p0 < 1 || p1 < 1 || p0 > 128 || p1 > 255) return VES3D_INVALID_PARAMETER;
  const PoleShape ps =
      g_pole_fused.load(std::memory_order_relaxed) ? pole_fused_shape(p0, p1) : PoleShape();
  // a latitude and its mirror, or two pairs of them
  if (rows_host) *rows_host = ps.kern ? 2 * pole_pairs(p1) : 0;
  if (threads_host) *threads_host = ps.kern ? kPtThreads : 0;
  if (workgroups_host) *workgroups_host = ps.blocks;
  return VES3D_SUCCESS;
}
int ves3d_hip_set_pole_kernel(int fused) {
  if (fused != 0 && fused != 1) return VES3D_INVALID_PARAMETER;
  g_pole_fused.store(fused);
  return VES3D_SUCCESS;
}
int ves3d_hip_singular_build_f64(const double *X0, size_t nves, int p0, int p1, double *SL,
                                 double *DL, ves3d_stream_t stream) {
  return singular_build<double>(X0, (long)nves, p0, p1, SL, DL, (hipStream_t)stream);
}
int ves3d_hip_singular_build_f32(const double *X0, size_t nves, int p0, int p1, float *SL,
                                 float *DL, ves3d_stream_t stream) {
  return singular_build<float>(X0, (long)nves, p0, p1, SL, DL, (hipStream_t)stream);
}
int ves3d_hip_self_apply_f64(const double *SL, const double *F, const double *DL,
                             const double *G, size_t nves, int p, double *V,
                             ves3d_stream_t stream) {
  return self_apply<double>(SL, F, DL, G, (long)nves, p, V, (hipStream_t)stream, false);
}
int ves3d_hip_self_apply_f32(const float *SL, const double *F, const float *DL,
                             const double *G, size_t nves, int p, double *V,
                             ves3d_stream_t stream) {
  return self_apply<float>(SL, F, DL, G, (long)nves, p, V, (hipStream_t)stream, false);
}
}
