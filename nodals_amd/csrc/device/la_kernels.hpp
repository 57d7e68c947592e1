// Sparse and dense linear-algebra kernels for gfx950 (64-lane wavefronts).
//
// Row-parallel kernels map one row to a group of LANES consecutive lanes of
// a wavefront (LANES in {4,8,16,32,64}), chosen from the mean row length so a
// 64-lane wavefront keeps its loads coalesced on short rows without idling on
// long ones.  Group reductions are cross-lane moves inside the group
// (laneSum), so every row's sum has a fixed order: results are deterministic run
// to run.  Global FP64
// reductions are two-stage (fixed grid of partial sums, then one block per
// output), also deterministic.  Nothing here uses atomics.
#pragma once

#include "common.hpp"

namespace nodals {
namespace dev {

constexpr int kReduceParts = 256;  // partial sums per reduction (grid size)

// Sum over groups of L consecutive lanes (every lane gets it) with cross-lane
// moves inside the registers: quad swaps, half-row and row mirrors (the
// mirrored lanes hold equal partial sums already), then 16- and 32-lane swaps.
template <int CTRL>
__device__ __forceinline__ int dppMove(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dppMove(float v) {
  return __int_as_float(dppMove<CTRL>(__float_as_int(v)));
}
__device__ __forceinline__ double fromWords(unsigned lo, unsigned hi) {
  return __longlong_as_double(((long long)(int)hi << 32) | lo);
}
template <int CTRL>
__device__ __forceinline__ double dppMove(double v) {
  const long long b = __double_as_longlong(v);
  return fromWords((unsigned)dppMove<CTRL>((int)b), (unsigned)dppMove<CTRL>((int)(b >> 32)));
}
__device__ __forceinline__ float swapAdd16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double swapAdd16(double v) {
  const long long b = __double_as_longlong(v);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  return fromWords(l[0], h[0]) + fromWords(l[1], h[1]);
}
__device__ __forceinline__ int swapAdd16(int v) {
  const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
  return (int)(r[0] + r[1]);
}
__device__ __forceinline__ int swapAdd32(int v) {
  const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
  return (int)(r[0] + r[1]);
}
__device__ __forceinline__ float swapAdd32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double swapAdd32(double v) {
  const long long b = __double_as_longlong(v);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  return fromWords(l[0], h[0]) + fromWords(l[1], h[1]);
}
template <int L, class T>
__device__ __forceinline__ T laneSum(T v) {
  if constexpr (L >= 2) v += dppMove<0xB1>(v);   // quad_perm [1,0,3,2]
  if constexpr (L >= 4) v += dppMove<0x4E>(v);   // quad_perm [2,3,0,1]
  if constexpr (L >= 8) v += dppMove<0x141>(v);  // row_half_mirror
  if constexpr (L >= 16) v += dppMove<0x140>(v);  // row_mirror
  if constexpr (L >= 32) v = swapAdd16(v);
  if constexpr (L >= 64) v = swapAdd32(v);
  return v;
}

// Maximum over the wavefront.
__device__ __forceinline__ double waveMax(double v) {
  v = fmax(v, dppMove<0xB1>(v));
  v = fmax(v, dppMove<0x4E>(v));
  v = fmax(v, dppMove<0x141>(v));
  v = fmax(v, dppMove<0x140>(v));
  for (int o = 16; o < 64; o <<= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// Transposing reduction: every lane of a group of L holds N partial sums
// v[0..N); afterwards lane l of the group holds the group's totals of entries
// (N / L) l .. (N / L) l + N / L - 1 in v[0..N / L).  Each stage halves the
// entries: a lane keeps the half its bit selects and adds its partner's
// partial sums of it, N - 1 exchanges in all instead of N log2 L.  Partners
// are the mirrored lanes, which differ in the stage's bit (and in lower ones,
// whose lanes still hold the same entries); at 16 and 32 lanes one swap of
// rows or halves serves both partners.
__device__ __forceinline__ double swapPair16(double a, double b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return fromWords(l[0], h[0]) + fromWords(l[1], h[1]);
}
__device__ __forceinline__ double swapPair32(double a, double b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return fromWords(l[0], h[0]) + fromWords(l[1], h[1]);
}
template <int CTRL>
__device__ __forceinline__ double mirrorPair(double a, double b, bool upper) {
  return (upper ? b : a) + dppMove<CTRL>(upper ? a : b);
}
template <int N, int L>
__device__ __forceinline__ void laneReduceScatter(double (&v)[N], int lane) {
  static_assert(N >= L && (L == 32 || L == 64), "entries over 32 or 64 lanes");
  if (L == 64) {
#pragma unroll
    for (int p = 0; p < N / 2; ++p) v[p] = swapPair32(v[p], v[p + N / 2]);
  }
  constexpr int n4 = L == 64 ? N / 2 : N;  // entries at the 16-lane stage
#pragma unroll
  for (int p = 0; p < n4 / 2; ++p) v[p] = swapPair16(v[p], v[p + n4 / 2]);
#pragma unroll
  for (int p = 0; p < n4 / 4; ++p) v[p] = mirrorPair<0x140>(v[p], v[p + n4 / 4], lane & 8);
#pragma unroll
  for (int p = 0; p < n4 / 8; ++p) v[p] = mirrorPair<0x141>(v[p], v[p + n4 / 8], lane & 4);
#pragma unroll
  for (int p = 0; p < n4 / 16; ++p) v[p] = mirrorPair<0x1B>(v[p], v[p + n4 / 16], lane & 2);
#pragma unroll
  for (int p = 0; p < n4 / 32; ++p) v[p] = mirrorPair<0xB1>(v[p], v[p + n4 / 32], lane & 1);
}

// A lane's share of a CSR row product: s = sum of val(k) * gather(col[k])
// over k = k0, k0 + LANES, ... < e, accumulated in exactly that order (the
// order of the one-at-a-time loop, so results are bit-identical to it).  Each
// step first issues U column loads, U value loads and U gathers and only then
// accumulates, so a lane keeps U independent memory chains in flight instead
// of one (measured on gfx950: the 40k-cell P0 Schur product, 65 nnz/row,
// 8.7 -> 6.9 us; the 64^3 P1 Laplacian, 15 nnz/row, 17.2 -> 12.2 us at four
// lanes).  Slots past the row end are predicated off and never touch s.
// Entries in column `skip` are left out (-1: none).
template <int LANES>
constexpr int rowUnroll() {
  return LANES == 4 ? 4 : 2;
}
template <int LANES, class TS, class Val, class Gather>
__device__ __forceinline__ TS rowDot(int k0, int e, const int* __restrict__ col, int skip, Val val, Gather gather) {
  constexpr int U = rowUnroll<LANES>();
  TS s = 0;
  for (int k = k0; k < e; k += U * LANES) {
    int c[U];
    TS a[U], v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = k + u * LANES;
      c[u] = kk < e ? col[kk] : -1;
      a[u] = kk < e ? val(kk) : TS(0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = c[u] >= 0 ? gather(c[u]) : TS(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c[u] >= 0 && c[u] != skip) s += a[u] * v[u];
  }
  return s;
}

// Row-block index for XCD locality.  Blocks go to the eight XCDs round
// robin, and each XCD has its own L2; with the grid padded to a multiple
// of eight, XCD x takes virtual blocks [x*g/8, (x+1)*g/8), one contiguous
// eighth of the rows, so a vector written by one such kernel is read back
// by the next from the same L2.  A bijection on [0, gridDim.x): blocks past
// the rows exit in the caller's bounds check, whatever the hardware's
// placement.
__device__ __forceinline__ int xcdBlock(int block, int grid) { return (block & 7) * (grid >> 3) + (block >> 3); }
__device__ __forceinline__ int xcdRowBlock() { return xcdBlock((int)blockIdx.x, (int)gridDim.x); }
inline int xcdGrid(int grid) { return (grid + 7) & ~7; }

// ---------------------------------------------------------------- BLAS-1
template <class T>
__global__ void k_fill(long long n, T* x, T a) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = a;
}
template <class TD, class TS>
__global__ void k_cast(long long n, const TS* __restrict__ a, TD* __restrict__ b) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (TD)a[i];
}
template <class T>
__global__ void k_axpy(long long n, double a, const T* __restrict__ x, T* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] += (T)a * x[i];
}
template <class T>
__global__ void k_scale_into(long long n, double a, const T* __restrict__ x, T* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (T)a * x[i];
}
template <class T>
__global__ void k_xpby(long long n, const T* __restrict__ x, double b, T* __restrict__ y) {
  // y = x + b*y
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i] + (T)b * y[i];
}
template <class T>
__global__ void k_axpy2(long long n, double a, const T* __restrict__ p, const T* __restrict__ q, T* __restrict__ x,
                        T* __restrict__ r) {
  // x += a p ; r -= a q
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const T aa = (T)a;
    x[i] += aa * p[i];
    r[i] -= aa * q[i];
  }
}
template <class T, class TB = T>
__global__ void k_jacobi_zero(int n, double omega, const TB* __restrict__ b, const T* __restrict__ d, T* __restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = (T)omega * (T)b[i] / d[i];
}

// Multi-vector update y -= sum_k c_k V_k (V column-major, stride n).
struct Coef32 {
  double c[32];
};
static __global__ void k_multi_axpy(long long n, int k, const double* __restrict__ V, Coef32 c, double* __restrict__ y,
                             double sign) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int j = 0; j < k; ++j) s += c.c[j] * V[(long long)j * n + i];
  y[i] += sign * s;
}
// Same with the coefficients read from device memory (k <= 32), so the
// update can follow a device-side reduction without a host round trip.
static __global__ void __launch_bounds__(256) k_multi_axpy_dev(long long n, int k, const double* __restrict__ V,
                                                                const double* __restrict__ coef,
                                                                double* __restrict__ y, double sign) {
  __shared__ double c[32];
  if (threadIdx.x < 32) c[threadIdx.x] = (int)threadIdx.x < k ? coef[threadIdx.x] : 0.0;
  __syncthreads();
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int j = 0; j < k; ++j) s += c[j] * V[(long long)j * n + i];
  y[i] += sign * s;
}
// ---------------------------------------------------------------- reductions
__device__ __forceinline__ double blockSum256(double v, double* sh) {
  v = laneSum<64>(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sh[w] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0) t = sh[0] + sh[1] + sh[2] + sh[3];
  __syncthreads();
  return t;
}

template <class TA, class TB>
__global__ void __launch_bounds__(256) k_dot_part(long long n, const TA* __restrict__ x, const TB* __restrict__ y,
                                                  double* __restrict__ part) {
  __shared__ double sh[4];
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    s += (double)x[i] * (double)y[i];
  s = blockSum256(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// K dot products against one vector: part[k*gridDim + block] = sum V_k . w;
// with NORM, entry k holds w . w (one pass over w for Gram-Schmidt + norm).
// Each wavefront reduces all its sums with cross-lane shuffles, then one
// barrier and one LDS pass combine the four wavefronts.
template <int KMAX, bool NORM>
__global__ void __launch_bounds__(256) k_multidot_part(long long n, int k, const double* __restrict__ V,
                                                       const double* __restrict__ w, double* __restrict__ part) {
  __shared__ double sh[4][KMAX + 1];
  double s[KMAX + 1];
#pragma unroll
  for (int j = 0; j <= KMAX; ++j) s[j] = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const double wi = w[i];
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (j < k) s[j] += V[(long long)j * n + i] * wi;
    if (NORM) s[KMAX] += wi * wi;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j <= KMAX; ++j) {
    if (j < k || (NORM && j == KMAX)) {
      const double t = laneSum<64>(s[j]);
      if (lane == 0) sh[wv][j] = t;
    }
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < k) part[(long long)t * gridDim.x + blockIdx.x] = sh[0][t] + sh[1][t] + sh[2][t] + sh[3][t];
  if (NORM && t == k)
    part[(long long)k * gridDim.x + blockIdx.x] = sh[0][KMAX] + sh[1][KMAX] + sh[2][KMAX] + sh[3][KMAX];
}

// out[b] = sum of part[b*nparts .. b*nparts+nparts)
static __global__ void __launch_bounds__(256) k_reduce_final(int nparts, const double* __restrict__ part, double* out) {
  __shared__ double sh[4];
  double s = 0.0;
  for (int i = threadIdx.x; i < nparts; i += 256) s += part[(long long)blockIdx.x * nparts + i];
  s = blockSum256(s, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// ---------------------------------------------------------------- CSR kernels
// y = A x (RESID=false) or y = b - A x (RESID=true); ACC=true adds into y.
template <int LANES, class TM, class TV, bool RESID, bool ACC>
__global__ void __launch_bounds__(256) k_spmv(int n, const int* __restrict__ row, const int* __restrict__ col,
                                              const TM* __restrict__ val, const TV* __restrict__ x,
                                              const TV* __restrict__ b, TV* __restrict__ y) {
  const int gid = blockIdx.x * 256 + threadIdx.x;
  const int r = gid / LANES;
  const int lane = gid % LANES;
  if (r >= n) return;
  TV s = rowDot<LANES, TV>(
      row[r] + lane, row[r + 1], col, -1, [&](int k) { return ld<TV>(val, k); }, [&](int j) { return x[j]; });
  s = laneSum<LANES>(s);
  if (lane == 0) {
    if (RESID) y[r] = b[r] - s;
    else if (ACC) y[r] += s;
    else y[r] = s;
  }
}

// y = A x of the P0 pressure Schur operator, the Krylov operator of the
// pressure solve (the body of k_spmv<LANES, double, double, false, false>
// under its own name, so profiles and launch probes see it apart from the
// AMG levels' products).
template <int LANES>
__global__ void __launch_bounds__(256) k_schur_spmv(int n, const int* __restrict__ row, const int* __restrict__ col,
                                                    const double* __restrict__ val, const double* __restrict__ x,
                                                    double* __restrict__ y) {
  const int gid = xcdRowBlock() * 256 + threadIdx.x;
  const int r = gid / LANES;
  const int lane = gid % LANES;
  if (r >= n) return;
  double s = rowDot<LANES, double>(
      row[r] + lane, row[r + 1], col, -1, [&](int k) { return val[k]; }, [&](int j) { return x[j]; });
  s = laneSum<LANES>(s);
  if (lane == 0) y[r] = s;
}

// Single-sweep Jacobi smoothing fused into the V-cycle residuals.
// Pre-smoothing from zero and its residual in one pass:
//   t = w b / d,   r = b - A t
// (t_j of every neighbour is formed from b_j and d_j as the separate
// smoother would, so the values equal the unfused sequence).
// b may be stored wider than TV (an FP64 Krylov vector entering an FP32
// hierarchy): it is rounded to TV on load, exactly as a separate cast pass
// would round it.
template <int LANES, class TM, class TV, class TB = TV>
__global__ void __launch_bounds__(256) k_jacobi_pre_resid(int n, const int* __restrict__ row,
                                                          const int* __restrict__ col, const TM* __restrict__ val,
                                                          const TB* __restrict__ b, const TV* __restrict__ d,
                                                          double omega, TV* __restrict__ t, TV* __restrict__ r) {
  const int gid = xcdRowBlock() * 256 + threadIdx.x;
  const int i = gid / LANES;
  const int lane = gid % LANES;
  if (i >= n) return;
  TV s = rowDot<LANES, TV>(
      row[i] + lane, row[i + 1], col, -1, [&](int k) { return ld<TV>(val, k); },
      [&](int j) { return (TV)omega * (TV)b[j] / d[j]; });
  s = laneSum<LANES>(s);
  if (lane == 0) {
    const TV bi = (TV)b[i];
    t[i] = (TV)omega * bi / d[i];
    r[i] = bi - s;
  }
}
// Residual and post-smoothing correction in one pass:
//   z = t + w (b - A t) / d      (z and t distinct)
// (b as above; z may be stored wider than TV and receives the TV result.)
template <int LANES, class TM, class TV, class TB = TV, class TZ = TV>
__global__ void __launch_bounds__(256) k_resid_jacobi_post(int n, const int* __restrict__ row,
                                                           const int* __restrict__ col, const TM* __restrict__ val,
                                                           const TB* __restrict__ b, const TV* __restrict__ d,
                                                           double omega, const TV* __restrict__ t,
                                                           TZ* __restrict__ z) {
  const int gid = xcdRowBlock() * 256 + threadIdx.x;
  const int i = gid / LANES;
  const int lane = gid % LANES;
  if (i >= n) return;
  TV s = rowDot<LANES, TV>(
      row[i] + lane, row[i + 1], col, -1, [&](int k) { return ld<TV>(val, k); }, [&](int j) { return t[j]; });
  s = laneSum<LANES>(s);
  if (lane == 0) {
    const TV r = (TV)b[i] - s;
    z[i] = (TZ)(t[i] + (TV)omega * r / d[i]);
  }
}

// A smoothing of two and more steps (Jacobi sweeps, Chebyshev), from zero, of
// the residual of x, added to x: its first and last kernel, the ones between
// being k_resid_jacobi_post.  kResid is the residual alone; b may be stored
// wider than TV as above.
//   kResid:  r = b - A x
//   kFirst:  r = b - A x,  c = w r / d
//   kLast:   z = y + (x + w (b - A x) / d)      (z may be y)
// Bound by the matrix; what a pass of its own for each product, step and sum
// cost on top was the launch and the vectors (2.0 to 4.1 us each, six of a
// two-step V-cycle's fourteen kernels): whole runs of 18k, 64k and 769k cells
// 22.5 -> 19.9, 36.0 -> 33.7 and 142.9 -> 139.8 ms.
enum { kResid, kFirst, kLast };
template <int LANES, int STEP, class TM, class TV, class TB, class TZ>
__global__ void __launch_bounds__(256) k_resid_step(int n, const int* __restrict__ row, const int* __restrict__ col,
                                                    const TM* __restrict__ val, const TB* __restrict__ b,
                                                    const TV* __restrict__ d, double omega, const TV* __restrict__ x,
                                                    TV* __restrict__ r, TV* __restrict__ c, const TV* y, TZ* z) {
  const int gid = xcdRowBlock() * 256 + threadIdx.x;
  const int i = gid / LANES;
  const int lane = gid % LANES;
  if (i >= n) return;
  TV s = rowDot<LANES, TV>(
      row[i] + lane, row[i + 1], col, -1, [&](int k) { return ld<TV>(val, k); }, [&](int j) { return x[j]; });
  s = laneSum<LANES>(s);
  if (lane != 0) return;
  const TV ri = (TV)b[i] - s;
  if (STEP != kLast) r[i] = ri;
  if (STEP == kFirst) c[i] = (TV)omega * ri / d[i];
  if (STEP == kLast) {
    const TV ci = x[i] + (TV)omega * ri / d[i];
    z[i] = (TZ)(y[i] + ci);
  }
}

// Product rounded on its own (never fused into a following add).
__device__ __forceinline__ float mulRn(float a, float b) { return __fmul_rn(a, b); }
__device__ __forceinline__ double mulRn(double a, double b) { return __dmul_rn(a, b); }

// The same with the coarse correction of an aggregation transfer (one
// entry per fine row: pcol[j], pval[j]) folded in: t'_j = t_j + pval_j
// xc[pcol_j] is formed on the fly for every row the pass reads, with the
// product rounded before the add, which is the value the separate
// prolongation kernel would have stored (its row sum is that single
// product).
template <int LANES, class TM, class TV, class TB = TV, class TZ = TV>
__global__ void __launch_bounds__(256) k_resid_jacobi_post_agg(
    int n, const int* __restrict__ row, const int* __restrict__ col, const TM* __restrict__ val,
    const TB* __restrict__ b, const TV* __restrict__ d, double omega, const TV* __restrict__ t,
    const int* __restrict__ pcol, const TV* __restrict__ pval, const TV* __restrict__ xc, TZ* __restrict__ z) {
  const int gid = blockIdx.x * 256 + threadIdx.x;
  const int i = gid / LANES;
  const int lane = gid % LANES;
  if (i >= n) return;
  TV s = rowDot<LANES, TV>(
      row[i] + lane, row[i + 1], col, -1, [&](int k) { return ld<TV>(val, k); },
      [&](int j) { return t[j] + mulRn(pval[j], xc[pcol[j]]); });
  s = laneSum<LANES>(s);
  if (lane == 0) {
    const TV ti = t[i] + mulRn(pval[i], xc[pcol[i]]);
    const TV r = (TV)b[i] - s;
    z[i] = (TZ)(ti + (TV)omega * r / d[i]);
  }
}

// l1[r] = sum_k |a_rk|
template <int LANES, class TM, class TV>
__global__ void __launch_bounds__(256) k_row_l1(int n, const int* __restrict__ row, const TM* __restrict__ val,
                                                TV* __restrict__ l1) {
  const int gid = blockIdx.x * 256 + threadIdx.x;
  const int r = gid / LANES;
  const int lane = gid % LANES;
  if (r >= n) return;
  TV s = 0;
  for (int k = row[r] + lane; k < row[r + 1]; k += LANES) {
    const TV v = ld<TV>(val, k);
    s += v >= TV(0) ? v : -v;
  }
  s = laneSum<LANES>(s);
  if (lane == 0) l1[r] = s;
}

template <class T>
__global__ void k_diag_gather(int n, const int* __restrict__ diagPos, const T* __restrict__ val, T* __restrict__ d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = val[diagPos[i]];
}

// ---------------------------------------------------------------- launch helpers
// Lanes per CSR row from the mean row length and the number of rows.  Four
// lanes (four loads in flight each) for rows up to 20 nonzeros, eight (two
// each) up to 128 (measured on gfx950: the 64^3 P1 Laplacian, 15 nnz/row,
// runs in 12.2 us at four lanes against 14.3 at eight; the 40k-cell P0 Schur
// operator, 65 nnz/row, in 6.9 us at eight against 9.7 at four and 7.5 at
// sixteen), wider groups for longer rows.  When the rows
// are too few to give the chip 2^17 threads (two waves per SIMD), the group
// widens further while every lane keeps at least two nonzeros: a 1,073-row
// coarse level with 88 nnz/row runs in 2.7 us at 32 lanes and 4.7 us at 8.
inline int lanesFor(double meanRow, long long rows) {
  int L = meanRow <= 20 ? 4 : meanRow <= 128 ? 8 : meanRow <= 256 ? 16 : meanRow <= 512 ? 32 : 64;
  while (L < 64 && rows * L < (1LL << 17) && 4.0 * L <= meanRow) L *= 2;
  return L;
}

template <class TM, class TV, bool RESID, bool ACC>
void spmv(hipStream_t s, int lanes, int n, const int* row, const int* col, const TM* val, const TV* x, const TV* b,
          TV* y, hipEvent_t start = nullptr, hipEvent_t stop = nullptr) {
  if (n <= 0) return;
  const int grid = blocksFor((long long)n * lanes);
  // With events, the launch goes through hipExtLaunchKernelGGL, which stamps
  // them from the kernel's own dispatch packet (its start and end), not from
  // separate marker packets.
#define NODALS_SPMV_LAUNCH(LN)                                                                             \
  if (start)                                                                                               \
    hipExtLaunchKernelGGL((k_spmv<LN, TM, TV, RESID, ACC>), dim3(grid), dim3(256), 0, s, start, stop, 0, n, \
                          row, col, val, x, b, y);                                                         \
  else                                                                                                     \
    hipLaunchKernelGGL((k_spmv<LN, TM, TV, RESID, ACC>), grid, 256, 0, s, n, row, col, val, x, b, y);
  switch (lanes) {
    case 4: NODALS_SPMV_LAUNCH(4) break;
    case 8: NODALS_SPMV_LAUNCH(8) break;
    case 16: NODALS_SPMV_LAUNCH(16) break;
    case 32: NODALS_SPMV_LAUNCH(32) break;
    default: NODALS_SPMV_LAUNCH(64) break;
  }
#undef NODALS_SPMV_LAUNCH
  NODALS_LAUNCHED();
}

inline void schurSpmv(hipStream_t s, int lanes, int n, const int* row, const int* col, const double* val,
                      const double* x, double* y, hipEvent_t start = nullptr, hipEvent_t stop = nullptr) {
  if (n <= 0) return;
  const int grid = xcdGrid(blocksFor((long long)n * lanes));  // the kernel maps blocks per XCD
#define NODALS_SCHUR_LAUNCH(LN)                                                                                  \
  if (start)                                                                                                    \
    hipExtLaunchKernelGGL((k_schur_spmv<LN>), dim3(grid), dim3(256), 0, s, start, stop, 0, n, row, col, val, x, y); \
  else                                                                                                          \
    hipLaunchKernelGGL((k_schur_spmv<LN>), grid, 256, 0, s, n, row, col, val, x, y);
  switch (lanes) {
    case 4: NODALS_SCHUR_LAUNCH(4) break;
    case 8: NODALS_SCHUR_LAUNCH(8) break;
    case 16: NODALS_SCHUR_LAUNCH(16) break;
    case 32: NODALS_SCHUR_LAUNCH(32) break;
    default: NODALS_SCHUR_LAUNCH(64) break;
  }
#undef NODALS_SCHUR_LAUNCH
  NODALS_LAUNCHED();
}

template <class TM, class TV, class TB = TV>
void jacobiPreResid(hipStream_t s, int lanes, int n, const int* row, const int* col, const TM* val, const TB* b,
                    const TV* d, double omega, TV* t, TV* r) {
  if (n <= 0) return;
  const int grid = xcdGrid(blocksFor((long long)n * lanes));  // the kernel maps blocks per XCD
#define NODALS_JPR(LN) \
  hipLaunchKernelGGL((k_jacobi_pre_resid<LN, TM, TV, TB>), grid, 256, 0, s, n, row, col, val, b, d, omega, t, r)
  switch (lanes) {
    case 4: NODALS_JPR(4); break;
    case 8: NODALS_JPR(8); break;
    case 16: NODALS_JPR(16); break;
    case 32: NODALS_JPR(32); break;
    default: NODALS_JPR(64); break;
  }
#undef NODALS_JPR
  NODALS_LAUNCHED();
}

template <class TM, class TV, class TB = TV, class TZ = TV>
void residJacobiPostAgg(hipStream_t s, int lanes, int n, const int* row, const int* col, const TM* val, const TB* b,
                        const TV* d, double omega, const TV* t, const int* pcol, const TV* pval, const TV* xc,
                        TZ* z) {
  if (n <= 0) return;
  const int grid = blocksFor((long long)n * lanes);
#define NODALS_RJPA(LN)                                                                                        \
  hipLaunchKernelGGL((k_resid_jacobi_post_agg<LN, TM, TV, TB, TZ>), grid, 256, 0, s, n, row, col, val, b, d, omega, \
                     t, pcol, pval, xc, z)
  switch (lanes) {
    case 4: NODALS_RJPA(4); break;
    case 8: NODALS_RJPA(8); break;
    case 16: NODALS_RJPA(16); break;
    case 32: NODALS_RJPA(32); break;
    default: NODALS_RJPA(64); break;
  }
#undef NODALS_RJPA
  NODALS_LAUNCHED();
}

template <class TM, class TV, class TB = TV, class TZ = TV>
void residJacobiPost(hipStream_t s, int lanes, int n, const int* row, const int* col, const TM* val, const TB* b,
                     const TV* d, double omega, const TV* t, TZ* z) {
  if (n <= 0) return;
  const int grid = xcdGrid(blocksFor((long long)n * lanes));  // the kernel maps blocks per XCD
#define NODALS_RJP(LN) \
  hipLaunchKernelGGL((k_resid_jacobi_post<LN, TM, TV, TB, TZ>), grid, 256, 0, s, n, row, col, val, b, d, omega, t, z)
  switch (lanes) {
    case 4: NODALS_RJP(4); break;
    case 8: NODALS_RJP(8); break;
    case 16: NODALS_RJP(16); break;
    case 32: NODALS_RJP(32); break;
    default: NODALS_RJP(64); break;
  }
#undef NODALS_RJP
  NODALS_LAUNCHED();
}

template <int STEP, class TM, class TV, class TB = TV, class TZ = TV>
void residStep(hipStream_t s, int lanes, int n, const int* row, const int* col, const TM* val, const TB* b,
               const TV* d, double omega, const TV* x, TV* r, TV* c, const TV* y, TZ* z) {
  if (n <= 0) return;
  const int grid = xcdGrid(blocksFor((long long)n * lanes));  // the kernel maps blocks per XCD
#define NODALS_RS(LN) \
  hipLaunchKernelGGL((k_resid_step<LN, STEP, TM, TV, TB, TZ>), grid, 256, 0, s, n, row, col, val, b, d, omega, x, r, c, y, z)
  switch (lanes) {
    case 4: NODALS_RS(4); break;
    case 8: NODALS_RS(8); break;
    case 16: NODALS_RS(16); break;
    case 32: NODALS_RS(32); break;
    default: NODALS_RS(64); break;
  }
#undef NODALS_RS
  NODALS_LAUNCHED();
}

template <class TM, class TV>
void rowL1(hipStream_t s, int lanes, int n, const int* row, const TM* val, TV* l1) {
  if (n <= 0) return;
  const int grid = blocksFor((long long)n * lanes);
  switch (lanes) {
    case 4: hipLaunchKernelGGL((k_row_l1<4, TM, TV>), grid, 256, 0, s, n, row, val, l1); break;
    case 8: hipLaunchKernelGGL((k_row_l1<8, TM, TV>), grid, 256, 0, s, n, row, val, l1); break;
    case 16: hipLaunchKernelGGL((k_row_l1<16, TM, TV>), grid, 256, 0, s, n, row, val, l1); break;
    case 32: hipLaunchKernelGGL((k_row_l1<32, TM, TV>), grid, 256, 0, s, n, row, val, l1); break;
    default: hipLaunchKernelGGL((k_row_l1<64, TM, TV>), grid, 256, 0, s, n, row, val, l1); break;
  }
  NODALS_LAUNCHED();
}

template <class T>
void fill(hipStream_t s, long long n, T* x, T a) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill<T>, blocksFor(n), 256, 0, s, n, x, a);
  NODALS_LAUNCHED();
}
template <class TD, class TS>
void cast(hipStream_t s, long long n, const TS* a, TD* b) {
  if (n <= 0) return;
  hipLaunchKernelGGL((k_cast<TD, TS>), blocksFor(n), 256, 0, s, n, a, b);
  NODALS_LAUNCHED();
}
template <class T>
void copy(hipStream_t s, long long n, const T* a, T* b) {
  if (n <= 0) return;
  NODALS_HIP(hipMemcpyAsync(b, a, (std::size_t)n * sizeof(T), hipMemcpyDeviceToDevice, s));
}
template <class T>
void axpy(hipStream_t s, long long n, double a, const T* x, T* y) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_axpy<T>, blocksFor(n), 256, 0, s, n, a, x, y);
  NODALS_LAUNCHED();
}

// Deterministic FP64 dot products; results land in pinned host memory.
class Reducer {
 public:
  Reducer() = default;
  ~Reducer() {
    if (host_) (void)hipHostFree(host_);
  }
  Reducer(const Reducer&) = delete;
  Reducer& operator=(const Reducer&) = delete;

  void init(int maxVectors) {
    maxVec_ = maxVectors;
    part_.alloc((std::size_t)kReduceParts * maxVectors);
    part2_.alloc((std::size_t)kReduceParts * maxVectors);
    if (host_) (void)hipHostFree(host_);
    // Coherent pinned memory: the final reduction kernel writes it directly
    // and the host reads it after the stream synchronisation.
    NODALS_HIP(hipHostMalloc((void**)&host_, sizeof(double) * (std::size_t)maxVectors, hipHostMallocCoherent));
  }

  template <class TA, class TB>
  void dotAsync(hipStream_t s, long long n, const TA* x, const TB* y) {
    hipLaunchKernelGGL((k_dot_part<TA, TB>), kReduceParts, 256, 0, s, n, x, y, part_.data());
    NODALS_LAUNCHED();
    hipLaunchKernelGGL(k_reduce_final, 1, 256, 0, s, kReduceParts, part_.data(), host_);
    NODALS_LAUNCHED();
  }
  template <class TA, class TB>
  double dot(hipStream_t s, long long n, const TA* x, const TB* y) {
    dotAsync(s, n, x, y);
    NODALS_HIP(hipStreamSynchronize(s));
    return host_[0];
  }
  // out[j] = V_j . w for j < k (V column-major with stride n); with
  // withNorm, out[k] = w . w from the same pass.
  void multidot(hipStream_t s, long long n, int k, const double* V, const double* w, double* out,
                bool withNorm = false) {
    const int outs = k + (withNorm ? 1 : 0);
    if (outs > maxVec_ || k > 32) fail("multidot width exceeds reducer capacity", kErrInternal);
    if (withNorm)
      hipLaunchKernelGGL((k_multidot_part<32, true>), kReduceParts, 256, 0, s, n, k, V, w, part_.data());
    else
      hipLaunchKernelGGL((k_multidot_part<32, false>), kReduceParts, 256, 0, s, n, k, V, w, part_.data());
    NODALS_LAUNCHED();
    hipLaunchKernelGGL(k_reduce_final, outs, 256, 0, s, kReduceParts, part_.data(), host_);
    NODALS_LAUNCHED();
    NODALS_HIP(hipStreamSynchronize(s));
    for (int j = 0; j < outs; ++j) out[j] = host_[j];
  }
  double* partials() { return part_.data(); }
  // a second partials area, for a kernel that reads partials() and writes
  // its own in the same launch
  double* partials2() { return part2_.data(); }
  // Partial sums only (kReduceParts per output, output q at q*kReduceParts),
  // for a consumer kernel that finishes the reduction itself.
  template <class TA, class TB>
  void dotPartials(hipStream_t s, long long n, const TA* x, const TB* y) {
    hipLaunchKernelGGL((k_dot_part<TA, TB>), kReduceParts, 256, 0, s, n, x, y, part_.data());
    NODALS_LAUNCHED();
  }
  void multidotPartials(hipStream_t s, long long n, int k, const double* V, const double* w) {
    if (k > maxVec_ || k > 32) fail("multidot width exceeds reducer capacity", kErrInternal);
    hipLaunchKernelGGL((k_multidot_part<32, false>), kReduceParts, 256, 0, s, n, k, V, w, part_.data());
    NODALS_LAUNCHED();
  }
  double* hostOut() { return host_; }
  const double* hostOut() const { return host_; }

 private:
  DBuf<double> part_, part2_;
  double* host_ = nullptr;
  int maxVec_ = 0;
};

}  // namespace dev
}  // namespace nodals
