// Dense coarse operator of the AMG V-cycle for gfx950.
//
// The values below the finest level are fixed once the hierarchy is built,
// so the cycle from a coarse level down (smoothing, residual, transfers,
// terminal solve) is one fixed linear map of that level's right-hand side.
// For a small level its many short launches are the time: about 2.2 us each,
// four passes per colour and cycle with MCGS smoothing.  Below the level
// that denseLevel() picks, setup applies the cycle to the unit vectors in FP64
// (all columns of a block at once) and the solver replaces the whole
// sub-cycle by one product with the resulting n x n matrix (rounded once to
// the hierarchy's type, as the terminal inverse is).
//
// The product is bound by reading the matrix once: n^2 values at about 4.5
// TB/s.  Measured without and with it, the rest of the code the same: three
// iterations of the wall-function loop on the 207k-cell helix (FP64, MCGS),
// whose CF level of 8,530 rows with the 47 + 46 colours below it becomes one 582
// MB product, 442 -> 287 ms; the 64^3 Poisson solve (1,073 rows, 44 colours)
// 18.4 -> 9.7 ms; 25k-cell helix (FP32, 7,205 rows) 112 -> 72 ms; the 40k
// pipe's fused Jacobi cycle (FP32, 2,443 rows) 52.1 -> 50.0 ms per 100
// iterations; the 64k pipe's Chebyshev cycle (FP64) 33.0 -> 32.9 per 40.
// Setting it up takes 115, 9, 48 and 1 ms.
#pragma once

#include <vector>

#include "la_kernels.hpp"

namespace nodals {
namespace dev {

// Leading dimension of a dense operator: rows start on 16 bytes.
inline int denseLd(int n) { return (n + 3) & ~3; }

// x = T b for a dense row-major n x n matrix with leading dimension ld.  A
// block takes R rows: each thread's pair of b values serves all of them.  Four
// rows once they fill the chip, one below that.
template <class TV, int R>
__global__ void __launch_bounds__(256) k_dense_mv(int n, int ld, const TV* __restrict__ T, const TV* __restrict__ b,
                                                  TV* __restrict__ x) {
  struct alignas(2 * sizeof(TV)) Pair {
    TV a, b;
  };
  __shared__ TV sh[4][R];
  const int r0 = blockIdx.x * R;
  TV s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) s[r] = TV(0);
  for (int j = 2 * threadIdx.x; j < n; j += 512) {
    const TV b0 = b[j], b1 = j + 1 < n ? b[j + 1] : TV(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const Pair t = *reinterpret_cast<const Pair*>(T + (long long)min(r0 + r, n - 1) * ld + j);
      s[r] += t.a * b0;
      s[r] += t.b * b1;
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s[r] = laneSum<64>(s[r]);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][r] = s[r];
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < R && r0 + t < n) x[r0 + t] = (sh[0][t] + sh[1][t]) + (sh[2][t] + sh[3][t]);
}

template <class TV>
void denseMv(hipStream_t s, int n, const TV* T, const TV* b, TV* x) {
  if (n <= 0) return;
  if (n >= 4096) hipLaunchKernelGGL((k_dense_mv<TV, 4>), (n + 3) / 4, 256, 0, s, n, denseLd(n), T, b, x);
  else hipLaunchKernelGGL((k_dense_mv<TV, 1>), n, 256, 0, s, n, denseLd(n), T, b, x);
  NODALS_LAUNCHED();
}

// Sum over a row of val * x[col][c] with eight gathers in flight (the row's
// columns and values are uniform over the block); column `skip` is left out.
__device__ __forceinline__ double colsRow(int k, int e, const int* __restrict__ col, const double* __restrict__ val,
                                          const double* x, int m, int c, int skip) {
  double s = 0.0;
  for (; k < e; k += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = x[(long long)col[min(k + u, e - 1)] * m + c];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < e && col[k + u] != skip) s += val[k + u] * v[u];
  }
  return s;
}

// The cycle on blocks of m columns, row-major: entry (i, c) at i*m + c.  One
// thread an entry; blockIdx.x is the row, so every column reads the row's
// values together.
// MODE 0: y = A x, 1: y = b - A x, 2: y += A x.
template <int MODE>
static __global__ void __launch_bounds__(256) k_cols_spmv(int m, const int* __restrict__ row,
                                                          const int* __restrict__ col, const double* __restrict__ val,
                                                          const double* __restrict__ x, const double* __restrict__ b,
                                                          double* __restrict__ y) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= m) return;
  const long long o = (long long)blockIdx.x * m + c;
  const double s = colsRow(row[blockIdx.x], row[blockIdx.x + 1], col, val, x, m, c, -1);
  y[o] = MODE == 0 ? s : MODE == 1 ? b[o] - s : y[o] + s;
}
// x = (add ? x : 0) + omega r / d
static __global__ void __launch_bounds__(256) k_cols_jacobi(int m, double omega, const double* __restrict__ r,
                                                            const double* __restrict__ d, double* __restrict__ x,
                                                            int add) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= m) return;
  const long long o = (long long)blockIdx.x * m + c;
  x[o] = (add ? x[o] : 0.0) + omega * r[o] / d[blockIdx.x];
}
// One Gauss-Seidel colour: rows begin + blockIdx.x.
static __global__ void __launch_bounds__(256) k_cols_gs(int m, int begin, const int* __restrict__ row,
                                                        const int* __restrict__ col, const double* __restrict__ val,
                                                        const double* __restrict__ d, const double* __restrict__ b,
                                                        double* x, double omega) {
  const int c = blockIdx.y * 256 + threadIdx.x, i = begin + blockIdx.x;
  if (c >= m) return;
  const double s = colsRow(row[i], row[i + 1], col, val, x, m, c, i);
  const long long o = (long long)i * m + c;
  const double old = x[o];
  x[o] = old + omega * ((b[o] - s) / d[i] - old);
}
// x = T b (T dense n x n)
static __global__ void __launch_bounds__(256) k_cols_dense(int n, int m, const double* __restrict__ T,
                                                           const double* __restrict__ b, double* __restrict__ x) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= m) return;
  double s = 0.0;
#pragma unroll 8
  for (int j = 0; j < n; ++j) s += T[(long long)blockIdx.x * n + j] * b[(long long)j * m + c];
  x[(long long)blockIdx.x * m + c] = s;
}
static __global__ void __launch_bounds__(256) k_cols_axpy(int m, const double* __restrict__ a, double* __restrict__ x) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= m) return;
  const long long o = (long long)blockIdx.x * m + c;
  x[o] += a[o];
}
// Unit vectors c0 .. c0 + m - 1.
static __global__ void __launch_bounds__(256) k_cols_unit(int m, int c0, double* __restrict__ b) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= m) return;
  b[(long long)blockIdx.x * m + c] = (int)blockIdx.x == c0 + c ? 1.0 : 0.0;
}
// Columns c0 .. c0 + m - 1 of the dense operator.
template <class TV>
__global__ void __launch_bounds__(256) k_cols_store(int m, int c0, int ld, const double* __restrict__ x,
                                                    TV* __restrict__ T) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= m) return;
  T[(long long)blockIdx.x * ld + c0 + c] = (TV)x[(long long)blockIdx.x * m + c];
}

// One level for the set-up of the dense operator: the operator (the level's
// pattern in its stored numbering, FP64 values), the transfers from the next
// finer level, the colour ranges and the column blocks.
struct DenseSetupLevel {
  int n = 0;
  const int *row = nullptr, *col = nullptr;
  DBuf<int> prow, pcol, trow, tcol;
  DBuf<double> val, diag, l1, pval, tval, b, x, r, corr;
  std::vector<int> colorOff;
  double lambda = 1.0;
};

}  // namespace dev
}  // namespace nodals
