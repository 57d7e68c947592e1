// Multicolour Gauss-Seidel on tiled ELL storage for gfx950.
//
// A colour pass is a chain of dependent memory round trips behind a launch:
// in CSR form the row list, the row pointers, the columns and values, then
// the gather of x.  On the sizes the AMG levels and the k-omega sweeps have
// (hundreds to thousands of rows a colour) that chain, not the bytes, is the
// time.  Here a colour's rows are laid out so that a wavefront computes the
// address of every column and value it needs from its index alone: rows are
// grouped into wave tiles of 64/L rows (L lanes a row), a tile holds U slots a
// lane, and slot u of the tile's 64 lanes is contiguous.  All loads of a row
// are issued at once, then all gathers, so the chain is two round trips.
// Unused slots hold column -1 and add nothing.
//
// The off-diagonal entries are split by colour: "lower" (colours before the
// row's) and "upper" (after it).  A pass from x = 0 needs only the half
// that has been computed, and in a symmetric sweep each pass needs only the
// half that has changed: the other half's row sum is the one the previous
// pass stored.  A forward and a backward pass from zero then read the matrix
// once instead of twice.
//
// Measured on gfx950, microseconds per colour pass in a replayed graph, CSR
// launches against these (a chain of empty launches takes 1.9):
//   207k-cell P0 Schur operator, 35 colours, 68 nonzeros a row: 5.4 -> 3.6
//   69k-row CF level, 39 colours, 74 a row: 4.6 -> 3.1
//   8.5k-row CF level, 47 colours, 102 a row: 3.8 -> 2.3
//   64^3 P1 Laplacian, 8 colours, 15 a row: 6.5 -> 4.0
#pragma once

#include <algorithm>
#include <vector>

#include "la_kernels.hpp"

namespace nodals {
namespace dev {

constexpr int kGsUnroll = 8;  // slots a lane loads before it gathers

// Which off-diagonal entries of a row a GsSlots holds.
enum class GsHalf { lower, upper, all };

// Host layout of one colour's slots: first tile, lanes a row, slots a lane.
struct GsColour {
  int tile = 0, L = 1, U = 1;
};

// Lanes a row for `count` rows of at most `width` entries: the fewest that
// leave a lane at most kGsUnroll/2 slots, widened while the colour is too small to
// give every SIMD a wavefront (2^16 threads) and a lane still holds two.
inline int gsLanes(int width, int count) {
  int L = 1;
  while (L < 64 && (width > L * (kGsUnroll / 2) || ((long long)count * L < (1 << 16) && width > 2 * L))) L *= 2;
  return L;
}

// Tiled slots of the chosen half of a coloured CSR operator (rows of colour
// c: rows[off[c]..off[c+1]), or those indices themselves when rows is null).
struct GsLayout {
  std::vector<GsColour> colour;
  std::vector<int> col, src;  // column (pad where unused), CSR position (-1 where unused)
};

template <class TI>
GsLayout gsLayout(int ncolors, const std::vector<int>& off, const int* rows, const std::vector<int>& colorOf,
                  const TI* row, const int* col, GsHalf half, int pad = -1, int forceL = 0, int minU = 1) {
  GsLayout G;
  G.colour.resize((std::size_t)ncolors);
  auto wanted = [&](int i, int j, int c) {
    if (j == i) return false;
    const int cj = colorOf[(std::size_t)j];
    return half == GsHalf::all || (half == GsHalf::lower ? cj < c : cj > c);
  };
  for (int c = 0; c < ncolors; ++c) {
    const int b = off[(std::size_t)c], n = off[(std::size_t)c + 1] - b;
    int width = 1;
    for (int q = 0; q < n; ++q) {
      const int i = rows ? rows[b + q] : b + q;
      int w = 0;
      for (TI k = row[i]; k < row[i + 1]; ++k) w += wanted(i, col[k], c) ? 1 : 0;
      width = std::max(width, w);
    }
    GsColour& C = G.colour[(std::size_t)c];
    C.L = forceL > 0 ? forceL : gsLanes(width, n);
    C.U = (width + C.L - 1) / C.L;
    if (C.U > kGsUnroll) C.U = (C.U + kGsUnroll - 1) / kGsUnroll * kGsUnroll;
    C.U = std::max(C.U, minU);
    C.tile = (int)(G.col.size() / 64);
    const int per = 64 / C.L, tiles = (n + per - 1) / per;
    G.col.resize(G.col.size() + (std::size_t)tiles * C.U * 64, pad);
    G.src.resize(G.col.size(), -1);
    for (int q = 0; q < n; ++q) {
      const int i = rows ? rows[b + q] : b + q;
      const std::size_t at = ((std::size_t)C.tile + (std::size_t)(q / per) * C.U) * 64 + (std::size_t)(q % per) * C.L;
      int w = 0;
      for (TI k = row[i]; k < row[i + 1]; ++k)
        if (wanted(i, col[k], c)) {
          const std::size_t s = at + (std::size_t)(w / C.L) * 64 + (std::size_t)(w % C.L);
          G.col[s] = col[k];
          G.src[s] = (int)k;
          ++w;
        }
    }
  }
  return G;
}

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

// Slot values gathered from the CSR values they mirror.
template <class TM>
__global__ void __launch_bounds__(256) k_gs_fill(long long n, const int* __restrict__ src, const TM* __restrict__ val,
                                                 TM* __restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int s = src[i];
  out[i] = s >= 0 ? val[s] : TM{};
}

// One colour pass over rows crow[begin + q] (begin + q without a list), q <
// count:  s = sum of the slots, plus other[i] when given (the row sum of the
// other half, unchanged since it was stored),
//   x_i <- x_i + omega ((b_i - s) / d_i - x_i)      (x_i = 0 when zero)
// and part[i] = the slots' sum when given.  Rows of one colour do not couple.
template <int L, int U, class TM, class TV>
__global__ void __launch_bounds__(256) k_gs_colour(int begin, int count, const int* __restrict__ crow, int chunks,
                                                   const int* __restrict__ col, const TM* __restrict__ val,
                                                   const TV* __restrict__ diag, const TV* __restrict__ b, TV* x,
                                                   const TV* __restrict__ other, TV* __restrict__ part, int zero,
                                                   double omega) {
  constexpr int per = 64 / L;
  const int lane = threadIdx.x & 63;
  const int tile = (blockIdx.x * 256 + threadIdx.x) >> 6;
  const int q = tile * per + lane / L;
  if (q >= count) return;
  const long long at = (long long)tile * (U * chunks) * 64 + lane;
  int c[U];
  TV a[U], v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    c[u] = col[at + u * 64];
    a[u] = ld<TV>(val, at + u * 64);
  }
  const int i = crow ? crow[begin + q] : begin + q;
  const TV bi = b[i], di = diag[i];
  const TV old = zero ? TV(0) : x[i];
  const TV so = other ? other[i] : TV(0);
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = c[u] >= 0 ? x[c[u]] : TV(0);
  const TV inv = TV(1) / di;
  TV s = 0;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (c[u] >= 0) s += a[u] * v[u];
  for (int k = 1; k < chunks; ++k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      c[u] = col[at + (long long)(k * U + u) * 64];
      a[u] = ld<TV>(val, at + (long long)(k * U + u) * 64);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = c[u] >= 0 ? x[c[u]] : TV(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c[u] >= 0) s += a[u] * v[u];
  }
  s = laneSum<L>(s);
  if (lane % L == 0) {
    if (part) part[i] = s;
    x[i] = old + (TV)omega * ((bi - (s + so)) * inv - old);
  }
}

template <int L, class TM, class TV>
void gsColourL(hipStream_t s, const GsColour& C, int begin, int count, const int* crow, const int* col, const TM* val,
               const TV* diag, const TV* b, TV* x, const TV* other, TV* part, bool zero, double omega) {
  const int per = 64 / L, grid = blocksFor((long long)((count + per - 1) / per) * 64);
  const long long o = (long long)C.tile * 64;
#define NODALS_GS_COLOUR(UN, CH)                                                                                      \
  hipLaunchKernelGGL((k_gs_colour<L, UN, TM, TV>), grid, 256, 0, s, begin, count, crow, CH, col + o, val + o, diag, b, \
                     x, other, part, zero ? 1 : 0, omega)
  switch (C.U) {
    case 1: NODALS_GS_COLOUR(1, 1); break;
    case 2: NODALS_GS_COLOUR(2, 1); break;
    case 3: NODALS_GS_COLOUR(3, 1); break;
    case 4: NODALS_GS_COLOUR(4, 1); break;
    case 5: NODALS_GS_COLOUR(5, 1); break;
    case 6: NODALS_GS_COLOUR(6, 1); break;
    case 7: NODALS_GS_COLOUR(7, 1); break;
    default: NODALS_GS_COLOUR(8, C.U / 8); break;
  }
#undef NODALS_GS_COLOUR
  NODALS_LAUNCHED();
}

template <class TM, class TV>
void gsColour(hipStream_t s, const GsColour& C, int begin, int count, const int* crow, const int* col, const TM* val,
              const TV* diag, const TV* b, TV* x, const TV* other, TV* part, bool zero, double omega) {
  if (count <= 0) return;
  switch (C.L) {
    case 1: gsColourL<1>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
    case 2: gsColourL<2>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
    case 4: gsColourL<4>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
    case 8: gsColourL<8>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
    case 16: gsColourL<16>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
    case 32: gsColourL<32>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
    default: gsColourL<64>(s, C, begin, count, crow, col, val, diag, b, x, other, part, zero, omega); break;
  }
}

// ---------------------------------------------------------------- one workgroup
// A step of the one-workgroup sweep: rows [row0, row0 + count) of one colour
// (the operator numbered in colour order), their first tile and slots a lane.
struct GsStep {
  int row0, count, tile, U;
};

template <int U, class TM, class TV>
struct GsRegs {
  int c[U];
  TM a[U];
  TV b, inv, other;
};

template <int L, int U, class TM, class TV>
__device__ __forceinline__ void gsLoad(const GsStep& st, const int* __restrict__ col, const TM* __restrict__ val,
                                       const TV* __restrict__ inv, const TV* __restrict__ b, const TV* part,
                                       GsRegs<U, TM, TV>& r) {
  constexpr int per = 64 / L;
  const int lane = threadIdx.x & 63, tiles = (st.count + per - 1) / per;
  const int w = min((int)(threadIdx.x >> 6), tiles - 1);  // a wavefront without rows loads the last tile
  const int q = w * per + lane / L, i = st.row0 + min(q, st.count - 1);
  const int at = (st.tile + w * U) * 64 + lane;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    r.c[u] = col[at + u * 64];
    r.a[u] = val[at + u * 64];
  }
  r.b = b[i];
  r.inv = inv[i];
  r.other = part[i];
}

// Barrier that orders LDS only: global loads in flight stay in flight.
__device__ __forceinline__ void ldsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int L, int U, class TM, class TV>
__device__ __forceinline__ void gsApply(const GsStep& st, const GsRegs<U, TM, TV>& r, TV* xs, TV* part, bool zero,
                                        bool useOther, double omega) {
  constexpr int per = 64 / L;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int q = w * per + lane / L, i = st.row0 + min(q, st.count - 1);
  const TV old = zero ? TV(0) : xs[i];
  TV v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = xs[r.c[u]];
  TV s = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) s += (TV)r.a[u] * v[u];
  s = laneSum<L>(s);
  if (lane % L == 0 && q < st.count) {
    if (part) part[i] = s;
    const TV t = useOther ? s + r.other : s;
    xs[i] = old + (TV)omega * ((r.b - t) * r.inv - old);
  }
  ldsBarrier();
}

// One pass over ns steps (backwards when rev): the next step's slots are
// loaded into registers before this one's gathers, so between two barriers
// only LDS reads, the row sums and the update remain.
template <int L, int U, class TM, class TV>
__device__ __forceinline__ void gsPass(int ns, bool rev, const GsStep* __restrict__ step, const int* __restrict__ col,
                                       const TM* __restrict__ val, const TV* __restrict__ inv,
                                       const TV* __restrict__ b, TV* xs, const TV* other, bool useOther, TV* part,
                                       bool zero, double omega) {
  auto at = [&](int k) {
    k = min(k, ns - 1);
    return step[rev ? ns - 1 - k : k];
  };
  GsRegs<U, TM, TV> A, B;
  GsStep s0 = at(0), s1 = at(1);
  gsLoad<L>(s0, col, val, inv, b, other, A);
  int k = 0;
  for (; k + 1 < ns; k += 2) {
    const GsStep s2 = at(k + 2), s3 = at(k + 3);
    gsLoad<L>(s1, col, val, inv, b, other, B);
    gsApply<L>(s0, A, xs, part, zero, useOther, omega);
    gsLoad<L>(s2, col, val, inv, b, other, A);
    gsApply<L>(s1, B, xs, part, zero, useOther, omega);
    s0 = s2;
    s1 = s3;
  }
  if (k < ns) gsApply<L>(s0, A, xs, part, zero, useOther, omega);
}

}  // namespace dev
}  // namespace nodals
