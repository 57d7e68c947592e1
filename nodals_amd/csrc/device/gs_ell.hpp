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
//   207k-cell P0 Schur operator, 35 colours, 68 nonzeros a row: 5.4 -> 3.5
//   69k-row CF level, 39 colours, 74 a row: 4.6 -> 2.9
//   8.5k-row CF level, 47 colours, 102 a row: 3.8 -> 2.3
//   64^3 P1 Laplacian, 8 colours, 15 a row: 6.5 -> 3.9
//   7.5k-row k-omega vertex operator, 10 colours, 14 a row: 3.7 -> 2.5
// Half of that is the reduction over lanes in registers, the exact slot count
// as a template argument and the missing row pointers; a fixed count of eight
// with predicated slots costs 0.3-0.4 us a pass more.
#pragma once

#include <vector>

#include "../host/gs_layout.hpp"
#include "la_kernels.hpp"

namespace nodals {
namespace dev {

// Slot values gathered from the CSR values they mirror.
template <class TO, class TI>
__global__ void __launch_bounds__(256) k_gs_fill(long long n, const int* __restrict__ src, const TI* __restrict__ val,
                                                 TO* __restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int s = src[i];
  out[i] = s >= 0 ? (TO)val[s] : TO{};
}

// One pass over a class of a colour: rows crow[begin + q] (begin + q without a
// list), q < count:  s = sum of the slots, plus other[i] when given (the row sum of the
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
    x[i] = old + (TV)omega * ((bi - (s + so)) / di - old);
  }
}

template <int L, class TM, class TV>
void gsClassL(hipStream_t s, const GsClass& C, const int* crow, const int* col, const TM* val, const TV* diag,
              const TV* b, TV* x, const TV* other, TV* part, bool zero, double omega) {
  const int per = 64 / L, grid = blocksFor((long long)((C.count + per - 1) / per) * 64);
  const long long o = (long long)C.tile * 64;
#define NODALS_GS_COLOUR(UN, CH)                                                                                       \
  hipLaunchKernelGGL((k_gs_colour<L, UN, TM, TV>), grid, 256, 0, s, C.begin, C.count, crow, CH, col + o, val + o, diag, \
                     b, x, other, part, zero ? 1 : 0, omega)
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

// Device slots of one half of an operator.
template <class TM>
struct GsSlots {
  std::vector<std::vector<GsClass>> colour;
  DBuf<int> col, src, rows;  // rows: the layout's own list, empty unless a colour was split
  DBuf<TM> val;
  // With the operator's values when they are fixed; otherwise fill() them.
  void upload(const GsLayout& G, const TM* csr) {
    colour = G.colour;
    rows.upload(G.rows);
    col.upload(G.col);
    if (!csr) {
      src.upload(G.src);
      val.alloc(G.src.size());
      return;
    }
    std::vector<TM> v(G.src.size(), TM{});
    for (std::size_t k = 0; k < v.size(); ++k)
      if (G.src[k] >= 0) v[k] = csr[G.src[k]];
    val.upload(v);
  }
  // Values from the operator's CSR values.
  template <class TI>
  void fill(hipStream_t s, const TI* csr) {
    const long long n = (long long)src.size();
    if (n == 0) return;
    hipLaunchKernelGGL((k_gs_fill<TM, TI>), blocksFor(n), 256, 0, s, n, src.data(), csr, val.data());
    NODALS_LAUNCHED();
  }
};

// A pass over colour c: one launch, or one a class where the colour is split.
// crow: the colouring's row list, null where colours are contiguous rows.
template <class TM, class TV>
void gsColour(hipStream_t s, const GsSlots<TM>& G, int c, const int* crow, const TV* diag, const TV* b, TV* x,
              const TV* other, TV* part, bool zero, double omega) {
  const int* list = G.rows.size() ? G.rows.data() : crow;
  for (const GsClass& C : G.colour[(std::size_t)c]) {
#define NODALS_GS_LANES(LN) \
  gsClassL<LN>(s, C, list, G.col.data(), G.val.data(), diag, b, x, other, part, zero, omega)
    switch (C.L) {
      case 1: NODALS_GS_LANES(1); break;
      case 2: NODALS_GS_LANES(2); break;
      case 4: NODALS_GS_LANES(4); break;
      case 8: NODALS_GS_LANES(8); break;
      case 16: NODALS_GS_LANES(16); break;
      case 32: NODALS_GS_LANES(32); break;
      default: NODALS_GS_LANES(64); break;
    }
#undef NODALS_GS_LANES
  }
}

}  // namespace dev
}  // namespace nodals
