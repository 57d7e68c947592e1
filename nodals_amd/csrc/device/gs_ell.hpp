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

#include <algorithm>
#include <thread>
#include <vector>

#include "../host/h8_setup.hpp"
#include "la_kernels.hpp"

namespace nodals {
namespace dev {

constexpr int kGsUnroll = 8;  // most slots a lane loads before it gathers

// Which off-diagonal entries of a row a GsSlots holds.
enum class GsHalf { lower, upper, all };

// Host layout of one colour's slots: first tile, lanes a row, slots a lane
// (at most kGsUnroll, or a multiple of it).
struct GsColour {
  int tile = 0, L = 1, U = 1;
};

// Lanes a row for `count` rows of at most `width` entries: the fewest that
// leave a lane at most kGsUnroll/2 slots, widened while the colour is too
// small to give every SIMD a wavefront (2^16 threads) and a lane still holds
// two: within 4% of the best of 1..64 lanes on every operator above.
inline int gsLanes(int width, int count) {
  int L = 1;
  while (L < 64 && (width > L * (kGsUnroll / 2) || ((long long)count * L < (1 << 16) && width > 2 * L))) L *= 2;
  return L;
}

// Tiled slots of the chosen half of a coloured CSR operator (rows of colour
// c: rows[off[c]..off[c+1]), or those indices themselves when rows is null).
// Colours are independent: they are counted, then filled, in parallel.
struct GsLayout {
  std::vector<GsColour> colour;
  std::vector<int> col, src;  // column (-1 where unused), CSR position (-1 where unused)
};

template <class TI>
GsLayout gsLayout(int ncolors, const std::vector<int>& off, const int* rows, const std::vector<int>& colorOf,
                  const TI* row, const int* col, GsHalf half) {
  GsLayout G;
  G.colour.resize((std::size_t)ncolors);
  auto wanted = [&](int i, int j, int c) {
    if (j == i) return false;
    const int cj = colorOf[(std::size_t)j];
    return half == GsHalf::all || (half == GsHalf::lower ? cj < c : cj > c);
  };
  auto eachColour = [&](auto&& body) {
    const int nt = std::max(1, std::min(ncolors, off.back() < 4096 ? 1 : hostThreads(0)));
    std::vector<std::thread> pool;
    for (int t = 0; t < nt; ++t)
      pool.emplace_back([&, t]() {
        for (int c = t; c < ncolors; c += nt) body(c, off[(std::size_t)c], off[(std::size_t)c + 1] - off[(std::size_t)c]);
      });
    for (std::thread& th : pool) th.join();
  };
  eachColour([&](int c, int b, int n) {
    int width = 1;
    for (int q = 0; q < n; ++q) {
      const int i = rows ? rows[b + q] : b + q;
      int w = 0;
      for (TI k = row[i]; k < row[i + 1]; ++k) w += wanted(i, col[k], c) ? 1 : 0;
      width = std::max(width, w);
    }
    GsColour& C = G.colour[(std::size_t)c];
    C.L = gsLanes(width, n);
    C.U = (width + C.L - 1) / C.L;
    if (C.U > kGsUnroll) C.U = (C.U + kGsUnroll - 1) / kGsUnroll * kGsUnroll;
  });
  long long tiles = 0;
  for (int c = 0; c < ncolors; ++c) {
    GsColour& C = G.colour[(std::size_t)c];
    const int n = off[(std::size_t)c + 1] - off[(std::size_t)c], per = 64 / C.L;
    C.tile = (int)tiles;
    tiles += (long long)((n + per - 1) / per) * C.U;
    require(tiles < (1ll << 31), "Gauss-Seidel slots too large for int32 tile indices");
  }
  G.col.assign((std::size_t)tiles * 64, -1);
  G.src.assign((std::size_t)tiles * 64, -1);
  eachColour([&](int c, int b, int n) {
    const GsColour& C = G.colour[(std::size_t)c];
    const int per = 64 / C.L;
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
  });
  return G;
}

// Slot values gathered from the CSR values they mirror.
template <class TO, class TI>
__global__ void __launch_bounds__(256) k_gs_fill(long long n, const int* __restrict__ src, const TI* __restrict__ val,
                                                 TO* __restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int s = src[i];
  out[i] = s >= 0 ? (TO)val[s] : TO{};
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

// Device slots of one half of an operator.
template <class TM>
struct GsSlots {
  std::vector<GsColour> colour;
  DBuf<int> col, src;
  DBuf<TM> val;
  // With the operator's values when they are fixed; otherwise fill() them.
  void upload(const GsLayout& G, const TM* csr) {
    colour = G.colour;
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

}  // namespace dev
}  // namespace nodals
