// Host layout of the tiled Gauss-Seidel slots (device/gs_ell.hpp): which CSR
// entry of a coloured operator goes into which slot.
#pragma once

#include <algorithm>
#include <exception>
#include <numeric>
#include <system_error>
#include <thread>
#include <vector>

#include "error.hpp"
#include "h8_setup.hpp"

namespace nodals {
namespace dev {

constexpr int kGsUnroll = 8;  // most slots a lane loads before it gathers

// Which off-diagonal entries of a row a layout holds.
enum class GsHalf { lower, upper, all };

// Rows of one colour that share their slots' shape: rows [begin, begin + count)
// of the row list, L lanes a row, U slots a lane (at most kGsUnroll, or a
// multiple of it), the first tile.
struct GsClass {
  int begin = 0, count = 0, tile = 0, L = 1, U = 1;
  long long tiles() const { return (long long)((count + 64 / L - 1) / (64 / L)) * U; }
};

// Lanes a row for `count` rows of at most `width` entries: the fewest that
// leave a lane at most kGsUnroll/2 slots, widened while the colour is too
// small to give every SIMD a wavefront (2^16 threads) and a lane still holds
// two: within 4% of the best of 1..64 lanes on every operator listed in
// gs_ell.hpp.
inline int gsLanes(int width, int count) {
  int L = 1;
  while (L < 64 && (width > L * (kGsUnroll / 2) || ((long long)count * L < (1 << 16) && width > 2 * L))) L *= 2;
  return L;
}
inline GsClass gsClass(int begin, int count, int width) {
  GsClass C;
  C.begin = begin;
  C.count = count;
  C.L = gsLanes(std::max(width, 1), count);
  C.U = (std::max(width, 1) + C.L - 1) / C.L;
  if (C.U > kGsUnroll) C.U = (C.U + kGsUnroll - 1) / kGsUnroll * kGsUnroll;
  return C;
}

// A colour is one class, padded to its widest row, unless that takes more
// than kGsFill slots per entry and row and kGsSlack slots on top.  (The
// meshes' operators take 1.2 to 2.6 per entry; single small colours take up to
// 7, but an extra launch, 2 us, is what half a million slots cost.)  A colour
// with a few overlong rows would otherwise grow with their length times its
// rows: it is cut, its rows in descending order of width, into classes that
// each keep the bound.
constexpr long long kGsFill = 4, kGsSlack = 1 << 16;

// Tiled slots of the chosen half of a coloured CSR operator (rows of colour
// c: order[off[c]..off[c+1]), or those indices themselves when order is null).
// Colours are independent: they are counted, then filled, in parallel.
struct GsLayout {
  std::vector<std::vector<GsClass>> colour;
  std::vector<int> rows;      // own row list when a colour was split, else empty
  std::vector<int> col, src;  // column (-1 where unused), CSR position (-1 where unused)
};

template <class TI>
GsLayout gsLayout(int ncolors, const std::vector<int>& off, const int* order, const std::vector<int>& colorOf,
                  const TI* row, const int* col, GsHalf half) {
  GsLayout G;
  G.colour.resize((std::size_t)ncolors);
  std::vector<std::vector<int>> split((std::size_t)ncolors);  // row order of the colours that are cut
  auto wanted = [&](int i, int j, int c) {
    if (j == i) return false;
    const int cj = colorOf[(std::size_t)j];
    return half == GsHalf::all || (half == GsHalf::lower ? cj < c : cj > c);
  };
  // body(colour, first row, rows) for every colour.  What a worker throws is
  // thrown here after all have ended; slices that get no thread run here.
  auto eachColour = [&](auto&& body) {
    const int nt = std::max(1, std::min(ncolors, off.back() < 4096 ? 1 : hostThreads(0)));
    std::vector<std::exception_ptr> error((std::size_t)nt);
    auto slice = [&](int t) {
      try {
        for (int c = t; c < ncolors; c += nt) body(c, off[(std::size_t)c], off[(std::size_t)c + 1] - off[(std::size_t)c]);
      } catch (...) {
        error[(std::size_t)t] = std::current_exception();
      }
    };
    std::vector<std::thread> pool;
    pool.reserve((std::size_t)nt);
    int t = 1;
    try {
      for (; t < nt; ++t) pool.emplace_back(slice, t);
    } catch (const std::system_error&) {
    }
    slice(0);
    for (; t < nt; ++t) slice(t);
    for (std::thread& th : pool) th.join();
    for (const std::exception_ptr& e : error)
      if (e) std::rethrow_exception(e);
  };
  eachColour([&](int c, int b, int n) {
    if (n <= 0) return;
    std::vector<int> w((std::size_t)n, 0);
    int width = 0;
    long long entries = 0;
    for (int q = 0; q < n; ++q) {
      const int i = order ? order[b + q] : b + q;
      for (TI k = row[i]; k < row[i + 1]; ++k) w[(std::size_t)q] += wanted(i, col[k], c) ? 1 : 0;
      width = std::max(width, w[(std::size_t)q]);
      entries += w[(std::size_t)q];
    }
    std::vector<GsClass>& K = G.colour[(std::size_t)c];
    K.push_back(gsClass(b, n, width));
    if (K[0].tiles() * 64 <= kGsFill * (entries + n) + kGsSlack) return;
    K.clear();
    std::vector<int> q((std::size_t)n);
    std::iota(q.begin(), q.end(), 0);
    std::stable_sort(q.begin(), q.end(), [&](int x, int y) { return w[(std::size_t)x] > w[(std::size_t)y]; });
    for (int s = 0; s < n;) {  // the longest run from s that keeps the bound
      const int widest = w[(std::size_t)q[(std::size_t)s]];
      int best = s + 1;
      long long sum = 0;
      for (int e = s; e < n; ++e) {
        sum += w[(std::size_t)q[(std::size_t)e]];
        if (gsClass(0, e + 1 - s, widest).tiles() * 64 <= kGsFill * (sum + e + 1 - s) + 64 * kGsUnroll) best = e + 1;
      }
      K.push_back(gsClass(b + s, best - s, widest));
      s = best;
    }
    for (int& r : q) r = order ? order[b + r] : b + r;
    split[(std::size_t)c] = std::move(q);
  });
  long long tiles = 0;
  bool cut = false;
  for (int c = 0; c < ncolors; ++c) {
    cut = cut || !split[(std::size_t)c].empty();
    for (GsClass& C : G.colour[(std::size_t)c]) {
      C.tile = (int)tiles;
      tiles += C.tiles();
      require(tiles < (1ll << 31), "Gauss-Seidel slots too large for int32 tile indices");
    }
  }
  if (cut) {
    G.rows.resize((std::size_t)off.back());
    for (int c = 0; c < ncolors; ++c) {
      const std::vector<int>& q = split[(std::size_t)c];
      for (int b = off[(std::size_t)c], t = b; t < off[(std::size_t)c + 1]; ++t)
        G.rows[(std::size_t)t] = !q.empty() ? q[(std::size_t)(t - b)] : order ? order[t] : t;
    }
    order = G.rows.data();
  }
  G.col.assign((std::size_t)tiles * 64, -1);
  G.src.assign((std::size_t)tiles * 64, -1);
  eachColour([&](int c, int, int) {
    for (const GsClass& C : G.colour[(std::size_t)c]) {
      const int per = 64 / C.L;
      for (int q = 0; q < C.count; ++q) {
        const int i = order ? order[C.begin + q] : C.begin + q;
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
  });
  return G;
}

}  // namespace dev
}  // namespace nodals
