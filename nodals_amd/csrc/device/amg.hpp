// Device AMG V-cycle over a host-built SA hierarchy.
//
// Cycle structure of G4AMG::apply / explicit_vcycle
// (gpu/serial_cuda/h8_main_base.cu:532-564): smoothers start from zero, the
// post-smoother is applied as a correction to the current residual, the
// terminal level is a dense inverse mat-vec.  Restriction is a gather SpMV
// with the stored transpose P^T (no atomics), prolongation adds P x_c.
//
// Template parameters: TF is the storage type of the finest operator values
// (double, float or bf16), TV the type of every vector and of the coarse
// levels (double, or float for the mixed-precision hierarchy).
#pragma once

#include <cmath>
#include <string>
#include <vector>

#include "../host/amg_setup.hpp"
#include "amg_dense.hpp"
#include "gs_ell.hpp"
#include "la_kernels.hpp"

namespace nodals {
namespace dev {

struct SmootherOptions {
  std::string kind = "jacobi";  // jacobi | l1jacobi | cheb2 | mcgs
  double jacobiOmega = 0.7;
  int jacobiFineSweeps = 1, jacobiCoarseSweeps = 1;
  int chebDegree = 2;
  double lambdaLowFraction = 0.05;
  double mcgsOmega = 1.0;
  int mcgsFineSweeps = 1, mcgsCoarseSweeps = 1;
  std::string mcgsOrder = "symmetric";  // forward | backward | symmetric
};

// View of the finest operator, owned elsewhere (refreshed each SIMPLE step).
template <class TF, class TV>
struct FineView {
  int n = 0;
  int lanes = 16;
  const int* row = nullptr;
  const int* col = nullptr;
  const TF* val = nullptr;
  const TV* diag = nullptr;
  const TV* l1 = nullptr;
};

template <class TV>
struct DevColoring {
  int ncolors = 0;
  std::vector<int> off;
  DBuf<int> rows;
  bool contiguous = false;  // the operator is numbered in colour order: colour c is rows [off[c], off[c+1])
  void upload(const Coloring& C) {
    ncolors = C.ncolors;
    off = C.offset;
    rows.upload(C.rows);
    contiguous = false;
  }
  void uploadContiguous(const Coloring& C) {
    ncolors = C.ncolors;
    off = C.offset;
    contiguous = true;
  }
  const int* rowList() const { return contiguous ? nullptr : rows.data(); }
};

// The slots an MCGS smoothing call reads: the half that a pass from x = 0
// needs, the other half for symmetric sweeps, and every off-diagonal entry
// for the later sweeps of a one-directional order.
template <class TM>
struct GsOperator {
  GsSlots<TM> lower, upper, all;
  template <class TI>
  void build(int ncolors, const std::vector<int>& off, const int* rows, int n, const TI* row, const int* col,
             const std::string& order, int sweeps, const TM* csr) {
    std::vector<int> colorOf((std::size_t)n, 0);
    for (int c = 0; c < ncolors; ++c)
      for (int q = off[(std::size_t)c]; q < off[(std::size_t)c + 1]; ++q) colorOf[(std::size_t)(rows ? rows[q] : q)] = c;
    if (order != "backward") lower.upload(gsLayout(ncolors, off, rows, colorOf, row, col, GsHalf::lower), csr);
    if (order != "forward") upper.upload(gsLayout(ncolors, off, rows, colorOf, row, col, GsHalf::upper), csr);
    if (order != "symmetric" && sweeps > 1)
      all.upload(gsLayout(ncolors, off, rows, colorOf, row, col, GsHalf::all), csr);
  }
  template <class TI>
  void fill(hipStream_t s, const TI* csr) {
    for (GsSlots<TM>* g : {&lower, &upper, &all}) g->fill(s, csr);
  }
};

template <class TF, class TV>
class DevAmg {
 public:
  struct Level {
    int n = 0, lanes = 8;
    DBuf<int> row, col;
    DBuf<TV> val, diag, l1, b, x, r, tmp, corr;
    double lambda = 1.0;
    DevColoring<TV> color;
    GsOperator<TV> gs;
  };
  struct Xfer {
    int nFine = 0, nCoarse = 0, lanesP = 8, lanesT = 8;
    bool aggregation = false;  // exactly one entry per fine row (row i holds entry i)
    DBuf<int> prow, pcol, trow, tcol;
    DBuf<TV> pval, tval;
  };

  void setup(const AmgHierarchy& H, int fineN, const SmootherOptions& o, const Coloring* fineColoring) {
    opt_ = o;
    // A Jacobi count below one is one step; a multicolour count below one, or
    // an order that is none of the three, makes no pass (the smoother is zero).
    for (int* m : {&opt_.jacobiFineSweeps, &opt_.jacobiCoarseSweeps}) *m = std::max(*m, 1);
    const bool ordered = o.mcgsOrder == "forward" || o.mcgsOrder == "backward" || o.mcgsOrder == "symmetric";
    for (int* m : {&opt_.mcgsFineSweeps, &opt_.mcgsCoarseSweeps}) *m = ordered ? std::max(*m, 0) : 0;
    fineN_ = fineN;
    fineLambda_ = H.fineLambda;
    const std::size_t nl = H.A.size();
    require(nl >= 1 && H.P.size() == nl, "AMG hierarchy shape mismatch", kErrInternal);
    L_.clear();
    P_.clear();
    L_.resize(nl);
    P_.resize(nl);
    // An MCGS-smoothed coarse level is stored renumbered in colour order
    // (the reference's greedy colouring, unchanged): every colour is then
    // a contiguous row range and a colour pass needs no row list.  Each
    // row keeps its entries in their order, and the transfers on both
    // sides are relabelled the same way, so every sum is formed in the
    // same order as in the original numbering and results are identical.
    // perm[l][new] = original row; empty = not renumbered.
    std::vector<std::vector<int>> perm(nl), inv(nl);
    std::vector<Coloring> colors(nl);
    for (std::size_t l = 0; opt_.kind == "mcgs" && l + 1 < nl; ++l)
      colors[l] = greedyColoring(H.A[l].n, H.A[l].row.data(), H.A[l].col.data());
    dense_ = denseLevel(H, colors);
    std::vector<DenseSetupLevel> D(nl);
    for (std::size_t l = 0; l < nl; ++l) {
      const CsrD& A = H.A[l];
      Level& Lv = L_[l];
      Lv.n = A.n;
      Lv.lanes = lanesFor(A.n ? (double)A.col.size() / A.n : 1.0, A.n);
      if (opt_.kind == "mcgs" && l + 1 < nl) {
        const Coloring& C = colors[l];
        perm[l].assign(C.rows.begin(), C.rows.end());
        inv[l].assign((std::size_t)A.n, 0);
        for (int i = 0; i < A.n; ++i) inv[l][(std::size_t)perm[l][(std::size_t)i]] = i;
        Lv.color.uploadContiguous(C);
      }
      const std::vector<int>& pm = perm[l];
      const std::vector<int>& iv = inv[l];
      auto orig = [&](int i) { return pm.empty() ? i : pm[(std::size_t)i]; };
      auto relabel = [&](int j) { return iv.empty() ? j : iv[(std::size_t)j]; };
      std::vector<int> r32((std::size_t)A.n + 1, 0), c32;
      std::vector<double> v64, d64((std::size_t)A.n), l1((std::size_t)A.n);
      c32.reserve(A.col.size());
      v64.reserve(A.col.size());
      for (int i = 0; i < A.n; ++i) {
        const int o = orig(i);
        double s = 0;
        for (std::int64_t k = A.row[(std::size_t)o]; k < A.row[(std::size_t)o + 1]; ++k) {
          c32.push_back(relabel(A.col[(std::size_t)k]));
          v64.push_back(A.val[(std::size_t)k]);
          s += std::abs(A.val[(std::size_t)k]);
        }
        r32[(std::size_t)i + 1] = (int)c32.size();
        d64[(std::size_t)i] = A.diag[(std::size_t)o];
        l1[(std::size_t)i] = s;
      }
      Lv.row.upload(r32);
      Lv.col.upload(c32);
      Lv.val.upload(castVec(v64));
      if (opt_.kind == "mcgs" && (int)l < dense_) {
        Lv.gs.build(Lv.color.ncolors, Lv.color.off, nullptr, A.n, r32.data(), c32.data(), opt_.mcgsOrder,
                    opt_.mcgsCoarseSweeps, castVec(v64).data());
      }
      // levelSpmv() reads the operator, x and tmp of any level; the cycle
      // the rest, down to the right-hand side of the dense level
      for (DBuf<TV>* v : {&Lv.x, &Lv.tmp}) v->alloc((std::size_t)A.n);
      Lv.x.upload(std::vector<TV>((std::size_t)A.n, TV(1)));
      if ((int)l <= dense_) Lv.b.alloc((std::size_t)A.n);
      if ((int)l < dense_) {
        Lv.diag.upload(castVec(d64));
        Lv.l1.upload(castVec(l1));
        for (DBuf<TV>* v : {&Lv.r, &Lv.corr}) v->alloc((std::size_t)A.n);
      }
      Lv.lambda = l < H.levelLambda.size() ? H.levelLambda[l] : 1.0;
      if ((int)l >= dense_) {
        D[l].n = A.n;
        D[l].row = Lv.row.data();
        D[l].col = Lv.col.data();
        D[l].val.upload(v64);
        D[l].diag.upload(d64);
        D[l].l1.upload(l1);
        D[l].lambda = Lv.lambda;
        D[l].colorOff = Lv.color.off;
      }
    }
    static const std::vector<int> none;
    for (std::size_t l = 0; l < nl; ++l)
      uploadTransfer(H.P[l], (int)l <= dense_ ? &P_[l] : nullptr, l > 0 ? inv[l - 1] : none, inv[l],
                     (int)l > dense_ ? &D[l] : nullptr);
    termN_ = H.terminalN;
    {
      const int ld = denseLd(termN_);
      std::vector<TV> t((std::size_t)termN_ * ld, TV(0));
      for (int i = 0; i < termN_; ++i)
        for (int j = 0; j < termN_; ++j)
          t[(std::size_t)i * ld + j] = (TV)H.terminalInv[(std::size_t)i * termN_ + j];
      tinv_.upload(t);
    }
    if (dense_ < (int)nl - 1) buildDense(H, D);
    for (DBuf<TV>* v : {&fr_, &ftmp_, &fcorr_}) v->alloc((std::size_t)fineN);
    if (steps(true) >= 2) fx_.alloc((std::size_t)fineN);
    if (opt_.kind == "mcgs") {
      require(fineColoring != nullptr, "MCGS smoother requires a fine coloring", kErrInternal);
      fineColor_.upload(*fineColoring);
      for (DBuf<TV>* v : {&gsA_, &gsB_}) v->alloc((std::size_t)fineN);
    }
  }

  // The finest operator, with its pattern on the host (row[n + 1], col).  Call
  // fineChanged() whenever its values have changed.
  void setFine(const FineView<TF, TV>& v, const int* hostRow, const int* hostCol, const Coloring* C) {
    fine_ = v;
    if (opt_.kind == "mcgs")
      fineGs_.build(C->ncolors, C->offset, C->rows.data(), v.n, hostRow, hostCol, opt_.mcgsOrder, opt_.mcgsFineSweeps,
                    nullptr);
  }
  void fineChanged(hipStream_t s) { fineGs_.fill(s, fine_.val); }
  // tmp = A_l x on explicit level l (measurement of the coarse SpMV).
  void levelSpmv(hipStream_t s, int l) {
    Level& A = L_[(std::size_t)l];
    spmv<TV, TV, false, false>(s, A.lanes, A.n, A.row.data(), A.col.data(), A.val.data(), A.x.data(), nullptr,
                               A.tmp.data());
  }
  int levels() const { return (int)L_.size(); }
  const Level& level(int l) const { return L_[(std::size_t)l]; }

  // apply() replayed from a captured HIP graph (b and z must stay fixed
  // buffers; the finest values behind the fine view may change in place).
  void applyGraphed(hipStream_t s, const TV* b, TV* z) {
    graph_.run(s, graphKey({b, z, fine_.val, fine_.diag}), [&]() { apply(s, b, z); });
  }

  // z = M^{-1} b for FP64 vectors b, z, replayed from one captured graph per
  // (b, z) pair: with the fused cycles the FP64 <-> TV roundings happen
  // inside their first and last kernels (identical values to separate casts);
  // otherwise through the fixed TV buffers.  Returns false (nothing done)
  // when neither fused cycle serves the fine level.
  bool applyWide(hipStream_t s, const double* b, double* z) {
    if (!fusedJacobi() && steps(true) < 2) return false;
    wide_.run(s, graphKey({b, z, fine_.val, fine_.diag}), [&]() {
      if (fusedJacobi()) fusedCycle<double, double>(s, b, z);
      else stepCycle<double, double>(s, b, z);
    });
    return true;
  }

  // z = M^{-1} b on the finest level.
  void apply(hipStream_t s, const TV* b, TV* z) {
    if (fusedJacobi()) {
      fusedCycle<TV, TV>(s, b, z);
      return;
    }
    if (steps(true) >= 2) {
      stepCycle<TV, TV>(s, b, z);
      return;
    }
    smoothFine(s, b, z);
    spmv<TF, TV, true, false>(s, fine_.lanes, fine_.n, fine_.row, fine_.col, fine_.val, z, b, fr_.data());
    Level& C = L_[0];
    restrictTo(s, P_[0], fr_.data(), C.b.data());
    vcycle(s, 0, C.b.data(), C.x.data());
    prolongAdd(s, P_[0], C.x.data(), z);
    spmv<TF, TV, true, false>(s, fine_.lanes, fine_.n, fine_.row, fine_.col, fine_.val, z, b, fr_.data());
    smoothFine(s, fr_.data(), fcorr_.data());
    axpy<TV>(s, fine_.n, 1.0, fcorr_.data(), z);
  }

 private:
  // Steps of the Jacobi or Chebyshev smoother on the fine (coarse) levels; 0
  // for MCGS.
  int steps(bool fine) const {
    if (opt_.kind == "mcgs") return 0;
    const int m = opt_.kind == "cheb2" ? opt_.chebDegree : fine ? opt_.jacobiFineSweeps : opt_.jacobiCoarseSweeps;
    return std::max(m, 1);
  }
  double stepWeight(int k, double lambda) const {
    if (opt_.kind == "jacobi" || opt_.kind == "l1jacobi") return opt_.jacobiOmega;
    if (opt_.kind != "cheb2") fail("unknown AMG smoother " + opt_.kind);
    const double lo = opt_.lambdaLowFraction * lambda;
    require(lambda > lo && lo > 0, "Chebyshev interval invalid");
    return 1.0 / chebRoot(lambda, lo, k, opt_.chebDegree);
  }

  // Smoothing of two and more steps before and after the coarse correction,
  // each step one matrix pass: x = S b, r = b - A x ...
  template <class TM, class TB>
  void stepPre(hipStream_t s, const FineView<TM, TV>& A, int m, double lambda, const TB* b, TV* x, TV* other, TV* r) {
    const TV* den = opt_.kind == "l1jacobi" ? A.l1 : A.diag;
    TV *from = m % 2 == 1 ? x : other, *to = m % 2 == 1 ? other : x;  // the last step lands in x
    hipLaunchKernelGGL((k_jacobi_zero<TV, TB>), blocksFor(A.n), 256, 0, s, A.n, stepWeight(0, lambda), b, den, from);
    NODALS_LAUNCHED();
    for (int k = 1; k < m; ++k, std::swap(from, to))
      residJacobiPost<TM, TV, TB, TV>(s, A.lanes, A.n, A.row, A.col, A.val, b, den, stepWeight(k, lambda), from, to);
    residStep<kResid, TM, TV, TB>(s, A.lanes, A.n, A.row, A.col, A.val, b, den, 0.0, from, r, (TV*)nullptr,
                                  (const TV*)nullptr, (TV*)nullptr);
  }
  // ... and z = x + S (b - A x).
  template <class TM, class TB, class TZ>
  void stepPost(hipStream_t s, const FineView<TM, TV>& A, int m, double lambda, const TB* b, const TV* x, TV* r, TV* c,
                TV* other, TZ* z) {
    const TV* den = opt_.kind == "l1jacobi" ? A.l1 : A.diag;
    residStep<kFirst, TM, TV, TB>(s, A.lanes, A.n, A.row, A.col, A.val, b, den, stepWeight(0, lambda), x, r, c,
                                  (const TV*)nullptr, (TV*)nullptr);
    for (int k = 1; k < m - 1; ++k, std::swap(c, other))
      residJacobiPost<TM, TV, TV, TV>(s, A.lanes, A.n, A.row, A.col, A.val, r, den, stepWeight(k, lambda), c, other);
    residStep<kLast, TM, TV, TV, TZ>(s, A.lanes, A.n, A.row, A.col, A.val, r, den, stepWeight(m - 1, lambda), c,
                                     (TV*)nullptr, (TV*)nullptr, x, z);
  }
  template <class TB, class TZ>
  void stepCycle(hipStream_t s, const TB* b, TZ* z) {
    const int m = steps(true);
    stepPre<TF>(s, fine_, m, fineLambda_, b, fx_.data(), ftmp_.data(), fr_.data());
    restrictTo(s, P_[0], fr_.data(), L_[0].b.data());
    vcycle(s, 0, L_[0].b.data(), L_[0].x.data());
    prolongAdd(s, P_[0], L_[0].x.data(), fx_.data());
    stepPost<TF>(s, fine_, m, fineLambda_, b, fx_.data(), fr_.data(), fcorr_.data(), ftmp_.data(), z);
  }

  template <class TB, class TZ>
  // Pre-smoothing + residual, coarse correction, residual + post-smoothing:
  // two fine passes instead of five kernels.
  void fusedCycle(hipStream_t s, const TB* b, TZ* z) {
    const TV* den = opt_.kind == "l1jacobi" ? fine_.l1 : fine_.diag;
    jacobiPreResid<TF, TV, TB>(s, fine_.lanes, fine_.n, fine_.row, fine_.col, fine_.val, b, den, opt_.jacobiOmega,
                               ftmp_.data(), fr_.data());
    Level& C = L_[0];
    restrictTo(s, P_[0], fr_.data(), C.b.data());
    vcycle(s, 0, C.b.data(), C.x.data());
    const Xfer& X = P_[0];
    // The fine level keeps the prolongation as its own pass: folded into the
    // post-smoothing gather (as on the coarse levels) its two-level gather
    // made the 40k-cell solve about 1% slower once the row loops kept
    // several loads in flight.
    prolongAdd(s, X, C.x.data(), ftmp_.data());
    residJacobiPost<TF, TV, TB, TZ>(s, fine_.lanes, fine_.n, fine_.row, fine_.col, fine_.val, b, den,
                                    opt_.jacobiOmega, ftmp_.data(), z);
  }

  template <class TS>
  static std::vector<TV> castVec(const std::vector<TS>& v) {
    std::vector<TV> o(v.size());
    for (std::size_t i = 0; i < v.size(); ++i) o[i] = (TV)v[i];
    return o;
  }

  // Upload transfer P (fine rows -> coarse columns) and its transpose, with
  // the fine side relabelled by invF and the coarse side by invC (original
  // -> stored index; empty = unchanged).  Rows keep their entries' order;
  // the transpose is formed in the original numbering (within a coarse row,
  // fine rows ascend) and relabelled afterwards, so its sums keep the
  // original order too.
  // To X for the cycle, to D in FP64 (with the coarse side's level) for the
  // set-up of the dense operator.
  static void uploadTransfer(const Transfer& P, Xfer* X, const std::vector<int>& invF,
                             const std::vector<int>& invC, DenseSetupLevel* D) {
    auto relF = [&](int i) { return invF.empty() ? i : invF[(std::size_t)i]; };
    auto relC = [&](int c) { return invC.empty() ? c : invC[(std::size_t)c]; };
    std::vector<int> origF((std::size_t)P.nFine), origC((std::size_t)P.nCoarse);
    for (int i = 0; i < P.nFine; ++i) origF[(std::size_t)relF(i)] = i;
    for (int c = 0; c < P.nCoarse; ++c) origC[(std::size_t)relC(c)] = c;
    std::vector<int> pr((std::size_t)P.nFine + 1, 0), pc;
    std::vector<double> pv;
    pc.reserve(P.col.size());
    pv.reserve(P.col.size());
    for (int i = 0; i < P.nFine; ++i) {
      const int o = origF[(std::size_t)i];
      for (std::int64_t k = P.row[(std::size_t)o]; k < P.row[(std::size_t)o + 1]; ++k) {
        pc.push_back(relC(P.col[(std::size_t)k]));
        pv.push_back(P.val[(std::size_t)k]);
      }
      pr[(std::size_t)i + 1] = (int)pc.size();
    }
    // Transpose for gather restriction, in the original numbering.
    std::vector<int> tr((std::size_t)P.nCoarse + 1, 0);
    for (int c : P.col) ++tr[(std::size_t)c + 1];
    for (int c = 0; c < P.nCoarse; ++c) tr[(std::size_t)c + 1] += tr[(std::size_t)c];
    std::vector<int> tc(P.col.size());
    std::vector<double> tv(P.col.size());
    std::vector<int> cur(tr.begin(), tr.end() - 1);
    for (int i = 0; i < P.nFine; ++i)
      for (std::int64_t k = P.row[(std::size_t)i]; k < P.row[(std::size_t)i + 1]; ++k) {
        const int c = P.col[(std::size_t)k];
        const int z = cur[(std::size_t)c]++;
        tc[(std::size_t)z] = i;
        tv[(std::size_t)z] = P.val[(std::size_t)k];
      }
    // ... then its rows reordered by the coarse relabelling and its columns
    // relabelled on the fine side.
    std::vector<int> tr2((std::size_t)P.nCoarse + 1, 0), tc2;
    std::vector<double> tv2;
    tc2.reserve(tc.size());
    tv2.reserve(tc.size());
    for (int c = 0; c < P.nCoarse; ++c) {
      const int o = origC[(std::size_t)c];
      for (int k = tr[(std::size_t)o]; k < tr[(std::size_t)o + 1]; ++k) {
        tc2.push_back(relF(tc[(std::size_t)k]));
        tv2.push_back(tv[(std::size_t)k]);
      }
      tr2[(std::size_t)c + 1] = (int)tc2.size();
    }
    if (X) {
      X->nFine = P.nFine;
      X->nCoarse = P.nCoarse;
      X->aggregation = (std::size_t)P.nFine == P.col.size();
      for (int i = 0; X->aggregation && i < P.nFine; ++i)
        X->aggregation = P.row[(std::size_t)i] == i && P.row[(std::size_t)i + 1] == i + 1;
      X->prow.upload(pr);
      X->pcol.upload(pc);
      X->pval.upload(castVec(pv));
      X->lanesP = lanesFor(P.nFine ? (double)P.col.size() / P.nFine : 1.0, P.nFine);
      X->trow.upload(tr2);
      X->tcol.upload(tc2);
      X->tval.upload(castVec(tv2));
      X->lanesT = lanesFor(P.nCoarse ? (double)P.col.size() / P.nCoarse : 1.0, P.nCoarse);
    }
    if (D) {
      D->prow.upload(pr);
      D->pcol.upload(pc);
      D->pval.upload(pv);
      D->trow.upload(tr2);
      D->tcol.upload(tc2);
      D->tval.upload(tv2);
    }
  }

  // Coarsest-first level from which the cycle is one dense product: the
  // finest level whose product (n^2 values at 4.5 TB/s, 3 us of launch) costs
  // less than the launches it replaces (2.2 us each: with MCGS two smoothing
  // calls of a pass per colour, with the others their vector passes and
  // residuals; about five more per level for transfers and residuals; the
  // fused Jacobi cycle has four in all).  nl - 1, the terminal level, when no
  // other pays.  kDenseRows bounds what a hierarchy keeps (0.65 GB in FP64)
  // and its set-up, not where the product pays: with MCGS and a bound of
  // 24,000, three iterations of the wall-function loop took 362 -> 314 ms on a
  // helix of 289k cells (12,200 rows, 1.1 GB more; FP32 333 -> 276 ms, 0.6 GB
  // and 0.3 s of set-up more) and 453 -> 429 ms on one of 425k (17,300 rows,
  // 2.2 GB more).
  static constexpr int kDenseRows = 9000;
  int denseLevel(const AmgHierarchy& H, const std::vector<Coloring>& colors) const {
    const int nl = (int)H.A.size();
    double below = 3.0;  // us of the cycle below the level: the terminal product
    int best = nl - 1;
    for (int l = nl - 2; l >= 0; --l) {
      const CsrD& A = H.A[(std::size_t)l];
      if (A.n > kDenseRows) break;
      double launches = 5.0;
      if (opt_.kind == "mcgs") {
        launches += 2.0 * opt_.mcgsCoarseSweeps * colors[(std::size_t)l].ncolors *
                    (opt_.mcgsOrder == "symmetric" ? 2.0 : 1.0);
      } else if (!fusedJacobi()) {
        launches += 2.0 * (1.0 + 2.0 * (steps(false) - 1)) + 2.0;
      }
      below += 2.2 * launches;
      const double product = 3.0 + (double)A.n * denseLd(A.n) * sizeof(TV) / 4.5e6;
      if (product < below) best = l;
    }
    return best;
  }

  // Sets denseT_ to the cycle from level dense_ down, column block by column
  // block in FP64.
  void buildDense(const AmgHierarchy& H, std::vector<DenseSetupLevel>& D) {
    const int nl = (int)D.size(), n = D[(std::size_t)dense_].n, ld = denseLd(n);
    const int block = std::min(n, 1024);
    hipStream_t s = nullptr;
    NODALS_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    try {
      denseT_.alloc((std::size_t)n * ld);
      fill<TV>(s, (long long)n * ld, denseT_.data(), TV(0));
      for (int l = dense_; l < nl; ++l) {
        DenseSetupLevel& L = D[(std::size_t)l];
        for (DBuf<double>* v : {&L.b, &L.x, &L.r, &L.corr}) v->alloc((std::size_t)L.n * block);
      }
      DBuf<double> tinv;
      tinv.upload(H.terminalInv);
      DenseSetupLevel& T = D[(std::size_t)dense_];
      for (int c0 = 0; c0 < n; c0 += block) {
        const int m = std::min(block, n - c0);
        const dim3 grid(n, (m + 255) / 256);
        hipLaunchKernelGGL(k_cols_unit, grid, 256, 0, s, m, c0, T.b.data());
        NODALS_LAUNCHED();
        colsCycle(s, D, dense_, m, tinv);
        hipLaunchKernelGGL(k_cols_store<TV>, grid, 256, 0, s, m, c0, ld, T.x.data(), denseT_.data());
        NODALS_LAUNCHED();
      }
      NODALS_HIP(hipStreamSynchronize(s));
      sweepScratch_.release();
    } catch (...) {
      (void)hipStreamSynchronize(s);
      (void)hipStreamDestroy(s);
      throw;
    }
    NODALS_HIP(hipStreamDestroy(s));
  }

  // vcycle() on m columns: D[l].x from D[l].b.
  void colsCycle(hipStream_t s, std::vector<DenseSetupLevel>& D, int l, int m, const DBuf<double>& tinv) {
    DenseSetupLevel& A = D[(std::size_t)l];
    const dim3 grid(A.n, (m + 255) / 256);
    if (l == (int)D.size() - 1) {
      hipLaunchKernelGGL(k_cols_dense, grid, 256, 0, s, A.n, m, tinv.data(), A.b.data(), A.x.data());
      NODALS_LAUNCHED();
      return;
    }
    DenseSetupLevel& C = D[(std::size_t)l + 1];
    colsSmooth(s, A, m, A.b.data(), A.x.data());
    hipLaunchKernelGGL((k_cols_spmv<1>), grid, 256, 0, s, m, A.row, A.col, A.val.data(), A.x.data(),
                       A.b.data(), A.r.data());
    hipLaunchKernelGGL((k_cols_spmv<0>), dim3(C.n, grid.y), 256, 0, s, m, C.trow.data(), C.tcol.data(), C.tval.data(),
                       A.r.data(), nullptr, C.b.data());
    NODALS_LAUNCHED();
    colsCycle(s, D, l + 1, m, tinv);
    hipLaunchKernelGGL((k_cols_spmv<2>), grid, 256, 0, s, m, C.prow.data(), C.pcol.data(), C.pval.data(), C.x.data(),
                       nullptr, A.x.data());
    hipLaunchKernelGGL((k_cols_spmv<1>), grid, 256, 0, s, m, A.row, A.col, A.val.data(), A.x.data(),
                       A.b.data(), A.r.data());
    NODALS_LAUNCHED();
    // the post-smoothing reads A.r and needs a residual of its own: A.b is
    // not read again
    colsSmooth(s, A, m, A.r.data(), A.corr.data());
    hipLaunchKernelGGL(k_cols_axpy, grid, 256, 0, s, m, A.corr.data(), A.x.data());
    NODALS_LAUNCHED();
  }

  // smooth() on m columns from x = 0.
  void colsSmooth(hipStream_t s, DenseSetupLevel& A, int m, const double* b, double* x) {
    const dim3 grid(A.n, (m + 255) / 256);
    if (opt_.kind == "mcgs") {
      fill<double>(s, (long long)A.n * m, x, 0.0);
      const int nc = (int)A.colorOff.size() - 1;
      auto pass = [&](bool reverse) {
        for (int q = 0; q < nc; ++q) {
          const int c = reverse ? nc - 1 - q : q;
          const int begin = A.colorOff[(std::size_t)c], count = A.colorOff[(std::size_t)c + 1] - begin;
          if (count <= 0) continue;
          hipLaunchKernelGGL(k_cols_gs, dim3(count, grid.y), 256, 0, s, m, begin, A.row, A.col,
                             A.val.data(), A.diag.data(), b, x, opt_.mcgsOmega);
          NODALS_LAUNCHED();
        }
      };
      for (int sw = 0; sw < opt_.mcgsCoarseSweeps; ++sw) {
        if (opt_.mcgsOrder != "backward") pass(false);
        if (opt_.mcgsOrder != "forward") pass(true);
      }
      return;
    }
    const int count = steps(false);
    const double* den = opt_.kind == "l1jacobi" ? A.l1.data() : A.diag.data();
    DBuf<double>& t = sweepScratch_;
    if (count > 1 && t.size() < (std::size_t)A.n * m) t.alloc((std::size_t)A.n * m);
    for (int k = 0; k < count; ++k) {
      const double w = stepWeight(k, A.lambda);
      const double* r = b;
      if (k > 0) {
        hipLaunchKernelGGL((k_cols_spmv<1>), grid, 256, 0, s, m, A.row, A.col, A.val.data(), x, b,
                           t.data());
        NODALS_LAUNCHED();
        r = t.data();
      }
      hipLaunchKernelGGL(k_cols_jacobi, grid, 256, 0, s, m, w, r, den, x, k > 0 ? 1 : 0);
      NODALS_LAUNCHED();
    }
  }

  void restrictTo(hipStream_t s, const Xfer& X, const TV* f, TV* c) {
    spmv<TV, TV, false, false>(s, X.lanesT, X.nCoarse, X.trow.data(), X.tcol.data(), X.tval.data(), f, nullptr, c);
  }
  void prolongAdd(hipStream_t s, const Xfer& X, const TV* c, TV* f) {
    spmv<TV, TV, false, true>(s, X.lanesP, X.nFine, X.prow.data(), X.pcol.data(), X.pval.data(), c, nullptr, f);
  }

  static double chebRoot(double hi, double lo, int k, int degree) {
    const double centre = .5 * (hi + lo), radius = .5 * (hi - lo);
    const double pi = 3.141592653589793238462643383279502884;
    return centre - radius * std::cos(pi * (2.0 * k + 1.0) / (2.0 * degree));
  }

  // MCGS smoothing from x = 0 (no pass reads an entry of x that an earlier
  // one has not written, so x is cleared only when there is no pass).  A
  // symmetric sweep's passes keep the row sum of the half that does not change
  // until the next pass.
  template <class TM>
  void mcgsSmooth(hipStream_t s, const GsOperator<TM>& G, const DevColoring<TV>& C, int sweeps, const TV* diag,
                  const TV* b, TV* x) {
    auto pass = [&](const GsSlots<TM>& S, bool reverse, const TV* other, TV* part, bool zero) {
      for (int q = 0; q < C.ncolors; ++q) {
        gsColour<TM, TV>(s, S, reverse ? C.ncolors - 1 - q : q, C.rowList(), diag, b, x, other, part, zero,
                         opt_.mcgsOmega);
      }
    };
    if (sweeps == 0) fill<TV>(s, C.off.back(), x, TV(0));
    const bool back = opt_.mcgsOrder == "backward";
    for (int sw = 0; sw < sweeps; ++sw) {
      const bool first = sw == 0, last = sw == sweeps - 1;
      if (opt_.mcgsOrder == "symmetric") {
        pass(G.lower, false, first ? nullptr : gsB_.data(), gsA_.data(), first);
        pass(G.upper, true, gsA_.data(), last ? nullptr : gsB_.data(), false);
      } else {
        pass(first ? (back ? G.upper : G.lower) : G.all, back, nullptr, nullptr, first);
      }
    }
  }

  // The one step of a one-step smoother, from x = 0.
  void smoothOnce(hipStream_t s, int n, const TV* diag, const TV* l1, double lambda, const TV* b, TV* x) {
    hipLaunchKernelGGL((k_jacobi_zero<TV, TV>), blocksFor(n), 256, 0, s, n, stepWeight(0, lambda), b,
                       opt_.kind == "l1jacobi" ? l1 : diag, x);
    NODALS_LAUNCHED();
  }

  void smoothFine(hipStream_t s, const TV* b, TV* x) {
    if (opt_.kind == "mcgs") {
      mcgsSmooth<TF>(s, fineGs_, fineColor_, opt_.mcgsFineSweeps, fine_.diag, b, x);
      return;
    }
    smoothOnce(s, fine_.n, fine_.diag, fine_.l1, fineLambda_, b, x);
  }

  void smoothLevel(hipStream_t s, Level& A, const TV* b, TV* x) {
    if (opt_.kind == "mcgs") {
      mcgsSmooth<TV>(s, A.gs, A.color, opt_.mcgsCoarseSweeps, A.diag.data(), b, x);
      return;
    }
    smoothOnce(s, A.n, A.diag.data(), A.l1.data(), A.lambda, b, x);
  }

  void vcycle(hipStream_t s, int l, const TV* b, TV* x) {
    Level& A = L_[(std::size_t)l];
    if (l == dense_) {  // the terminal level, or the whole sub-cycle in one product
      denseMv<TV>(s, A.n, dense_ == (int)L_.size() - 1 ? tinv_.data() : denseT_.data(), b, x);
      return;
    }
    if (fusedJacobi()) {
      const TV* den = opt_.kind == "l1jacobi" ? A.l1.data() : A.diag.data();
      jacobiPreResid<TV, TV>(s, A.lanes, A.n, A.row.data(), A.col.data(), A.val.data(), b, den, opt_.jacobiOmega,
                             A.tmp.data(), A.r.data());
      Level& C = L_[(std::size_t)l + 1];
      const Xfer& X = P_[(std::size_t)l + 1];
      restrictTo(s, X, A.r.data(), C.b.data());
      vcycle(s, l + 1, C.b.data(), C.x.data());
      if (X.aggregation) {
        residJacobiPostAgg<TV, TV>(s, A.lanes, A.n, A.row.data(), A.col.data(), A.val.data(), b, den,
                                   opt_.jacobiOmega, A.tmp.data(), X.pcol.data(), X.pval.data(), C.x.data(), x);
        return;
      }
      prolongAdd(s, X, C.x.data(), A.tmp.data());
      residJacobiPost<TV, TV>(s, A.lanes, A.n, A.row.data(), A.col.data(), A.val.data(), b, den, opt_.jacobiOmega,
                              A.tmp.data(), x);
      return;
    }
    if (const int m = steps(false); m >= 2) {
      FineView<TV, TV> V;
      V.n = A.n;
      V.lanes = A.lanes;
      V.row = A.row.data();
      V.col = A.col.data();
      V.val = A.val.data();
      V.diag = A.diag.data();
      V.l1 = A.l1.data();
      stepPre<TV>(s, V, m, A.lambda, b, x, A.tmp.data(), A.r.data());
      Level& C = L_[(std::size_t)l + 1];
      restrictTo(s, P_[(std::size_t)l + 1], A.r.data(), C.b.data());
      vcycle(s, l + 1, C.b.data(), C.x.data());
      prolongAdd(s, P_[(std::size_t)l + 1], C.x.data(), x);
      stepPost<TV>(s, V, m, A.lambda, b, x, A.r.data(), A.corr.data(), A.tmp.data(), x);
      return;
    }
    smoothLevel(s, A, b, x);
    spmv<TV, TV, true, false>(s, A.lanes, A.n, A.row.data(), A.col.data(), A.val.data(), x, b, A.r.data());
    Level& C = L_[(std::size_t)l + 1];
    restrictTo(s, P_[(std::size_t)l + 1], A.r.data(), C.b.data());
    vcycle(s, l + 1, C.b.data(), C.x.data());
    prolongAdd(s, P_[(std::size_t)l + 1], C.x.data(), x);
    spmv<TV, TV, true, false>(s, A.lanes, A.n, A.row.data(), A.col.data(), A.val.data(), x, b, A.r.data());
    smoothLevel(s, A, A.r.data(), A.corr.data());
    axpy<TV>(s, A.n, 1.0, A.corr.data(), x);
  }

  // One Jacobi sweep before and after on every level: the fused kernels.
  bool fusedJacobi() const {
    return (opt_.kind == "jacobi" || opt_.kind == "l1jacobi") && opt_.jacobiFineSweeps == 1 &&
           opt_.jacobiCoarseSweeps == 1;
  }

  SmootherOptions opt_;
  int fineN_ = 0;
  double fineLambda_ = 1.0;
  FineView<TF, TV> fine_;
  DevColoring<TV> fineColor_;
  GsOperator<TF> fineGs_;
  DBuf<TV> gsA_, gsB_;  // row sums kept between the passes of a symmetric sweep
  std::vector<Level> L_;
  std::vector<Xfer> P_;
  DBuf<TV> tinv_, denseT_;
  DBuf<double> sweepScratch_;  // dense set-up only
  int termN_ = 0, dense_ = 0;
  DBuf<TV> fr_, ftmp_, fcorr_, fx_;
  GraphCache graph_;
  GraphSet wide_;
};

}  // namespace dev
}  // namespace nodals
