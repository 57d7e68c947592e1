// The multi-point Spalding fit of sst_physics.hpp (fitActive, fitProfile5)
// with eight lanes a wall point, for gfx950.
//
// Lane m of a group owns active sample m: its pointwise root, and its term of
// every objective, gradient and Hessian evaluation.  The terms are then
// gathered from the lanes and summed in sample order by the same
// expressions, so all lanes of a group take the same branches and the search
// takes the steps of the one-thread fit; what the compiler fuses may round
// differently, which the golden section's branches can turn into its
// resolution of 1e-5.  The fit is a serial chain of exponentials; five of its
// six evaluations a step run side by side here.
#pragma once

#include "sst_physics.hpp"

namespace nodals {
namespace dev {

constexpr int kFitLanes = 8;

// Sum of r_m^2 over samples m < n in order, / n; 1e300 for a non-finite one.
__device__ inline double fitMeanSquare(double r, int n) {
  double J = 0.0;
  bool finite = true;
  for (int m = 0; m < n; ++m) {
    const double rm = __shfl(r, m, kFitLanes);
    finite = finite && isfinite(rm);
    J += rm * rm;
  }
  return finite ? J / (double)n : 1.0e300;
}

// U, y: this lane's sample.
__device__ inline double fitObjective(double U, double y, int n, double nu, double ut) {
  if (!(ut > 0.0) || !(nu > 0.0) || !isfinite(ut)) return 1.0e300;
  return fitMeanSquare(sst::yPlusOf(U / ut, sst::kKappa, sst::kB) - y * ut / nu, n);
}

__device__ inline bool fitGaussNewton(double U, double y, int n, double nu, double ut, double& J, double& g,
                                      double& h) {
  if (!(nu > 0.0 && ut > 0.0) || !isfinite(ut)) return false;
  const double up = U / ut;
  const double r = sst::yPlusOf(up, sst::kKappa, sst::kB) - y * ut / nu;
  const double dr = -(up / ut) * sst::dYPlusOf(up, sst::kKappa, sst::kB) - y / nu;
  double sum = 0.0;
  g = 0.0;
  h = 0.0;
  bool finite = true;
  for (int m = 0; m < n; ++m) {
    const double rm = __shfl(r, m, kFitLanes), dm = __shfl(dr, m, kFitLanes);
    finite = finite && isfinite(rm) && isfinite(dm);
    sum += rm * rm;
    g += rm * dm;
    h += dm * dm;
  }
  J = sum / (double)n;
  return finite && isfinite(J) && isfinite(g) && isfinite(h);
}

// fitActive with the speeds as signed speeds; U, y: lane m's active sample (lanes past
// n repeat sample n - 1).  Every lane returns the group's profile.
__device__ inline sst::Profile fitActiveGroup(double U, double y, int n, double nu) {
  sst::Profile p{0, 0, 0, 0, 0, 0, 0};
  if (n < 1 || n > 5 || !(nu > 0.0)) return p;
  double root = 0.0, yp = 0.0, bt = 0.0;
  const bool rooted = sst::spaldingRoot(U, y, nu, root, yp, bt) && root > 0.0 && isfinite(root);
  double minRoot = 1.0e300, maxRoot = 0.0, sumRoot = 0.0, Umax = 0.0, yPrev = 0.0;
  int nRoot = 0;
  bool ok = true;
  for (int m = 0; m < n; ++m) {
    const double Um = __shfl(U, m, kFitLanes), ym = __shfl(y, m, kFitLanes), rm = __shfl(root, m, kFitLanes);
    const int has = __shfl(rooted ? 1 : 0, m, kFitLanes);
    if (n < 5) ok = ok && ym > 0.0 && isfinite(ym) && isfinite(Um) && (m == 0 || ym > yPrev);
    else ok = ok && (m == 0 || yPrev < ym);
    yPrev = ym;
    Umax = fmax(Umax, Um);
    if (has) {
      minRoot = fmin(minRoot, rm);
      maxRoot = fmax(maxRoot, rm);
      sumRoot += rm;
      ++nRoot;
    }
  }
  if (!ok) return p;
  const int mid = n / 2;
  const double yMid = __shfl(y, mid, kFitLanes);
  p.uMid = __shfl(U, mid, kFitLanes);
  if (Umax <= 1.0e-14) {
    p.beta = nu / yMid;
    p.valid = isfinite(p.beta) && p.beta > 0.0;
    return p;
  }
  double scale = nRoot > 0 ? sumRoot / (double)nRoot : sqrt(nu * Umax / fmax(yMid, 1.0e-30));
  if (!(scale > 0.0) || !isfinite(scale)) scale = 1.0;
  double lo = fmax(0.05 * scale, 1.0e-10);
  double hi = fmax(20.0 * scale, 100.0 * lo);
  if (nRoot > 0) {
    lo = fmax(fmin(lo, 0.20 * minRoot), 1.0e-10);
    hi = fmax(hi, 5.0 * maxRoot);
  }
  double ut = fmin(hi, fmax(lo, scale));
  bool gnOK = true;
  for (int it = 0; it < 12; ++it) {
    double J0 = 0.0, g = 0.0, h = 0.0;
    if (!fitGaussNewton(U, y, n, nu, ut, J0, g, h) || J0 >= 1.0e299 || !(h > 0.0)) {
      gnOK = false;
      break;
    }
    double step = g / h;
    double trial = fmin(hi, fmax(lo, ut - step));
    double Jt = fitObjective(U, y, n, nu, trial);
    for (int ls = 0; ls < 10 && (!isfinite(Jt) || Jt >= 1.0e299 || Jt > J0); ++ls) {
      step *= 0.5;
      trial = fmin(hi, fmax(lo, ut - step));
      Jt = fitObjective(U, y, n, nu, trial);
    }
    if (!isfinite(Jt) || Jt >= 1.0e299 || Jt > J0) {
      gnOK = false;
      break;
    }
    const double rel = fabs(trial - ut) / fmax(ut, 1.0e-30);
    ut = trial;
    if (rel < 1.0e-10) break;
  }
  double J = fitObjective(U, y, n, nu, ut);
  if (!gnOK || !(ut > 0.0) || !isfinite(ut) || !isfinite(J) || J >= 1.0e299) {
    // golden-section search on log(ut) over [lo, hi]
    double xa = log(lo), xb = log(hi);
    const double phi = 0.6180339887498948482;
    double x1 = xb - phi * (xb - xa), x2 = xa + phi * (xb - xa);
    double f1 = fitObjective(U, y, n, nu, exp(x1));
    double f2 = fitObjective(U, y, n, nu, exp(x2));
    for (int it = 0; it < 28; ++it) {
      if (f1 <= f2) {
        xb = x2;
        x2 = x1;
        f2 = f1;
        x1 = xb - phi * (xb - xa);
        f1 = fitObjective(U, y, n, nu, exp(x1));
      } else {
        xa = x1;
        x1 = x2;
        f1 = f2;
        x2 = xa + phi * (xb - xa);
        f2 = fitObjective(U, y, n, nu, exp(x2));
      }
    }
    ut = exp(f1 <= f2 ? x1 : x2);
    J = f1 <= f2 ? f1 : f2;
  }
  if (!(ut > 0.0) || !isfinite(ut) || !isfinite(J) || J >= 1.0e299) return p;
  p.uTau = ut;
  p.yPlus = yMid * ut / nu;
  const double Ua = fabs(p.uMid);
  p.beta = Ua > 1.0e-14 ? ut * ut / Ua : nu / yMid;
  p.fitRms = sqrt(fmax(J, 0.0));
  p.span = (nRoot >= 2 && maxRoot >= minRoot && minRoot < 1.0e299) ? (maxRoot - minRoot) / fmax(ut, 1.0e-30) : 0.0;
  p.valid = isfinite(p.yPlus) && isfinite(p.beta) && p.beta > 0.0 && isfinite(p.fitRms) && isfinite(p.span);
  return p;
}

}  // namespace dev
}  // namespace nodals
