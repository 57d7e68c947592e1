// k-omega SST volume terms of one tetrahedron for the scalar k or omega
// equation, on the P1+BF3 element (4 vertex + 4 face-bubble functions):
//   A_ab = sum_q w_q det [ D_q grad(phi_a).grad(phi_b) + R_q phi_a phi_b ]
//   b_a  = sum_q w_q det S_q phi_a
// with D = sigma_{k|w} nu_t, R = beta* omega (k) or beta omega (omega),
// S = P_k (k) or the omega production plus cross diffusion, all from the
// SST-2003 local state at each of the 24 points of Keast's degree-6 rule
// (reference kernel sst_tet_volume,
// turbulence/sst_gpu_v2/source/puretet_profile5_eq5_hxt5b/modules/transport/
// tet_volume_kernel.inc:1-30, with volume_coefficients,
// modules/transport/portable/transport_core.hpp:14-25).  Every cell writes
// its own 8x8 block (no atomics).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <vector>

#include "la_kernels.hpp"
#include "sst_physics.hpp"

namespace nodals {

// Keast's 24-point rule on the reference tetrahedron (degree 6; weights sum
// to 1/6): three 4-point orbits (a,a,a,b) and one 12-point orbit of the
// distinct permutations of (a,a,b,c), in the point order of the reference
// table (hxt5a_mixlen.cuh:37-142).  Rows of (l0, l1, l2, l3, w).
inline std::vector<double> keast24() {
  std::vector<double> q;
  auto put = [&](const double l[4], double w) {
    for (int i = 0; i < 4; ++i) q.push_back(l[i]);
    q.push_back(w);
  };
  struct Orbit {
    double a, b, w;
    bool bFirst;  // b at slot i (else at slot 3 - i) for point i of the orbit
  };
  const Orbit o4[3] = {{0.214602871259151673, 0.356191386222544926, 0.00665379170969464511, false},
                       {0.0406739585346113375, 0.87797812439616596, 0.00167953517588677629, false},
                       {0.322337890142275652, 0.0329863295731730594, 0.00922619692394239903, true}};
  for (const Orbit& o : o4)
    for (int i = 0; i < 4; ++i) {
      double l[4] = {o.a, o.a, o.a, o.a};
      l[o.bFirst ? i : 3 - i] = o.b;
      put(l, o.w);
    }
  const double v[3] = {0.0636610018750175255, 0.269672331458315873, 0.603005664791649076};
  std::array<int, 4> rank = {0, 0, 1, 2};
  do {
    const double l[4] = {v[rank[0]], v[rank[1]], v[rank[2]], v[rank[3]]};
    put(l, 0.00803571428571428319);
  } while (std::next_permutation(rank.begin(), rank.end()));
  return q;
}

namespace dev {

constexpr int kSstQ = 24;

// P1 + face-bubble basis (bubble i opposite vertex i: 27 prod_{j != i} l_j)
// and its reference gradients.
__device__ inline void p1bf3Basis(const double l[4], double phi[8], double gr[8][3]) {
  const double gl[4][3] = {{-1, -1, -1}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
  for (int i = 0; i < 4; ++i) {
    phi[i] = l[i];
    for (int d = 0; d < 3; ++d) gr[i][d] = gl[i][d];
  }
  for (int i = 0; i < 4; ++i) {
    int js[3], k = 0;
    for (int j = 0; j < 4; ++j)
      if (j != i) js[k++] = j;
    phi[4 + i] = 27.0 * l[js[0]] * l[js[1]] * l[js[2]];
    for (int d = 0; d < 3; ++d)
      gr[4 + i][d] = 27.0 * (gl[js[0]][d] * l[js[1]] * l[js[2]] + l[js[0]] * gl[js[1]][d] * l[js[2]] +
                             l[js[0]] * l[js[1]] * gl[js[2]][d]);
  }
}

// Inputs per cell: DOF refs (>= 0 device free DOF, < 0 -(fixed slot + 1)),
// invJ (row-major dxi_j/dx_d), det, the (x, y) of the four vertices relative
// to the pipe axis; fields: velocity (xyz interleaved, free and fixed) and
// k, omega (free and fixed).  Outputs: mat[c][64], rhs[c][8].
// Transport-step form: with sref (scalar DOF of every cell basis) k and
// omega are read as kf[sref], wf[sref]; nuBase is added to the diffusion
// coefficient (the molecular part, which Keast's rule integrates exactly
// for this basis) and conv[c][64], when given, is added to the matrix (conv
// may be mat itself: every lane reads and writes only its own entry).
// equation 2 is the momentum form: the eddy-viscosity diffusion block
// sum_q w_q det nu_t grad phi_a . grad phi_b only (no reaction, no rhs).
// With dmat (momentum form only) every cell also writes the deviatoric
// cross-component tensor of the implicit deviatoric stress
// (modules/coupling/implicit_dev_volume_tet.inc:1-68):
//   dmat[c][ab][3i+j] = sum_q w_q det (nu + nu_t)
//                       (d_j phi_a d_i phi_b - (2/3) d_i phi_a d_j phi_b).
//
// Two cells per wavefront, 32 lanes a cell, one lane a quadrature point (the
// last eight idle with zero weights).  A lane evaluates its point, forms all 64
// products of the block from registers, and a transposing reduction over the
// 32 lanes leaves entries 2l and 2l + 1 in lane l, so the block is written
// in one coalesced store and no LDS is needed.  The point evaluation (the SST
// state, two tanh and a dozen divisions) is then the time.  The form with
// 24 of 64 lanes evaluating and 64 lanes each looping over points staged in
// LDS took 334 us on the 40k pipe; this one 104 us.
//
// The deviatoric tensor is the 24 x 24 product G^T N G of the points'
// gradients (row 3a + i): DMAT stages G and N in LDS and forms it with
// v_mfma_f64_16x16x4 (four tiles, six steps; operand lane l supplies row l%16
// of k = l/16, accumulator register r holds row l/16 + 4r, column l%16), then
// combines entries (3a+j, 3b+i) and (3a+i, 3b+j) from LDS.  On the 207k helix
// an iteration's three calls (one with the tensor) took 6.6 ms, now 1.9 ms.
struct SstVolArgs {
  int nc;
  const int* cref;
  const double *cinvJ, *cdet, *cxy, *u, *ufix, *kf, *kfix, *wf, *wfix, *quad;
  double radius, nu;
  int equation;
  double kFloor, omFloor;
  int deviatoric;
  double *mat, *rhs;
  const int* sref;
  double nuBase;
  const double *conv, *vdist;
  double* dmat;
};

typedef double f64x4 __attribute__((ext_vector_type(4)));

template <bool DMAT>
static __global__ void __launch_bounds__(256, 2) k_sst_volume(SstVolArgs A) {
  constexpr int kComp = 24, kPad = 25;  // a point's gradient components, padded rows
  __shared__ double GS[DMAT ? 8 * kSstQ * kPad : 1], NS[DMAT ? 8 * kSstQ : 1];
  const int lane = threadIdx.x & 63, half = lane >> 5, lq = lane & 31;
  const int wave = threadIdx.x >> 6, slot = 2 * wave + half;
  const int cell = blockIdx.x * 8 + slot;
  const bool live = cell < A.nc;
  const int c = live ? cell : A.nc - 1;
  const bool point = live && lq < kSstQ;
  const double* Q = A.quad + 5 * (lq < kSstQ ? lq : 0);
  const double l[4] = {Q[0], Q[1], Q[2], Q[3]};
  double phi[8], G[8][3];
  double DWq, RWq, SWq, NWq;
  {
    double gr[8][3];
    p1bf3Basis(l, phi, gr);
    const double* I = A.cinvJ + (long long)c * 9;
    double gu[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, gk[3] = {0, 0, 0}, gw[3] = {0, 0, 0}, kv = 0, wvv = 0;
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const int r = A.cref[(long long)c * 8 + a];
      const double* U = r >= 0 ? A.u + 3ll * r : A.ufix + 3ll * (-r - 1);
      double Ka, Wa;
      if (A.sref) {
        const int g = A.sref[(long long)c * 8 + a];
        Ka = A.kf[g];
        Wa = A.wf[g];
      } else {
        Ka = r >= 0 ? A.kf[r] : A.kfix[-r - 1];
        Wa = r >= 0 ? A.wf[r] : A.wfix[-r - 1];
      }
      const double pa = phi[a];
      kv += Ka * pa;
      wvv += Wa * pa;
      for (int d = 0; d < 3; ++d) {
        const double gd = gr[a][0] * I[d] + gr[a][1] * I[3 + d] + gr[a][2] * I[6 + d];
        G[a][d] = gd;
        gk[d] += Ka * gd;
        gw[d] += Wa * gd;
        gu[d] += U[0] * gd;
        gu[3 + d] += U[1] * gd;
        gu[6 + d] += U[2] * gd;
      }
    }
    double dq;
    if (A.vdist) {  // P1 interpolation of the vertex wall-distance field
      double dd = 0;
      for (int a = 0; a < 4; ++a) dd += l[a] * A.vdist[A.sref[(long long)c * 8 + a]];
      dq = sst::floorDistance(fmax(0.0, dd), A.radius);
    } else {
      double xq = 0, yq = 0;
      for (int a = 0; a < 4; ++a) {
        xq += l[a] * A.cxy[(long long)c * 8 + 2 * a];
        yq += l[a] * A.cxy[(long long)c * 8 + 2 * a + 1];
      }
      dq = sst::pipeDistance(xq, yq, A.radius);
    }
    const sst::Local s = sst::local(dq, A.nu, gu, kv, wvv, gk, gw, A.kFloor, A.omFloor, A.deviatoric != 0);
    const double wt = A.cdet[c] * Q[4];
    const bool isK = A.equation == 0;
    if (A.equation == 2) {
      DWq = wt * s.nut;
      RWq = 0.0;
      SWq = 0.0;
      NWq = (A.nu + s.nut) * wt;
    } else {
      DWq = wt * ((isK ? s.sigmaK : s.sigmaW) * s.nut + A.nuBase);
      RWq = wt * (isK ? s.reactK : s.reactOmega);
      SWq = wt * (isK ? s.pk : s.srcOmega);
      NWq = 0.0;
    }
    if (!point) DWq = RWq = SWq = NWq = 0.0;
  }
  if (DMAT) {
    if (lq < kSstQ) {
      double* g = GS + ((long long)slot * kSstQ + lq) * kPad;
      for (int a = 0; a < 8; ++a)
        for (int d = 0; d < 3; ++d) g[3 * a + d] = G[a][d];
      NS[slot * kSstQ + lq] = NWq;
    }
  }
  {
    double v[64];
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const double h0 = DWq * G[a][0], h1 = DWq * G[a][1], h2 = DWq * G[a][2], hp = RWq * phi[a];
#pragma unroll
      for (int b = 0; b < 8; ++b) v[8 * a + b] = h0 * G[b][0] + h1 * G[b][1] + h2 * G[b][2] + hp * phi[b];
    }
    laneReduceScatter<64, 32>(v, lane);
    if (live) {
      const long long o = (long long)c * 64 + 2 * lq;
      A.mat[o] = A.conv ? v[0] + A.conv[o] : v[0];
      A.mat[o + 1] = A.conv ? v[1] + A.conv[o + 1] : v[1];
    }
  }
  if (A.rhs) {
    double r[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) r[a] = SWq * phi[a];
#pragma unroll
    for (int p = 0; p < 4; ++p) r[p] = mirrorPair<0x140>(r[p], r[p + 4], lane & 8);
#pragma unroll
    for (int p = 0; p < 2; ++p) r[p] = mirrorPair<0x141>(r[p], r[p + 2], lane & 4);
    r[0] = mirrorPair<0x1B>(r[0], r[1], lane & 2);
    r[0] += dppMove<0xB1>(r[0]);
    r[0] = swapAdd16(r[0]);
    if (live && lq < 16 && !(lq & 1)) A.rhs[(long long)c * 8 + (lq >> 1)] = r[0];
  }
  if (DMAT) {
    __syncthreads();
    // both cells of the wavefront in turn: O = G^T N G, 24 x 24
    const int i = lane & 15, kk = lane >> 4;
    f64x4 acc[2][2][2];
#pragma unroll
    for (int z = 0; z < 2; ++z) {
      const double* g = GS + (long long)(2 * wave + z) * kSstQ * kPad;
      const double* n = NS + (2 * wave + z) * kSstQ;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[z][x][y] = f64x4{0, 0, 0, 0};
      const int i1 = 16 + (i & 7);  // rows 24..31 of the second tile repeat 16..23 and are not used
#pragma unroll
      for (int k0 = 0; k0 < kSstQ; k0 += 4) {
        const double* gk = g + (k0 + kk) * kPad;
        const double nk = n[k0 + kk], b0 = gk[i], b1 = gk[i1];
        const double a0 = nk * b0, a1 = nk * b1;
        acc[z][0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[z][0][0], 0, 0, 0);
        acc[z][0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[z][0][1], 0, 0, 0);
        acc[z][1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[z][1][0], 0, 0, 0);
        acc[z][1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[z][1][1], 0, 0, 0);
      }
    }
    __syncthreads();
    // the products replace the gradients: row p of a cell at p * kPad
#pragma unroll
    for (int z = 0; z < 2; ++z) {
      double* O = GS + (long long)(2 * wave + z) * kSstQ * kPad;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int p = 16 * x + kk + 4 * r, q = 16 * y + i;
            if (p < kComp && q < kComp) O[p * kPad + q] = acc[z][x][y][r];
          }
    }
    __syncthreads();
    const int a = lane >> 3, b = lane & 7;
#pragma unroll
    for (int z = 0; z < 2; ++z) {
      const int cz = blockIdx.x * 8 + 2 * wave + z;
      if (cz >= A.nc) break;
      const double* O = GS + (long long)(2 * wave + z) * kSstQ * kPad;
      double* D = A.dmat + ((long long)cz * 64 + lane) * 9;
      for (int ii = 0; ii < 3; ++ii)
        for (int j = 0; j < 3; ++j)
          D[3 * ii + j] = O[(3 * a + j) * kPad + 3 * b + ii] - (2.0 / 3.0) * O[(3 * a + ii) * kPad + 3 * b + j];
    }
  }
}

inline void launchSstVolume(hipStream_t s, const SstVolArgs& A) {
  if (A.dmat) hipLaunchKernelGGL((k_sst_volume<true>), (A.nc + 7) / 8, 256, 0, s, A);
  else hipLaunchKernelGGL((k_sst_volume<false>), (A.nc + 7) / 8, 256, 0, s, A);
  NODALS_LAUNCHED();
}

}  // namespace dev
}  // namespace nodals
