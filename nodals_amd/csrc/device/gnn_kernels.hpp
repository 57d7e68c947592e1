// Kernels of the message-passing network that predicts the initial pressure
// correction: one kernel per layer and direction, the reduction of the
// gradient's partial sums, and Adam.
//
// Matrices are row-major FP32 in HBM with the row count padded to a multiple
// of 32.  GEMM inputs are rounded to BF16 (round to nearest even) as they go
// into the LDS tiles that feed the matrix cores; weights are kept as BF16
// copies of the FP32 master values.  All sums are FP32.
//
// v_mfma_f32_32x32x16_bf16 (gfx950): lane l supplies row l%32 of the 32x16
// A tile and column l%32 of the 16x32 B tile, each with the eight k values
// 8*(l/32) .. 8*(l/32)+7; accumulator register r of lane l holds output row
// 8*(r/4) + 4*(l/32) + r%4, column l%32.
//
// A row has 256 bytes per matrix and 16 kFLOP per layer, so the layers are
// bound by latency and memory passes: the neighbour mean is gathered straight
// into the GEMM's tile, the backward gather into the tile that feeds both
// gradient GEMMs, and one ReLU bit per entry replaces the pre-activations.
// Measured at 40,320 rows: forward 74 us (5 launches), backward 134 us (6),
// where separate mean, GEMM, mask, transposed-mean, column-sum and partial-sum
// kernels (a forward of 11, a backward of 31 launches) took about 900 us for
// both; a forward and a gradient call with their host copies 1.51 -> 0.60 ms.
#pragma once

#include "common.hpp"
#include "la_kernels.hpp"

namespace nodals {
namespace gnn {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWidth = 64, kTile = 64;  // features, and rows per block step

__device__ __forceinline__ short bfBits(float f) { return (short)floatToBf16(f).bits; }
__device__ __forceinline__ float bfRound(float f) { return bf16ToFloat(floatToBf16(f)); }

__device__ __forceinline__ f32x16 mfma(const s16x8& a, const s16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.0f;
  return z;
}
__device__ __forceinline__ int outRow(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }
__device__ __forceinline__ s16x4 bf4(float a, float b, float c, float d) {
  s16x4 v;
  v[0] = bfBits(a);
  v[1] = bfBits(b);
  v[2] = bfBits(c);
  v[3] = bfBits(d);
  return v;
}
// Eight BF16 of an LDS row whose stride keeps only 8-byte alignment.
__device__ __forceinline__ s16x8 ld8(const short* p) {
  const s16x4 a = *reinterpret_cast<const s16x4*>(p), b = *reinterpret_cast<const s16x4*>(p + 4);
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void add4(float4& a, const float4& b) {
  a.x += b.x;
  a.y += b.y;
  a.z += b.z;
  a.w += b.w;
}

// Four rows r .. r+3 of a block's tile, four features from c on, per thread:
// g[p] = sum over the neighbours of row r+p of F[neighbour][c .. c+3] in
// adjacency order, deg[p] its neighbours (rows >= n: none).  A tetrahedron has
// at most four, which are loaded together for all four rows; a longer list
// goes on one by one.
__device__ __forceinline__ void gather4(int n, int r, int c, const float* __restrict__ F, const int* __restrict__ off,
                                        const int* __restrict__ nbr, float4 (&g)[4], int (&deg)[4]) {
  int b[4], j[4][4];
  float4 v[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const bool in = r + p < n;
    b[p] = in ? off[r + p] : 0;
    deg[p] = in ? off[r + p + 1] - b[p] : 0;
  }
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) j[p][q] = nbr[q < deg[p] ? b[p] + q : 0];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) v[p][q] = ld4(F + (long long)j[p][q] * kWidth + c);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    g[p] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < deg[p]) add4(g[p], v[p][q]);
    for (int q = 4; q < deg[p]; ++q) add4(g[p], ld4(F + (long long)nbr[b[p] + q] * kWidth + c));
  }
}

// One ReLU bit per entry of a 32x32 output tile: word `nt` of its rows.
__device__ __forceinline__ void storeMask(const f32x16& z, int M, int r0, int nt, int lane, unsigned* __restrict__ mask) {
  unsigned word = 0u;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const unsigned long long bal = __ballot(z[r] > 0.0f);
    if ((lane & 31) == r) word = lane < 32 ? (unsigned)bal : (unsigned)(bal >> 32);
  }
  const int row = r0 + outRow(lane & 15, lane);
  if ((lane & 31) < 16 && row < M) mask[2 * row + nt] = word;
}

// H0 = relu(X W0 + b0), X (M x 16, rows >= n zero): one wavefront per 32 rows.
static __global__ void __launch_bounds__(256) k_encode(int M, const float* __restrict__ X, const bf16* __restrict__ Wt,
                                                       const float* __restrict__ bias, float* __restrict__ H,
                                                       unsigned* __restrict__ mask) {
  const int lane = threadIdx.x & 63;
  const int r0 = ((blockIdx.x * 256 + threadIdx.x) >> 6) * 32;
  if (r0 >= M) return;
  const int kh = (lane >> 5) * 8;
  const float* xp = X + (long long)(r0 + (lane & 31)) * 16 + kh;
  const float4 a0 = ld4(xp), a1 = ld4(xp + 4);
  const s16x8 av = __builtin_shufflevector(bf4(a0.x, a0.y, a0.z, a0.w), bf4(a1.x, a1.y, a1.z, a1.w), 0, 1, 2, 3, 4, 5,
                                           6, 7);
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int col = 32 * nt + (lane & 31);
    const s16x8 bv = *reinterpret_cast<const s16x8*>(reinterpret_cast<const short*>(Wt) + col * 16 + kh);
    f32x16 z = mfma(av, bv, zero16());
    const float bb = bias[col];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      z[r] += bb;
      H[(long long)(r0 + outRow(r, lane)) * kWidth + col] = fmaxf(z[r], 0.0f);
    }
    storeMask(z, M, r0, nt, lane, mask);
  }
}

// Layer: Xm = mean of Hp over the graph neighbours, H = Hp + relu([Hp | Xm] W
// + b) and its ReLU bits; 64 rows a block, a wavefront per 32x32 output tile.
// LAST also decodes: y[i] = sum_k bf16(H[i][k]) bf16(w[k]) + bout + X[i][skip]
// (the network learns a correction to one input column, the previous pressure
// correction, so an untrained network already predicts that column).
template <bool LAST>
__global__ void __launch_bounds__(256) k_layer(int M, int n, const float* __restrict__ Hp, const int* __restrict__ off,
                                               const int* __restrict__ nbr, const bf16* __restrict__ Wt,
                                               const float* __restrict__ bias, float* __restrict__ Xm,
                                               float* __restrict__ H, unsigned* __restrict__ mask,
                                               const float* __restrict__ w, const float* __restrict__ bout,
                                               const float* __restrict__ X, int skip, float* __restrict__ y) {
  __shared__ __align__(16) short Xs[kTile][2 * kWidth + 8];
  __shared__ float ys[2][kTile];
  const int r0 = dev::xcdRowBlock() * kTile;
  if (r0 >= M) return;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nt = wv & 1, m0 = (wv >> 1) * 32;
  const int col = 32 * nt + (lane & 31), kh = (lane >> 5) * 8;
  s16x8 wf[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    wf[k] = *reinterpret_cast<const s16x8*>(reinterpret_cast<const short*>(Wt) + col * 2 * kWidth + 16 * k + kh);
  {
    const int c = 4 * (threadIdx.x & 15), q = 4 * (threadIdx.x >> 4);
    float4 h[4], g[4];
    int deg[4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
      h[p] = r0 + q + p < n ? ld4(Hp + (long long)(r0 + q + p) * kWidth + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    gather4(n, r0 + q, c, Hp, off, nbr, g, deg);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (deg[p] > 0) {
        const float d = (float)deg[p];
        g[p] = make_float4(g[p].x / d, g[p].y / d, g[p].z / d, g[p].w / d);
      }
      if (r0 + q + p < n) *reinterpret_cast<float4*>(Xm + (long long)(r0 + q + p) * kWidth + c) = g[p];
      *reinterpret_cast<s16x4*>(&Xs[q + p][c]) = bf4(h[p].x, h[p].y, h[p].z, h[p].w);
      *reinterpret_cast<s16x4*>(&Xs[q + p][kWidth + c]) = bf4(g[p].x, g[p].y, g[p].z, g[p].w);
    }
  }
  __syncthreads();
  f32x16 z = zero16();
#pragma unroll
  for (int k = 0; k < 8; ++k)
    z = mfma(*reinterpret_cast<const s16x8*>(&Xs[m0 + (lane & 31)][16 * k + kh]), wf[k], z);
  const float bb = bias[col], wc = LAST ? bfRound(w[col]) : 0.0f;
  float keep = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = r0 + m0 + outRow(r, lane);
    z[r] += bb;
    float h = 0.0f;
    if (row < M) {
      const long long o = (long long)row * kWidth + col;
      h = Hp[o] + fmaxf(z[r], 0.0f);
      H[o] = h;
    }
    if (LAST) {
      const float s = dev::laneSum<32>(bfRound(h) * wc);
      if ((lane & 31) == r) keep = s;
    }
  }
  storeMask(z, M, r0 + m0, nt, lane, mask);
  if (LAST) {
    if ((lane & 31) < 16) ys[nt][m0 + outRow(lane & 15, lane)] = keep;
    __syncthreads();
    const int i = r0 + threadIdx.x;
    if (threadIdx.x < kTile && i < M)
      y[i] = ys[0][threadIdx.x] + ys[1][threadIdx.x] + bout[0] + X[(long long)i * 16 + skip];
  }
}

// Backward of one layer, 64 rows a step, every block over its own run of
// steps; its share of the gradients stays in registers until the end and goes
// to `part` (one parameter-shaped vector per block, summed by k_grad_sum).
//   dH: kTop:  dy bf16(w), dy = 2 (y - t) / n; also the decoder's gradient
//              and the loss
//       else:  D1 + sum over the neighbours of D2 (the adjacency is symmetric)
//   dZ = dH where the ReLU bit is set;  dW = [Hp | Xm]^T dZ, db = sum dZ
//   dX = dZ W^T:  D1o = dH + dX[:, :64],  D2o = dX[:, 64:] / deg
// kBottom is the encoder: [Hp | Xm] is the input X (M x 16) and dX not needed.
// Two blocks a CU need the registers held to half: 42.7 -> 26.9 us a layer.
// D1o may be D1 (a row is read by the block that writes it), D2o not D2.
enum { kTop, kMiddle, kBottom };
template <int MODE>
__global__ void __launch_bounds__(256, 2) k_layer_back(
    int M, int n, const float* __restrict__ y, const float* __restrict__ t, const float* __restrict__ Htop,
    const float* __restrict__ w, const float* D1, const float* __restrict__ D2, const int* __restrict__ off,
    const int* __restrict__ nbr, const unsigned* __restrict__ mask, const float* __restrict__ Hp,
    const float* __restrict__ Xm, const bf16* __restrict__ W, float* D1o, float* __restrict__ D2o,
    float* __restrict__ part, int np, int oW, int ob, int ow) {
  constexpr int kFeat = MODE == kBottom ? 16 : 2 * kWidth;
  constexpr int kLd = kTile + 4;  // LDS stride of the transposed tiles: 8-byte aligned, writes two lanes a bank
  __shared__ __align__(16) short Zt[kWidth][kLd];
  __shared__ __align__(16) short Xt[MODE == kBottom ? 32 : kFeat][kLd];
  __shared__ __align__(16) short Zs[MODE == kBottom ? 1 : kTile][kWidth + 8];
  __shared__ __align__(16) float dHs[MODE == kBottom ? 32 : kTile][kWidth + 4];
  __shared__ float degs[kTile];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, kh = (lane >> 5) * 8;
  const int sub = threadIdx.x & 15, slot = threadIdx.x >> 4, c = 4 * sub, q = 4 * slot;
  const int block = dev::xcdRowBlock(), tiles = (M + kTile - 1) / kTile;
  const int tEnd = (int)((long long)(block + 1) * tiles / gridDim.x);
  s16x8 wf[4];
  if (MODE != kBottom) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      wf[k] = *reinterpret_cast<const s16x8*>(reinterpret_cast<const short*>(W) +
                                              (32 * wv + (lane & 31)) * kWidth + 16 * k + kh);
  } else {
    for (int i = threadIdx.x; i < 16 * kLd; i += 256) Xt[16 + i / kLd][i % kLd] = 0;
  }
  f32x16 dW[2] = {zero16(), zero16()};
  float4 db = make_float4(0.0f, 0.0f, 0.0f, 0.0f), dw = db;
  float dbout = 0.0f, loss = 0.0f;
  for (int tile = (int)((long long)block * tiles / gridDim.x); tile < tEnd; ++tile) {
    const int r0 = tile * kTile;
    float4 dh[4], x0[4], x1[4];
    int deg[4];
    unsigned bits[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int row = r0 + q + p;
      const bool in = row < n;
      const float4 none = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      bits[p] = in ? mask[2 * row + (sub >> 3)] >> (c & 31) : 0u;
      if (MODE != kBottom) {
        x0[p] = in ? ld4(Hp + (long long)row * kWidth + c) : none;
        x1[p] = in ? ld4(Xm + (long long)row * kWidth + c) : none;
      } else {
        x0[p] = in && sub < 4 ? ld4(Hp + (long long)row * 16 + c) : none;
      }
      if (MODE == kTop) {
        deg[p] = in ? off[row + 1] - off[row] : 0;
        float g = 0.0f;
        if (in) {
          const float d = y[row] - t[row];
          g = 2.0f * d / (float)n;
          if (sub == 0) {
            loss += d * d;
            dbout += g;
          }
          const float4 h = ld4(Htop + (long long)row * kWidth + c);
          add4(dw, make_float4(bfRound(h.x) * g, bfRound(h.y) * g, bfRound(h.z) * g, bfRound(h.w) * g));
        }
        dh[p] = make_float4(g * bfRound(w[c]), g * bfRound(w[c + 1]), g * bfRound(w[c + 2]), g * bfRound(w[c + 3]));
      } else {
        dh[p] = in ? ld4(D1 + (long long)row * kWidth + c) : none;
      }
    }
    if (MODE != kTop) {
      float4 g[4];
      gather4(n, r0 + q, c, D2, off, nbr, g, deg);
#pragma unroll
      for (int p = 0; p < 4; ++p) add4(dh[p], g[p]);
    }
    float4 dz[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      dz[p] = make_float4(bits[p] & 1u ? dh[p].x : 0.0f, bits[p] & 2u ? dh[p].y : 0.0f, bits[p] & 4u ? dh[p].z : 0.0f,
                          bits[p] & 8u ? dh[p].w : 0.0f);
      add4(db, dz[p]);
      if (MODE != kBottom) {
        *reinterpret_cast<s16x4*>(&Zs[q + p][c]) = bf4(dz[p].x, dz[p].y, dz[p].z, dz[p].w);
        *reinterpret_cast<float4*>(&dHs[q + p][c]) = dh[p];
        if (sub == 0) degs[q + p] = (float)deg[p];
      }
    }
    auto put = [&](short (*T)[kLd], int col, const float4 (&v)[4]) {
      *reinterpret_cast<s16x4*>(&T[col][q]) = bf4(v[0].x, v[1].x, v[2].x, v[3].x);
      *reinterpret_cast<s16x4*>(&T[col + 1][q]) = bf4(v[0].y, v[1].y, v[2].y, v[3].y);
      *reinterpret_cast<s16x4*>(&T[col + 2][q]) = bf4(v[0].z, v[1].z, v[2].z, v[3].z);
      *reinterpret_cast<s16x4*>(&T[col + 3][q]) = bf4(v[0].w, v[1].w, v[2].w, v[3].w);
    };
    put(Zt, c, dz);
    if (MODE != kBottom || sub < 4) put(Xt, c, x0);
    if (MODE != kBottom) put(Xt, kWidth + c, x1);
    __syncthreads();
    if (MODE != kBottom || wv < 2) {
#pragma unroll
      for (int k = 0; k < kTile / 16; ++k) {
        const int xr = MODE == kBottom ? 0 : 32 * wv;
        const s16x8 xf = ld8(&Xt[xr + (lane & 31)][16 * k + kh]);
#pragma unroll
        for (int nt = 0; nt < (MODE == kBottom ? 1 : 2); ++nt)
          dW[nt] = mfma(xf, ld8(&Zt[32 * (MODE == kBottom ? wv : nt) + (lane & 31)][16 * k + kh]), dW[nt]);
      }
    }
    if (MODE != kBottom) {
      const int col = 32 * (wv & 1) + (lane & 31);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        f32x16 dX = zero16();
#pragma unroll
        for (int k = 0; k < 4; ++k)
          dX = mfma(*reinterpret_cast<const s16x8*>(&Zs[32 * mt + (lane & 31)][16 * k + kh]), wf[k], dX);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = 32 * mt + outRow(r, lane);
          if (r0 + m >= n) continue;
          const long long o = (long long)(r0 + m) * kWidth + col;
          if (wv < 2) D1o[o] = dHs[m][col] + dX[r];
          else D2o[o] = dX[r] / degs[m];
        }
      }
    }
    __syncthreads();
  }
  float* P = part + (long long)block * (np + 1);
  if (MODE != kBottom || wv < 2) {
#pragma unroll
    for (int nt = 0; nt < (MODE == kBottom ? 1 : 2); ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k = (MODE == kBottom ? 0 : 32 * wv) + outRow(r, lane);
        const int col = 32 * (MODE == kBottom ? wv : nt) + (lane & 31);
        if (k < kFeat) P[oW + k * kWidth + col] = dW[nt][r];
      }
  }
  // column sums over the 16 row slots
  *reinterpret_cast<float4*>(&dHs[slot][c]) = db;
  if (MODE == kTop) *reinterpret_cast<float4*>(&dHs[16 + slot][c]) = dw;
  if (MODE == kTop && sub == 0) {
    degs[slot] = dbout;
    degs[16 + slot] = loss;
  }
  __syncthreads();
  const int col = threadIdx.x & 63;
  if (wv == 0 || (MODE == kTop && wv == 1)) {
    float s = 0.0f;
    for (int i = 0; i < 16; ++i) s += dHs[16 * wv + i][col];
    P[(wv == 0 ? ob : ow) + col] = s;
  }
  if (MODE == kTop && wv == 2 && lane < 2) {
    float s = 0.0f;
    for (int i = 0; i < 16; ++i) s += degs[16 * lane + i];
    P[lane == 0 ? ow + kWidth : np] = s;  // the output bias follows w
  }
}

// grad[i] = sum over the blocks of part[block][i], and the loss behind it:
// four wavefronts share 64 columns' rows (fixed order).  15 us for 512 blocks'
// 70 MB, 4.6 TB/s.
static __global__ void __launch_bounds__(256) k_grad_sum(int blocks, int np, const float* __restrict__ part,
                                                         float* __restrict__ grad, float* __restrict__ loss) {
  __shared__ float sh[4][64];
  const int i = blockIdx.x * 64 + (threadIdx.x & 63), g = threadIdx.x >> 6;
  float s = 0.0f;
  if (i <= np) {
#pragma unroll 8
    for (int b = g; b < blocks; b += 4) s += part[(long long)b * (np + 1) + i];
  }
  sh[g][threadIdx.x & 63] = s;
  __syncthreads();
  if (g != 0 || i > np) return;
  s = (sh[0][threadIdx.x] + sh[1][threadIdx.x]) + (sh[2][threadIdx.x] + sh[3][threadIdx.x]);
  if (i < np) grad[i] = s;
  else loss[0] = s;
}

__device__ __forceinline__ float blockSum(float v) {  // 256 threads; thread 0 has the sum
  __shared__ float sh[4];
  v = dev::laneSum<64>(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// part[block] = sum of (y - t)^2 over the block's rows, and a sum of a vector.
static __global__ void __launch_bounds__(256) k_sq_error(int n, const float* __restrict__ y,
                                                         const float* __restrict__ t, float* __restrict__ part) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const float d = i < n ? y[i] - t[i] : 0.0f;
  const float s = blockSum(d * d);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
static __global__ void __launch_bounds__(256) k_sum(int n, const float* __restrict__ x, float* __restrict__ out) {
  float s = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) s += x[i];
  s = blockSum(s);
  if (threadIdx.x == 0) out[0] = s;
}

// BF16 copies of the GEMM weights for parameter i (W, K x 64, and its
// transpose 64 x K); the parameter vector holds W0 (16 x 64), b0, then W
// (128 x 64) and b of each layer, then w and its bias.
__device__ __forceinline__ void copyWeight(int i, int layers, float p, bf16* __restrict__ W16, bf16* __restrict__ Wt16) {
  constexpr int kEnc = 16 * kWidth, kW = 2 * kWidth * kWidth;
  int e = i, K = 16, base = 0;
  if (i >= kEnc) {
    const int j = i - kEnc - kWidth, l = j / (kW + kWidth);
    if (j < 0 || l >= layers) return;
    e = j % (kW + kWidth);
    if (e >= kW) return;
    K = 2 * kWidth;
    base = kEnc + l * kW;
  }
  const bf16 b = floatToBf16(p);
  W16[base + e] = b;
  Wt16[base + (e % kWidth) * K + e / kWidth] = b;
}
static __global__ void k_weight_bf16(int np, int layers, const float* __restrict__ p, bf16* __restrict__ W16,
                                     bf16* __restrict__ Wt16) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < np) copyWeight(i, layers, p[i], W16, Wt16);
}

// Adam step on the FP32 master parameters (Kingma & Ba 2015, bias-corrected)
// and the BF16 copies of the new weights.
static __global__ void k_adam(int np, int layers, float* __restrict__ p, const float* __restrict__ g,
                              float* __restrict__ m, float* __restrict__ v, float lr, float b1, float b2, float eps,
                              float c1, float c2, bf16* __restrict__ W16, bf16* __restrict__ Wt16) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  copyWeight(i, layers, pi, W16, Wt16);
}

}  // namespace gnn
}  // namespace nodals
