// sublayer_tile.hpp -- host-side launch interface of sublayer_tile.hip's products on 64 x 64 tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mla {

// Y_i[r][n] = sum_k X[r][k] W_i, i < n <= 3; bf16, X and Y_i [R][C], W_i [C][C], C a multiple of 64.
struct TileRows {
  const uint16_t* x;
  const uint16_t* w[3];
  uint16_t* y[3];
  int n, R, C;
  // the phase encoder's additions to a product of one weight, all optional:
  const uint16_t* add;  // sum[r][n] = bf16(add + Y) (residualAdd)
  uint16_t* sum;
  const uint16_t* O;  // heads of 64 features: Dv[b][h][t] = computeD of Y and O, H heads, T rows a batch
  float* Dv;
  int T, H;
  float *zero0, *zero1;  // C floats each set to 0
};
// wt: W_i indexed [n][k], else [k][n].
hipError_t launch_tile_rows(const TileRows& a, bool wt, hipStream_t s);

// The gradient products that a call asks for: the weights w0 .. w1 - 1 (from 0, or one alone) of (0 dQw, 1 dKw, 2 dVw, 3
// dProjw), each dW[w] = x[w]^T . g[w] over R rows (a multiple of 64), dQw with the fp32 dQ for g[0];
// and computeGradDx (dQ, dK = g[1], dV = g[2]) where dX is set. Destinations are added into, or
// written as 0 + the sum: dX and dQw fp32, the other weights bf16.
struct TileGrad {
  float* dX;
  const float* dQ;
  const uint16_t* W[3];  // q_w, k_w, v_w (dX only)
  const uint16_t* x[4];
  const uint16_t* g[4];
  void* dW[4];
  int w0, w1, R, C;
  // set by launch_tile_grad: row chunks of dQw and of each other weight (1: the destination is
  // written directly; more: fp32 partials [nq + others * nkv][C][C], added by a second kernel)
  int nq, nkv;
  float* part;
};
// Floats of `partial` that launch_tile_grad needs for these products (0: none).
size_t tile_grad_partial_floats(int R, int C, int w0, int w1, bool dx);
// The most it needs for any multiple of 64 rows up to R.
size_t tile_grad_partial_bound(int R, int C, int w0, int w1, bool dx);
hipError_t launch_tile_grad(TileGrad a, float* partial, bool accumulate, hipStream_t s);

}  // namespace mla
