// ads_mlp.h -- the flux-correction network's device parameters and kernel
// launchers (ads_mlp.hip). Internal header.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace f3d {

// flat FP32 parameter vector: W1[32][64], b1[64], W2[64][64], b2[64], w3[64], b3
constexpr int MLP_NIN = 32, MLP_NH = 64;
constexpr int MLP_OFF_W1 = 0;
constexpr int MLP_OFF_B1 = MLP_OFF_W1 + 32 * 64;
constexpr int MLP_OFF_W2 = MLP_OFF_B1 + 64;
constexpr int MLP_OFF_B2 = MLP_OFF_W2 + 64 * 64;
constexpr int MLP_OFF_W3 = MLP_OFF_B2 + 64;
constexpr int MLP_OFF_B3 = MLP_OFF_W3 + 64;
constexpr int MLP_NPARAM = MLP_OFF_B3 + 1;  // 6337

// BF16 MFMA operands of the current weights (see k_pack)
struct PackedWeights {
  __bf16 w1t[4][64][8];
  __bf16 w2t[4][2][64][8];
  __bf16 w2[4][2][64][8];
  float b1[64], b2[64], w3[64];
  float b3;
  float pad[63];
};

hipError_t mlp_pack(const float *params, PackedWeights *w, hipStream_t st);
// y[r] = net(x[r]) for r < n; x: n rows of 32 bf16 (bit patterns)
hipError_t mlp_forward(const PackedWeights *w, const uint16_t *x, long n, float *y, hipStream_t st);
// Rows of a batch: position r is row hash(seed, step, r) mod count, or r
// itself when count is 0.
struct BatchRows {
  long count;
  unsigned long long inv;  // floor((2^64 - 1) / count)
  unsigned long long seed;
  int step;
};
// One Adam update: master parameters, moments, the operands of the next pass
// and the batch's sum of squared errors.
struct AdamUpdate {
  float *p, *m, *v;
  PackedWeights *w;
  float *loss;
  int step;
  float lr, beta1, beta2, eps;
};
// floats of scratch of a batch of n rows: rows of kGradRow floats, one per
// wave of 32 batch rows and one per slot of their sum
constexpr int kGradRow = (MLP_NPARAM + 1 + 3) / 4 * 4;
size_t mlp_grad_scratch(long n);
// grad[0..NPARAM) = d/dparams of scale * sum_r (net(x[r]) - t[r])^2 over rows
// 0..n, grad[NPARAM] = sum of squared errors. part: mlp_grad_scratch(n) floats.
hipError_t mlp_grad(const PackedWeights *w, const uint16_t *x, const float *t, long n, float scale, float *part,
                    float *grad, hipStream_t st);
// the same gradient over a batch of n rows, and one Adam update with it
hipError_t mlp_update(const uint16_t *x, const float *t, const BatchRows &rows, long n, float scale, float *part,
                      const AdamUpdate &u, hipStream_t st);

}  // namespace f3d
