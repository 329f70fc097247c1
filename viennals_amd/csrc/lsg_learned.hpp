// Launchers of the learned-weno5 kernels (lsg_learned.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace lsg {

constexpr int MLP_PSTRIDE = 1348;  // partial-gradient row: 1347 parameters + squared-residual sum

// Workgroups (= partial rows) of a gradient over n >= 1 samples, at most `most`.
int mlpGradRows(uint32_t n, int most);
// Gradient of the mean squared loss over samples X[n][8], T[n] at the fp32
// parameters P: per-workgroup partials (rows x MLP_PSTRIDE floats, rows >= 1)
// summed into grad[MLP_PSTRIDE] (grad[1347] = sum of squared residuals).  With
// M and V, one Adam step (beta1 0.9, beta2 0.999, eps 1e-8) on P at step >= 1.
void launchMlpGrad(hipStream_t s, const float *X, const float *T, uint32_t n, float *P, float *partials, int rows,
                   float *grad, float *M = nullptr, float *V = nullptr, int step = 0, float lr = 0.f);
// Learned weno5 on n stencils (x[n*7]) with bf16 parameters.
void launchWenoLearned(hipStream_t s, uint32_t n, const double *x, double dx, int plus, const uint16_t *prm,
                       double *out);

}  // namespace lsg
