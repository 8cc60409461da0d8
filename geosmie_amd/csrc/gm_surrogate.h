// Output transform of the LUT surrogate, shared by its own kernel
// (gm_surrogate.hip, which states the formulas) and the network kernel that
// writes table rows directly (gm_mlp.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace gm {

constexpr int kSurrIn = 6;

// ln B of one query; FP32 throughout, log domain.
__device__ __forceinline__ float rayleigh_log_b(const float* __restrict__ qi, float mw_re) {
  const float dry = 1.0f - qi[5];
  const float lx = qi[0] - logf(qi[4]) + 1.8378770664093453f;   // ln x_eff
  const float ls = logf(qi[1]);
  const float mr = mw_re + (qi[2] - mw_re) * dry, mi = expf(qi[3]) * dry;
  const float a = mr * mr - mi * mi, b = 2.0f * mr * mi;          // m^2 = a + i b
  const float den = (a + 2.0f) * (a + 2.0f) + b * b;
  const float k2 = ((a - 1.0f) * (a - 1.0f) + b * b) / den;      // |K|^2
  const float ln_sca = 0.98082925301172f + logf(k2) + 4.0f * lx + 6.0f * ls * ls;   // ln 8/3
  const float ln_abs = 1.38629436111989f + logf(3.0f * b / den) + lx;               // ln 4
  const float hi = fmaxf(ln_sca, ln_abs), lo = fminf(ln_sca, ln_abs);
  const float lq = hi + log1pf(expf(lo - hi));                   // ln Q_R
  const float u = lq - 0.69314718055995f;                        // ln(Q_R / 2)
  return lq - (fmaxf(u, 0.0f) + log1pf(expf(-fabsf(u))));        // ln Q_R - ln(1 + Q_R/2)
}

// Table value j from the de-standardised output t; lnb = ln B (0: no baseline).
__device__ __forceinline__ float surr_row_value(int j, float t, float lnb) {
  if (j == 0) return expf(t + lnb);
  if (j == 1) return fminf(expf(t), 1.0f);
  if (j == 2) return expf(t);
  return (float)(2 * (j - 3) + 1) * t;
}

}  // namespace gm
