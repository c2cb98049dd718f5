// One element of the diagonal Gaussian draw, shared by the sampling launch of
// the rollout step and the paired towers' step kernel: the formulas at the top
// of sample.hip.
#pragma once
#include "common.h"
#include "threefry.h"

#include <math.h>

namespace ppo {
namespace gauss {

constexpr float HALF_LOG_2PI = 0.91893853320467274f;

__device__ __forceinline__ float softplus_acc(float x) {
  // jax.nn.softplus = logaddexp(x, 0)
  return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
}

__device__ __forceinline__ float erfinv_giles(float x) {
  float w = -log1pf(-(x * x));
  float p;
  if (w < 5.0f) {
    w = w - 2.5f;
    p = 2.81022636e-08f;
    p = 3.43273939e-07f + p * w;
    p = -3.5233877e-06f + p * w;
    p = -4.39150654e-06f + p * w;
    p = 0.00021858087f + p * w;
    p = -0.00125372503f + p * w;
    p = -0.00417768164f + p * w;
    p = 0.246640727f + p * w;
    p = 1.50140941f + p * w;
  } else {
    w = sqrtf(w) - 3.0f;
    p = -0.000200214257f;
    p = 0.000100950558f + p * w;
    p = 0.00134934322f + p * w;
    p = -0.00367342844f + p * w;
    p = 0.00573950773f + p * w;
    p = -0.0076224613f + p * w;
    p = 0.00943887047f + p * w;
    p = 1.00167406f + p * w;
    p = 2.83297682f + p * w;
  }
  return fabsf(x) == 1.0f ? x * INFINITY : p * x;
}

// The action of mean and raw scale at word i of the key's stream; adds the
// element's terms of the log-probability: its density to lpx, log sigma to logdet.
__device__ __forceinline__ float draw(float mean, float raw, uint32_t k0, uint32_t k1, uint64_t i, float temperature,
                                      float& lpx, float& logdet) {
  const float lo = -0.99999994f;  // nextafter(-1, 0)
  const float span = 1.0f - lo;   // maxval - minval, rounded to float32
  const float f = ppo::unit_float(ppo::random_word(k0, k1, i));
  const float u = fmaxf(lo, f * span + lo);
  const float eps = 1.41421356237309515f * erfinv_giles(u);
  const float sig = temperature * (softplus_acc(raw) + 1e-3f);
  lpx += -0.5f * (eps * eps) - HALF_LOG_2PI;
  logdet += logf(sig);
  return sig * eps + mean;
}

}  // namespace gauss
}  // namespace ppo
