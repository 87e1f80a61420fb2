// What the recurrences with a decay per key channel do to their raw inputs.
#pragma once
#include "common.h"

enum { DECAY_PER_HEAD = 0, DECAY_SIGMOID_ROOT = 1, DECAY_EXP_EXP = 2, DECAY_READY = 3 };   // READY: z holds the decays themselves

__device__ __forceinline__ float exact_silu(float z) { return z / (1.f + expf(-z)); }

// The decay of a raw value.  sigmoid(z)^(1/tau) = exp(-softplus(-z) / tau), with softplus(x) = max(x, 0) + log1p(e^-|x|).
__device__ __forceinline__ float decay_of(float z, int kind, float inv_tau) {
  if (kind == DECAY_SIGMOID_ROOT) {
    const float x = -z;
    const float sp = fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
    return expf(-sp * inv_tau);
  }
  return expf(-expf(z));
}
