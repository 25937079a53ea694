#pragma once

#include <hip/hip_runtime.h>

#include <math.h>

// log(sigmoid(z)) without overflow: min(z, 0) - log(1 + exp(-|z|))
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
