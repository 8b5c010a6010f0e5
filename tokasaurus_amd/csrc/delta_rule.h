// What the kernels of the gated delta rule share.
#pragma once

#include "common.h"

#define DR_MAX_TAPS 16

__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + expf(-x)); }
