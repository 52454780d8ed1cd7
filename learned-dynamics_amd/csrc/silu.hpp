// SiLU and its first two derivatives, for the kernels of the layers under differentiation.
#pragma once
#include <hip/hip_runtime.h>

namespace mg {

// s = sigma(z), p = s (1 - s)
struct Silu { float f, d1, d2; };
__device__ __forceinline__ Silu silu(float z) {
    const float s = 1.0f / (1.0f + expf(-z));
    const float p = s * (1.0f - s);
    return {z * s, s + z * p, p * (2.0f + z * (1.0f - 2.0f * s))};
}

}  // namespace mg
