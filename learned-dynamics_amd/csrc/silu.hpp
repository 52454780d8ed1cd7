// SiLU and its first two derivatives, for the kernels of the layers under differentiation.
#pragma once
#include <hip/hip_runtime.h>

namespace mg {

// s = sigma(z), p = s (1 - s)
struct Silu { float f, d1, d2; };
__device__ __forceinline__ Silu silu_of(float z, float s) {
    const float p = s * (1.0f - s);
    return {z * s, s + z * p, p * (2.0f + z * (1.0f - 2.0f * s))};
}
__device__ __forceinline__ Silu silu(float z) { return silu_of(z, 1.0f / (1.0f + expf(-z))); }

// The same where the instructions count: exp(-z) = 2^t (1 + ln 2 lo) with t + lo = -z log2 e to twice the precision, the reciprocal
// with one Newton step.  rms error of f 4.4e-8 (expf and a division: 4.1e-8) in a third of their instructions.  (z is held to +-88:
// beyond, s is 0 or 1 to any precision that z s could show.)
__device__ __forceinline__ Silu silu_short(float z) {
    const float c = -fminf(fmaxf(z, -88.f), 88.f);
    const float t = c * 1.44269502f, lo = fmaf(c, 1.92596299e-8f, fmaf(c, 1.44269502f, -t));
    const float e = __builtin_amdgcn_exp2f(t), d = 1.0f + fmaf(e, lo * 0.693147181f, e);
    const float r = __builtin_amdgcn_rcpf(d);
    return silu_of(z, fmaf(r, fmaf(-d, r, 1.0f), r));
}

}  // namespace mg
