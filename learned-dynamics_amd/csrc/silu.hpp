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

// The same where the instructions count, and no less exact than with expf and a division: exp(-z) as 2^n 2^a with n + a
// = -z log2 e, a to its own last place, and 1 / (1 + e) by a reciprocal whose Newton step also takes what the sum
// 1 + e was rounded by.  rms error of f 3.9e-8 (expf and a division 4.0e-8).  (z is held to +-88: beyond, s is 0 or 1 to any precision that z s could show.)
__device__ __forceinline__ Silu silu_short(float z) {
    const float c = -fminf(fmaxf(z, -88.f), 88.f);
    const float n = __builtin_rintf(c * 1.44269502f), part = fmaf(c, 1.92596299e-8f, fmaf(c, 1.44269502f, -n));
    const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(part), (int)n), d = 1.0f + e;
    const float rest = fminf(e, 1.0f) - (d - fmaxf(e, 1.0f));
    const float r = __builtin_amdgcn_rcpf(d);
    return silu_of(z, fmaf(r, fmaf(-r, rest, fmaf(-r, d, 1.0f)), r));
}

}  // namespace mg
