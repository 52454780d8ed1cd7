// What the kernels that hold a slice of the PaiNN filter grid in LDS share: the shape of a slice, and the sums over the 16
// edges that a wave takes at once.
#pragma once
#include "common.hpp"

namespace mg {

constexpr int kSliceChan = 16, kSliceCols = 4 * kSliceChan, kSliceRowF = kSliceCols + 4, kSliceMaxRows = 512;
constexpr int kSliceExtraRows = 3;

// Sum of 16 per-lane values over the 16 lanes that share (lane & 3), leaving value s of the 16 in the lane with
// (lane >> 2) == s: each step pairs the registers, exchanges the halves two lanes do not keep and adds, so the whole
// reduction is 15 additions instead of 16 x 4.  Lane halves (xor 32) and odd / even rows of 16 lanes (xor 16) are
// exchanged by the swap instructions, lanes 8 and 4 apart by LDS-crossbar swizzles.
__device__ __forceinline__ void swap_add32(float& a, const float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]) + __uint_as_float(r[1]);        // lanes 0..31: a over both halves; 32..63: b
}
__device__ __forceinline__ void swap_add16(float& a, const float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]) + __uint_as_float(r[1]);        // even rows of 16 lanes: a; odd rows: b
}
template <int XOR>
__device__ __forceinline__ void swizzle_add(float& a, const float b, bool upper) {
    const float keep = upper ? b : a, send = upper ? a : b;
    constexpr int pattern = (XOR << 10) | 0x1f;               // lane' = lane ^ XOR inside each group of 32
    a = keep + __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(send), pattern));
}
__device__ __forceinline__ float sum_over_slots(float (&acc)[16], int lane) {
    // value index = bit2 + 2 bit3 + 4 bit4 + 8 bit5 of the lane id
#pragma unroll
    for (int k = 0; k < 8; k++) swap_add32(acc[k], acc[k + 8]);          // registers 0..7: value k + 8 bit5
#pragma unroll
    for (int k = 0; k < 4; k++) swap_add16(acc[k], acc[k + 4]);          // registers 0..3: value k + 4 bit4 + 8 bit5
#pragma unroll
    for (int k = 0; k < 2; k++) swizzle_add<8>(acc[k], acc[k + 2], (lane & 8) != 0);
    swizzle_add<4>(acc[0], acc[1], (lane & 4) != 0);
    return acc[0];
}

}  // namespace mg
