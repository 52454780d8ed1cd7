// Split-fp16 arithmetic shared by the kernels that run fp32 GEMMs on the fp16 matrix cores:
// a value v scaled by a power of two s is carried as hi + lo with hi = fp16(v s), lo = fp16(v s - hi),
// and a product takes three MFMAs (lo hi, hi lo, hi hi) accumulated in fp32.
#pragma once
#include <hip/hip_runtime.h>

namespace mg {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));


// power of two s with amax * s in [2^14, 2^15); *inv = 1/s.  amax >= 0; zero, tiny, inf and nan give
// a finite in-range scale.  Rows that beyond_split tells apart are not for the fp16 pieces
__device__ __forceinline__ float pow2_scale(float amax, float* inv) {
    int e = (int)(__float_as_uint(amax) >> 23) & 0xff;
    int se = 268 - e;                   // 127 + 14 - (e - 127)
    if (e == 255) se = 127;
    se = se < 1 ? 1 : (se > 253 ? 253 : se);
    *inv = __uint_as_float((unsigned)(254 - se) << 23);
    return __uint_as_float((unsigned)se << 23);
}

// A row of x with an infinity (its low piece would be inf - inf), or so large that the scaled sum times 1 / s could overflow
// before the weight's scale brings it back: the linear kernels take such a row in fp32 (row_in_fp32).  A bound that
// has overflowed by itself, as one carried through several layers may, only costs time.
__device__ __forceinline__ bool beyond_split(float amax) { return !(amax < 0x1p96f); }
// The inverse scale of a weight's row that holds an infinity or NaN: a NaN whose low bits are the exponent of the inverse scale
// of the row's finite entries.  Every kernel that multiplies by it gives NaN; the linear kernels take the column in fp32.
__device__ __forceinline__ float mark_weight(float inv) { return __uint_as_float(0x7fc00000u | (__float_as_uint(inv) >> 23)); }
__device__ __forceinline__ float unmark_weight(float iw) { return iw == iw ? iw : __uint_as_float((__float_as_uint(iw) & 0xffu) << 23); }

struct HalfSplit4 {
    halfx4 hi, lo;
};

__device__ __forceinline__ HalfSplit4 split(float4 v, float s) {
    HalfSplit4 r;
    const float in[4] = {v.x * s, v.y * s, v.z * s, v.w * s};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const _Float16 h = (_Float16)in[k];
        r.hi[k] = h;
        r.lo[k] = (_Float16)(in[k] - (float)h);
    }
    return r;
}

// Two values at a time: three instructions each (the low piece by one fused multiply-add of mixed widths; v s is exact, s a power of
// two).
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split_pair(float v0, float v1, float s0, float s1, halfx2& hi, halfx2& lo) {
    hi = __builtin_convertvector((floatx2{v0 * s0, v1 * s1}), halfx2);
    lo = __builtin_convertvector((floatx2{__builtin_fmaf(v0, s0, -(float)hi[0]), __builtin_fmaf(v1, s1, -(float)hi[1])}), halfx2);
}

// Between a wave's writes to its own LDS and reads of them by other lanes, or those reads and the next writes: LDS keeps the order of
// one wave, this keeps the compiler to it (the barrier by itself is nothing that memory instructions may not cross)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

constexpr int kCK = 32;                     // k per chunk (two MFMA steps)

// Packed planes of a weight (O, I): in the order the matrix cores read them.  A block of 32 output rows x one chunk of 32
// k is 1024 halves: step s of the chunk (512 halves), lane = row % 32 + 32 g of the fragment, its 8 consecutive
// k = 32 c + 16 g + 8 s .. + 8.  Blocks of rows outermost, then chunks.  A wave's fragment load is one contiguous
// kilobyte, from memory or from LDS (no padding, no bank conflicts); in row-major planes the 64 lanes of such a load sat in
// 32 rows and the vector-memory front end took them line by line.
__host__ __device__ __forceinline__ long packed_index(long o, int k, int I) {
    return ((o >> 5) * (I >> 5) + (k >> 5)) * 1024L + ((k >> 3) & 1) * 512 + ((((k >> 4) & 1) << 5) + (o & 31)) * 8 + (k & 7);
}
// the i-th 16-byte piece (i = 128 block + 64 s + lane) of chunk 0 of a tile of output rows that starts at n0 (a multiple
// of 32); chunk k0 / 32 of the same piece is kPackedChunk * (k0 / 32) = 32 k0 halves further on
__device__ __forceinline__ long packed_piece(int n0, int i, int I) {
    return ((long)((n0 >> 5) + (i >> 7)) * (I >> 5)) * 1024L + (i & 127) * 8;
}

// x . w in fp32, k in order, with weight row n put together from its pieces (a weight below 2^-39 of its row's largest is zero
// there) and iw its inverse scale: what the linear kernels give for the rows and columns marked above.
__device__ inline float row_in_fp32(const float* x, const _Float16* planes, long plane_elems, long n, int I, float iw) {
    const float inv = unmark_weight(iw);
    float sum = 0.f;
#pragma unroll 1
    for (int k = 0; k < I; k += 8) {
        const long at = packed_index(n, k, I);
        const halfx8 hi = *reinterpret_cast<const halfx8*>(planes + at), lo = *reinterpret_cast<const halfx8*>(planes + plane_elems + at);
        const float4 x0 = *reinterpret_cast<const float4*>(x + k), x1 = *reinterpret_cast<const float4*>(x + k + 4);
        const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float h = (float)hi[j];
            sum = fmaf(v[j], (fabsf(h) < __builtin_inff() ? h + (float)lo[j] : h) * inv, sum);
        }
    }
    return sum;
}

// Issue order of one chunk of a tile that is 256 output columns wide (16 fragment pairs, 48 matrix instructions): four
// fragments are read ahead, then three matrix instructions alternate with the two reads of the pair after next.  Left
// alone the compiler reads a pair, waits for it and multiplies, and the matrix cores idle for the latency of the LDS:
// 0.90 -> 0.925 PFLOP/s (counting the three fp16 products) at 1.05 M rows x 512 x 512.  Only the order of issue changes.
// The narrower tiles have more waves per SIMD to hide the reads behind and are left to the compiler.
template <int NI>
__device__ __forceinline__ void order_chunk() {
    if constexpr (NI == 8) {
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);       // LDS reads
#pragma unroll
        for (int k = 0; k < 14; k++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);   // matrix instructions
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
    }
}

}  // namespace mg
