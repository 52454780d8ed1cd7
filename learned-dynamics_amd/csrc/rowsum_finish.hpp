// Finishing pass of the GEMMs that sum the rows of each segment in their epilogue: every block of 32 rows left
// two partial rows (slot A: the run that starts at the block's first row, slot B: a later run that ends at its
// last row); runs strictly inside a block were written to `out` directly.
#pragma once
#include "common.hpp"

namespace mg {
namespace {

// out[s] = scale * (slots of the blocks the rows of segment s lie in, in block order); segments strictly inside
// one block were written by the kernel above, empty segments get zero.  One thread per four columns.
__global__ void __launch_bounds__(256)
rowsum_finish_kernel(const int* __restrict__ row_ptr, long n_out, long n_blocks, int O, const float* __restrict__ slots,
                     float scale, float* __restrict__ out) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int quads = O / 4;
    if (idx >= n_out * quads) return;
    const long s_id = idx / quads;
    const int x = (int)(idx - s_id * quads) * 4;
    const long lo = row_ptr[s_id], hi = row_ptr[s_id + 1];
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (hi > lo) {
        const long b_lo = lo / 32, b_hi = (hi - 1) / 32;
        if (b_lo == b_hi && lo > 32 * b_lo && hi - 1 < 32 * b_lo + 31) return;   // written directly
        for (long b = b_lo; b <= b_hi; b++) {
            const float* slot = 32 * b >= lo ? slots + b * O : slots + (n_blocks + b) * O;
            const float4 t = *reinterpret_cast<const float4*>(slot + x);
            s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
        }
    }
    *reinterpret_cast<float4*>(out + s_id * O + x) = make_float4(scale * s.x, scale * s.y, scale * s.z, scale * s.w);
}

// The same into rows of a wider matrix (stride floats apart) whose bounds the linear behind it takes: row_max[s max_stride + p] is the
// largest magnitude among columns 256 p .. 256 p + 255 of the sum, a wave to each (O a multiple of 256).  base (n_out, O): the number of
// rows of s times bias is added to it, or written with fresh != 0: the bias of a linear whose rows were summed before it.
__global__ void __launch_bounds__(256)
rowsum_finish_into_kernel(const int* __restrict__ row_ptr, long n_out, long n_blocks, int O, const float* __restrict__ slots,
                          float scale, float* __restrict__ out, long stride, float* __restrict__ row_max, int max_stride,
                          const float* __restrict__ bias, float* __restrict__ base, int fresh) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int quads = O / 4;
    if (idx >= n_out * quads) return;                              // (whole waves)
    const long s_id = idx / quads;
    const int x = (int)(idx - s_id * quads) * 4;
    const long lo = row_ptr[s_id], hi = row_ptr[s_id + 1];
    float* const to = out + s_id * stride + x;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    const long b_lo = lo / 32, b_hi = (hi - 1) / 32;
    if (hi > lo && b_lo == b_hi && lo > 32 * b_lo && hi - 1 < 32 * b_lo + 31) {
        s = *reinterpret_cast<const float4*>(to);                  // written directly
    } else {
        if (hi > lo)
            for (long b = b_lo; b <= b_hi; b++) {
                const float* slot = 32 * b >= lo ? slots + b * O : slots + (n_blocks + b) * O;
                const float4 t = *reinterpret_cast<const float4*>(slot + x);
                s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
            }
        s = make_float4(scale * s.x, scale * s.y, scale * s.z, scale * s.w);
        *reinterpret_cast<float4*>(to) = s;
    }
    if (base) {
        const float count = (float)(hi - lo);
        const float4 c = *reinterpret_cast<const float4*>(bias + x);
        float4* const at = reinterpret_cast<float4*>(base + s_id * O + x);
        const float4 was = fresh ? make_float4(0.f, 0.f, 0.f, 0.f) : *at;
        *at = make_float4(was.x + count * c.x, was.y + count * c.y, was.z + count * c.z, was.w + count * c.w);
    }
    float mx = fmaxf(fmaxf(fabsf(s.x), fabsf(s.y)), fmaxf(fabsf(s.z), fabsf(s.w)));
    for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
    if ((threadIdx.x & 63) == 0) row_max[s_id * max_stride + x / 256] = mx;
}

}  // namespace
}  // namespace mg
