// Rows of activations that stay in LDS as fp16 pieces (f16x2.hpp), in the order the matrix cores read them, and products with packed
// weights whose fragments come straight from memory.
#pragma once
#include "f16x2.hpp"

namespace mg {
namespace {

__device__ __forceinline__ int pad256(int o) { return (o + 255) / 256 * 256; }
__device__ __forceinline__ bool has_marks(const float* inv, int O, int lane) {
    const int* marks = reinterpret_cast<const int*>(inv + pad256(O));
    return __any(lane < (O + 31) / 32 && marks[lane < (O + 31) / 32 ? lane : 0] != 0);
}

// acc[mi][ni] = rows (pieces in LDS, xh at the first row block, mi_stride halves between them, lo pieces x_lo halves further on)
// times the 32 NI weight rows whose fragments start at wp.  The two small products of a step have an accumulator of their own, and
// with SUMS = 2 the large ones have two: the large sum is rounded once per 16 or 32 k instead of three times per 16.
// ROWS_FIRST: the rows are the A operand, and a lane holds sixteen rows of one column.  ni_blocks: blocks of 32 weight rows from one
// fragment to the next.
template <int MI, int NI, int SUMS, bool ROWS_FIRST = false>
__device__ __forceinline__ void multiply(const _Float16* __restrict__ wp, long w_lo, int K, const _Float16* xh, int mi_stride,
                                         int x_lo, int lane, floatx16 (&acc)[MI][NI], int ni_blocks = 1) {
    constexpr int kX = SUMS;                                       // (buffers of x: what the registers hold)
    const int steps = K >> 4;                                      // (even)
    const unsigned at = lane * 8;
    const long ni_stride = (long)(K >> 5) * 1024 * ni_blocks;
    xh += at;
    halfx8 wh[2][NI], wl[2][NI], bh[kX][MI], bl[kX][MI];
    floatx16 large[SUMS][MI][NI], small[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int q = 0; q < 16; q++) {
                small[mi][ni][q] = 0.f;
#pragma unroll
                for (int k = 0; k < SUMS; k++) large[k][mi][ni][q] = 0.f;
            }
    auto mfma = [](const halfx8& w, const halfx8& x, const floatx16& c) {
        return ROWS_FIRST ? __builtin_amdgcn_mfma_f32_32x32x16_f16(x, w, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_32x32x16_f16(w, x, c, 0, 0, 0);
    };
    auto load_w = [&](int u, int s) {
        const _Float16* p = wp + 512L * (s < steps ? s : steps - 1);      // (surplus loads of the last trip are never used)
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            wh[u][ni] = *reinterpret_cast<const halfx8*>(p + ni * ni_stride + at);
            wl[u][ni] = *reinterpret_cast<const halfx8*>(p + w_lo + ni * ni_stride + at);
        }
    };
    auto load_x = [&](int u, int s) {
        const int off = 512 * (s < steps ? s : steps - 1);
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            bh[u][mi] = *reinterpret_cast<const halfx8*>(xh + mi * mi_stride + off);
            bl[u][mi] = *reinterpret_cast<const halfx8*>(xh + x_lo + mi * mi_stride + off);
        }
    };
    load_w(0, 0);
    load_w(1, 1);
    if (kX == 2) load_x(0, 0);
    for (int s = 0; s < steps; s += 2) {                           // (no branch inside: the loads stay in flight across trips)
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int x = kX == 2 ? u : 0;
            __builtin_amdgcn_sched_barrier(0);                     // keep this issue order
            load_x(kX == 2 ? 1 - u : 0, kX == 2 ? s + u + 1 : s + u);
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int ni = 0; ni < NI; ni++) {
                    small[mi][ni] = mfma(wh[u][ni], bl[x][mi], small[mi][ni]);
                    large[u % SUMS][mi][ni] = mfma(wh[u][ni], bh[x][mi], large[u % SUMS][mi][ni]);
                }
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
                    small[mi][ni] = mfma(wl[u][ni], bh[x][mi], small[mi][ni]);
            __builtin_amdgcn_sched_barrier(0);
            load_w(u, s + u + 2);
        }
    }
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            acc[mi][ni] = small[mi][ni] + large[0][mi][ni];
            if (SUMS == 2) acc[mi][ni] += large[SUMS - 1][mi][ni];
        }
}

// Where k of a row lies among the pieces of its row block: step, lane of the fragment, k & 7
__device__ __forceinline__ int piece_at(int row, int k) {
    return (((k >> 5) * 2 + ((k >> 3) & 1)) * 64 + row + 32 * ((k >> 4) & 1)) * 8 + (k & 7);
}

// four consecutive k of a row as pieces, or the bits of the fp32 values where the pieces cannot carry the row
__device__ __forceinline__ void store_pieces(_Float16* xh, int x_lo, int at, const float (&v)[4], float scale) {
    halfx4 hi, lo;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float x = v[i] * scale;
        const _Float16 h = (_Float16)x;
        hi[i] = h;
        lo[i] = (_Float16)(x - (float)h);
    }
    *reinterpret_cast<halfx4*>(xh + at) = hi;
    *reinterpret_cast<halfx4*>(xh + x_lo + at) = lo;
}
__device__ __forceinline__ void store_bits(_Float16* xh, int x_lo, int at, const float (&v)[4]) {
    ushort4 hi, lo;
    const unsigned b[4] = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    hi = make_ushort4(b[0] >> 16, b[1] >> 16, b[2] >> 16, b[3] >> 16);
    lo = make_ushort4(b[0] & 0xffff, b[1] & 0xffff, b[2] & 0xffff, b[3] & 0xffff);
    *reinterpret_cast<ushort4*>(xh + at) = hi;
    *reinterpret_cast<ushort4*>(xh + x_lo + at) = lo;
}

// x . w in fp32, k in order, for a row that lies in LDS as bits; weight row n put together from its pieces (row_in_fp32)
__device__ __noinline__ float lds_row_in_fp32(const _Float16* xh, int x_lo, int row, const _Float16* planes, long plane_elems, long n,
                                              int K, float iw) {
    const float inv = unmark_weight(iw);
    float sum = 0.f;
#pragma unroll 1
    for (int k = 0; k < K; k += 8) {
        const int xa = piece_at(row, k);
        const long at = packed_index(n, k, K);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const unsigned hi = __builtin_bit_cast(unsigned short, xh[xa + j]), lo = __builtin_bit_cast(unsigned short, xh[x_lo + xa + j]);
            const float h = (float)planes[at + j], l = (float)planes[plane_elems + at + j];
            sum = fmaf(__uint_as_float(hi << 16 | lo), (fabsf(h) < __builtin_inff() ? h + l : h) * inv, sum);
        }
    }
    return sum;
}

}  // namespace
}  // namespace mg
