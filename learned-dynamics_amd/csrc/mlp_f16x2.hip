// Linear, SiLU, Linear, SiLU, Linear on node- and edge-sized arrays of rows as one kernel, forward and adjoint, in the
// split-fp16 arithmetic of f16x2.hpp.
//
// A workgroup takes 32 MI rows through all layers.  Their activations stay in LDS as fp16 pieces, in the order the matrix cores
// read them; wave w owns the output columns [32 w, + 32) of every layer and reads the fragments of its part of the packed
// weight straight from memory (one contiguous kilobyte per load, resident in the L2).  No barrier stands in
// the loop over k; two stand between layers.  The weight is the A operand of v_mfma_f32_32x32x16_f16 and the rows are B, so
// that a lane of the product holds 16 columns of ONE row in groups of four: bias and activation need no exchange, a row's
// maximum takes one shuffle and a line of LDS, and the next layer's pieces are written eight bytes at a time, whole
// rows being known to the workgroup: a layer's operand is scaled by its rows' own maxima.
//
// Layer by layer (three launches of linear_rows_f16x2_kernel) the same work writes and reads the hidden rows through memory, splits
// a row once per column tile and carries bounds instead of maxima: 128 -> 512 -> 512 -> 512 on 16 336 rows 98 us there, 69 us
// here, 4096 rows 62 and 34 us; 256 -> 384 87 and 52 us; 64 -> 256 53 and 26 us.  What bounds it: with 64 rows a workgroup the matrix cores are
// busy for 25 of 40 thousand cycles of a 512 x 512 layer (sixteen waves issue in turn, waiting for fragments that 32 KB per step
// and CU of L1 traffic delay), and 8 thousand go to activation, split and the two barriers; in long runs the board's power
// (1.1 PFLOP/s for this mix of loads and products on its own, 0.9 here).  Eight waves with two column blocks each were slower
// everywhere (78 us, 40 us): fewer waves to wait beside.
#include "common.hpp"
#include "f16x2.hpp"
#include "rows_in_lds.hpp"
#include "rowsum_finish.hpp"
#include "silu.hpp"

namespace mg {
namespace {

enum { kInfer = 0, kTrain = 1, kAdjoint = 2 };

constexpr int kMaxDim = 512;       // widest layer: 64 rows of it are 128 KB of pieces
constexpr int kMaxWaves = 16;

struct MlpArgs {
    const float* x;
    long R;                        // rows of values; as many rows of tangents lie behind them in the dual kernels
    int K, O, N;                   // columns of x, of the hidden layers, of y
    const _Float16* planes[3];
    const float* inv[3];           // inverse scales of the weights' rows, marks behind them
    const float* bias[3];
    float* y;
    const float* z_in[2];          // adjoint: the hidden layers' inputs of their activation, in the order they are met
    float *z[2], *h[2], *h_max[2]; // training: kept for the adjoint; adjoint: h, h_max are the gradients of z and their row maxima
    float* x_max;
    // LEAKY: x is added to the result (K == N).  127 456 rows, 256 -> 512 -> 256: 10 us forward and 20 in the adjoint (590, 738) for
    // the rows that the workgroup read before, where an addition of its own took 57.
    bool residual;
};

// lanes 16 .. 31 (48 .. 63) of a and lanes 0 .. 15 (32 .. 47) of b change places; done twice, all is as before
__device__ __forceinline__ void swap_rows(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// The rows of x, row(mi, mm) in memory, as pieces, their maxima to row_max: eight lanes to a row, whole rows in registers
// between the maximum and the split
template <int MI, typename Row>
__device__ __forceinline__ void split_rows(_Float16* xh, float* row_max, int K, bool marked, int wave, int waves, int lane, Row row_of) {
    const int x_lo = 32 * MI * K, p = lane & 7;
    for (int grp = wave; grp < 4 * MI; grp += waves) {
        const int lr = grp * 8 + (lane >> 3), mi = lr >> 5, mm = lr & 31;
        const float* row = row_of(mi, mm) + 4 * p;
        float v[kMaxDim / 32][4];
        float mx = 0.f;
#pragma unroll
        for (int j = 0; j < kMaxDim / 32; j++)
            if (32 * j < K) {
                const float4 f = *reinterpret_cast<const float4*>(row + 32 * j);
                v[j][0] = f.x; v[j][1] = f.y; v[j][2] = f.z; v[j][3] = f.w;
            }
#pragma unroll
        for (int j = 0; j < kMaxDim / 32; j++)
            if (32 * j < K)
#pragma unroll
                for (int i = 0; i < 4; i++) mx = fmaxf(mx, fabsf(v[j][i]));
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
        float inv;
        const float scale = pow2_scale(mx, &inv);
        const bool bits = marked || beyond_split(mx);
        const int at = mi * 32 * K + piece_at(mm, 4 * p);
#pragma unroll
        for (int j = 0; j < kMaxDim / 32; j++)
            if (32 * j < K) store_pieces(xh, x_lo, at + 1024 * j, v[j], scale);
        if (__any(bits))                                           // (rare)
#pragma unroll
            for (int j = 0; j < kMaxDim / 32; j++)
                if (32 * j < K && bits) store_bits(xh, x_lo, at + 1024 * j, v[j]);
        if (p == 0) row_max[lr] = mx;
    }
}

// DUAL: the 32 rows of a block are 16 values and their 16 tangents.  LEAKY: LeakyReLU(0.1) in SiLU's place, whose input need not be
// kept (h has its sign), and a last layer of N columns.
template <int MI, int NI, int MODE, bool DUAL, bool LEAKY>
__device__ __forceinline__ void mlp_rows(const MlpArgs& a, long tile, int widest) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    static_assert(!DUAL || MI == 1, "one block of values and tangents");
    static_assert(!LEAKY || (!DUAL && MODE != kInfer), "LeakyReLU: values under differentiation");
    constexpr bool kTail = MODE == kAdjoint || LEAKY;              // the last layer is not O columns wide
    constexpr int TM = 32 * MI, kRows = DUAL ? 16 : TM;
    constexpr int kSums = MI * NI == 1 ? 2 : 1;                    // (what 128 registers hold)
    const int O = a.O;
    _Float16* const xh = reinterpret_cast<_Float16*>(lds);
    float* const row_max = reinterpret_cast<float*>(lds + (size_t)TM * widest * 4);      // [waves][TM]
    float* const fixed = row_max + kMaxWaves / NI * TM;                                  // [kMaxDim]

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int m = lane & 31, G = lane >> 5;
    const long r0 = tile * kRows;
    const bool tangent = DUAL && m >= 16;
    // rows past the end repeat the last one and are not written
    auto row_of = [&](int mi, int mm) {
        const long r = r0 + (DUAL ? mm & 15 : 32 * mi + mm);
        return (r < a.R ? r : a.R - 1) + (DUAL && mm >= 16 ? a.R : 0);
    };
    auto live = [&](int mi) { return r0 + (DUAL ? m & 15 : 32 * mi + m) < a.R; };

    float isx[MI];
    bool odd[MI];
    {
        const bool marked = has_marks(a.inv[0], a.O, lane);
        split_rows<MI>(xh, row_max, a.K, marked, wave, waves, lane, [&](int mi, int mm) { return a.x + row_of(mi, mm) * a.K; });
        __syncthreads();
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            const float mx = row_max[32 * mi + m];
            pow2_scale(mx, &isx[mi]);
            odd[mi] = marked || beyond_split(mx);
            if (MODE != kInfer && a.x_max && wave == 0 && G == 0 && live(mi)) a.x_max[row_of(mi, m)] = mx;
        }
        __syncthreads();                                           // (row_max is written again below)
    }

    constexpr int kFull = kTail ? 2 : 3;                           // layers with O columns
    int K = a.K;
#pragma unroll 1
    for (int l = 0; l < kFull; l++) {
        const int x_lo = TM * K;
        const long w_lo = (long)pad256(O) * K;
        const float* inv = a.inv[l];
        floatx16 acc[MI][NI];
        multiply<MI, NI, kSums>(a.planes[l] + (long)(wave * NI) * (K >> 5) * 1024, w_lo, K, xh, 32 * K, x_lo, lane, acc);

        // rows that the pieces cannot carry (all waves see the same ones)
        bool any_odd = false;
#pragma unroll
        for (int mi = 0; mi < MI; mi++) any_odd |= __any(odd[mi]);
        if (any_odd) {
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
                unsigned rows = (unsigned)__ballot(odd[mi]);
                while (rows) {
                    const int r = __builtin_ctz(rows);
                    rows &= rows - 1;
                    for (int n = tid; n < O; n += blockDim.x)
                        fixed[n] = lds_row_in_fp32(xh + mi * 32 * K, x_lo, r, a.planes[l], w_lo, n, K, inv[n]);
                    __syncthreads();
#pragma unroll
                    for (int ni = 0; ni < NI; ni++)
#pragma unroll
                        for (int q = 0; q < 16; q++) {
                            const float f = fixed[32 * (wave * NI + ni) + 8 * (q / 4) + 4 * G + q % 4];
                            if (m == r) acc[mi][ni][q] = f;
                        }
                    __syncthreads();
                }
            }
        }

        const bool last = !kTail && l == kFull - 1;
        float mx[MI];
#pragma unroll
        for (int mi = 0; mi < MI; mi++) mx[mi] = 0.f;
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int half = 0; half < 2; half++) {                 // (columns in two groups of four, 16 apart)
                const int col = 32 * (wave * NI + ni) + 8 * half + 4 * G;
                float iw[2][4], b[2][4];
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const float4 w4 = *reinterpret_cast<const float4*>(inv + col + 16 * k);
                    iw[k][0] = w4.x; iw[k][1] = w4.y; iw[k][2] = w4.z; iw[k][3] = w4.w;
                    float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (MODE != kAdjoint && a.bias[l] && !tangent) b4 = *reinterpret_cast<const float4*>(a.bias[l] + col + 16 * k);
                    b[k][0] = b4.x; b[k][1] = b4.y; b[k][2] = b4.z; b[k][3] = b4.w;
                }
#pragma unroll
                for (int mi = 0; mi < MI; mi++) {
                    float v[2][4];
                    const bool alive = live(mi);
                    const long at = row_of(mi, m) * O + col;
#pragma unroll
                    for (int k = 0; k < 2; k++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const float p = acc[mi][ni][8 * k + 4 * half + i];
                            v[k][i] = (odd[mi] ? p : p * isx[mi] * iw[k][i]) + b[k][i];
                        }
                    auto put = [&](float* dst) {
                        if (!alive) return;
#pragma unroll
                        for (int k = 0; k < 2; k++) *reinterpret_cast<float4*>(dst + at + 16 * k) = make_float4(v[k][0], v[k][1], v[k][2], v[k][3]);
                    };
                    if (last) {
                        put(a.y);
                        continue;
                    }
                    if constexpr (MODE == kInfer) {
#pragma unroll
                        for (int k = 0; k < 2; k++)
#pragma unroll
                            for (int i = 0; i < 4; i++) v[k][i] = v[k][i] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[k][i]));
                    } else if constexpr (LEAKY) {
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            float h[4] = {1.f, 1.f, 1.f, 1.f};
                            if (MODE == kAdjoint) {
                                const float4 h4 = *reinterpret_cast<const float4*>(a.z_in[l] + at + 16 * k);
                                h[0] = h4.x; h[1] = h4.y; h[2] = h4.z; h[3] = h4.w;
                            }
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                v[k][i] = (MODE == kAdjoint ? h[i] : v[k][i]) > 0.f ? v[k][i] : 0.1f * v[k][i];
                        }
                        put(a.h[l]);
                    } else if constexpr (MODE == kTrain) {
                        put(a.z[l]);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if constexpr (DUAL) {                  // this lane: value and tangent of one of the two columns
                                swap_rows(v[0][i], v[1][i]);
                                const Silu s = silu_short(v[0][i]);
                                v[0][i] = s.f;
                                v[1][i] *= s.d1;
                                swap_rows(v[0][i], v[1][i]);
                            } else {
                                v[0][i] = silu_short(v[0][i]).f;
                                v[1][i] = silu_short(v[1][i]).f;
                            }
                        }
                        put(a.h[l]);
                    } else {
                        float z[2][4];
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            const float4 z4 = *reinterpret_cast<const float4*>(a.z_in[l] + at + 16 * k);
                            z[k][0] = z4.x; z[k][1] = z4.y; z[k][2] = z4.z; z[k][3] = z4.w;
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if constexpr (DUAL) {
                                swap_rows(v[0][i], v[1][i]);
                                swap_rows(z[0][i], z[1][i]);
                                const Silu s = silu_short(z[0][i]);
                                v[0][i] = v[0][i] * s.d1 + v[1][i] * z[1][i] * s.d2;
                                v[1][i] *= s.d1;
                                swap_rows(v[0][i], v[1][i]);
                            } else {
                                v[0][i] *= silu_short(z[0][i]).d1;
                                v[1][i] *= silu_short(z[1][i]).d1;
                            }
                        }
                        put(a.h[l]);
                    }
#pragma unroll
                    for (int k = 0; k < 2; k++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            acc[mi][ni][8 * k + 4 * half + i] = v[k][i];
                            mx[mi] = fmaxf(mx[mi], fabsf(v[k][i]));
                        }
                }
            }
        if (last) return;

        // the next layer's rows: their maxima, then their pieces in the place of this layer's
        const bool marked = has_marks(a.inv[l + 1 < kFull ? l + 1 : kFull - 1], O, lane) ||
                            (kTail && l + 1 == kFull && a.y && has_marks(a.inv[2], a.N, lane));
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            mx[mi] = fmaxf(mx[mi], __shfl_xor(mx[mi], 32));
            if (G == 0) row_max[wave * TM + 32 * mi + m] = mx[mi];
        }
        __syncthreads();
        K = O;
        const int lo = TM * O;
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            float top = 0.f;
            for (int w = 0; w < waves; w++) top = fmaxf(top, row_max[w * TM + 32 * mi + m]);
            const float scale = pow2_scale(top, &isx[mi]);
            odd[mi] = marked || beyond_split(top);
            if (MODE != kInfer && wave == 0 && G == 0 && live(mi)) a.h_max[l][row_of(mi, m)] = top;
            auto each = [&](auto store) {
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const float v[4] = {acc[mi][ni][4 * t], acc[mi][ni][4 * t + 1], acc[mi][ni][4 * t + 2], acc[mi][ni][4 * t + 3]};
                        store(mi * 32 * O + piece_at(m, 32 * (wave * NI + ni) + 8 * t + 4 * G), v);
                    }
            };
            each([&](int at, const float (&v)[4]) { store_pieces(xh, lo, at, v, scale); });
            if (__any(odd[mi]))                                    // (rare)
                each([&](int at, const float (&v)[4]) { if (odd[mi]) store_bits(xh, lo, at, v); });
        }
        __syncthreads();
    }

    // adjoint: the gradient of x; O -> N columns, 32 to a wave at a time
    if constexpr (kTail) {
        if (!a.y) return;
        const int N = a.N, x_lo = TM * O;
        const long w_lo = (long)pad256(N) * O;
        const float* inv = a.inv[2];
#pragma unroll 1
        for (int nb = wave; nb < N / 32; nb += waves) {
            floatx16 acc[MI][1];
            multiply<MI, 1, kSums>(a.planes[2] + (long)nb * (O >> 5) * 1024, w_lo, O, xh, 32 * O, x_lo, lane, acc);
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
                if (!live(mi)) continue;
                float* out = a.y + row_of(mi, m) * N + 32 * nb + 4 * G;
                const float* res = LEAKY && a.residual ? a.x + row_of(mi, m) * N + 32 * nb + 4 * G : nullptr;
                const float* bias = MODE == kAdjoint ? nullptr : a.bias[2];
                if (odd[mi]) {
#pragma unroll 1
                    for (int q = 0; q < 16; q++) {
                        const int c = 8 * (q / 4) + q % 4, n = 32 * nb + 4 * G + c;
                        out[c] = lds_row_in_fp32(xh + mi * 32 * O, x_lo, m, a.planes[2], w_lo, n, O, inv[n]) + (bias ? bias[n] : 0.f) +
                                 (res ? res[c] : 0.f);
                    }
                    continue;
                }
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const float4 iw = *reinterpret_cast<const float4*>(inv + 32 * nb + 8 * t + 4 * G);
                    float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (bias) b = *reinterpret_cast<const float4*>(bias + 32 * nb + 8 * t + 4 * G);
                    if (res) {
                        const float4 r = *reinterpret_cast<const float4*>(res + 8 * t);
                        b.x += r.x; b.y += r.y; b.z += r.z; b.w += r.w;
                    }
                    *reinterpret_cast<float4*>(out + 8 * t) =
                        make_float4(acc[mi][0][4 * t] * isx[mi] * iw.x + b.x, acc[mi][0][4 * t + 1] * isx[mi] * iw.y + b.y,
                                    acc[mi][0][4 * t + 2] * isx[mi] * iw.z + b.z, acc[mi][0][4 * t + 3] * isx[mi] * iw.w + b.w);
                }
            }
        }
    }
}

template <int MI, int NI, int MODE, bool DUAL, bool LEAKY = false>
__global__ void __launch_bounds__(64 * kMaxWaves / NI, 4) mlp_f16x2_kernel(const MlpArgs a) {
    mlp_rows<MI, NI, MODE, DUAL, LEAKY>(a, blockIdx.x, a.K > a.O ? a.K : a.O);
}

// Several MLPs whose layers are equally wide in one launch: workgroups first[k] .. first[k + 1] - 1 are the k-th one's
constexpr int kMany = 16;          // (2.9 KB of kernel arguments)
struct MlpMany {
    MlpArgs job[kMany];
    unsigned first[kMany + 1];
    int widest;
};
template <int MI>
__global__ void __launch_bounds__(64 * kMaxWaves, 4) mlp_many_f16x2_kernel(const MlpMany p) {
    int k = 0;
    while (blockIdx.x >= p.first[k + 1]) k++;                      // (the last one ends with the grid)
    mlp_rows<MI, 1, kInfer, false, false>(p.job[k], blockIdx.x - p.first[k], p.widest);
}

// Linear, LeakyReLU(0.1), Linear, LeakyReLU(0.1), then the sum over the rows of each segment (seg ascending); the hidden rows stay in
// LDS and the second layer's in registers.  64 rows a workgroup, wave w owns 32 columns of both layers.  In the second
// layer the rows are the A operand: a lane holds rows of ONE column, and after a swap of the halves of the wave lanes 0 .. 31
// hold all rows of the first block of 32 and lanes 32 .. 63 those of the second, so that a segment's rows add up in row
// order in a register, at 64 additions a wave.  Partial rows of segments that leave a block go to slots A / B (rowsum_finish.hpp).
// A plain linear that stores its rows and a second that reads them and sums (the route for wider layers) took, with 256 -> 512 ->
// 512 and 15 rows a segment, 446 us for 131 072 rows against 341 here, 109 and 98 for 32 768, 55 and 39 for 8192; 128 -> 256 149
// and 106, 51 and 29, 38 and 18; 64 -> 128 80 and 42, 38 and 17, 22 and 16.  Bound as the kernel above: 0.9 PFLOP/s, counting the
// three products, in long runs.
struct RowsumArgs {
    const float* x;
    long R;
    int K, O;
    const _Float16* planes[2];
    const float* inv[2];
    const float* bias[2];
    const int* seg;
    long n_blocks, out_stride;
    float *slots, *out;
};

__device__ __forceinline__ float leaky(float v) { return v >= 0.f ? v : 0.1f * v; }

__global__ void __launch_bounds__(64 * kMaxWaves, 4) mlp_rowsum_f16x2_kernel(const RowsumArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int MI = 2, TM = 32 * MI;
    const int O = a.O, widest = a.K > O ? a.K : O;
    _Float16* const xh = reinterpret_cast<_Float16*>(lds);
    float* const row_max = reinterpret_cast<float*>(lds + (size_t)TM * widest * 4);      // [waves][TM]
    float* const row_inv = row_max + kMaxWaves * TM;                                     // [TM]
    float* const fixed = row_inv + TM;                                                   // [kMaxDim]

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int m = lane & 31, G = lane >> 5;
    const long r0 = (long)blockIdx.x * TM;
    // rows past the end repeat the last one and are not summed
    auto row_of = [&](int r) { return r0 + r < a.R ? r0 + r : a.R - 1; };

    float isx[MI];
    bool odd[MI];
    floatx16 acc[MI][1];
    auto each_odd_row = [&](int l, int K, auto set) {              // set(mi, row, its sums in `fixed`)
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            unsigned rows = (unsigned)__ballot(odd[mi]);
            while (rows) {
                const int r = __builtin_ctz(rows);
                rows &= rows - 1;
                for (int n = tid; n < O; n += blockDim.x)
                    fixed[n] = lds_row_in_fp32(xh + mi * 32 * K, TM * K, r, a.planes[l], (long)pad256(O) * K, n, K, a.inv[l][n]);
                __syncthreads();
                set(mi, r);
                __syncthreads();
            }
        }
    };

    {
        const bool marked = has_marks(a.inv[0], O, lane);
        split_rows<MI>(xh, row_max, a.K, marked, wave, waves, lane, [&](int mi, int mm) { return a.x + row_of(32 * mi + mm) * a.K; });
        __syncthreads();
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            const float mx = row_max[32 * mi + m];
            pow2_scale(mx, &isx[mi]);
            odd[mi] = marked || beyond_split(mx);
        }
        __syncthreads();                                           // (row_max is written again below)
    }
    multiply<MI, 1, 1>(a.planes[0] + (long)wave * (a.K >> 5) * 1024, (long)pad256(O) * a.K, a.K, xh, 32 * a.K, TM * a.K, lane, acc);
    if (__any(odd[0] || odd[1]))
        each_odd_row(0, a.K, [&](int mi, int r) {
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const float f = fixed[32 * wave + 8 * (q / 4) + 4 * G + q % 4];
                if (m == r) acc[mi][0][q] = f;
            }
        });
    float mx[MI] = {0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int col = 32 * wave + 8 * t + 4 * G;
        const float4 w4 = *reinterpret_cast<const float4*>(a.inv[0] + col);
        const float4 b4 = a.bias[0] ? *reinterpret_cast<const float4*>(a.bias[0] + col) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float iw[4] = {w4.x, w4.y, w4.z, w4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float p = acc[mi][0][4 * t + i];
                const float v = leaky((odd[mi] ? p : p * isx[mi] * iw[i]) + b[i]);
                acc[mi][0][4 * t + i] = v;
                mx[mi] = fmaxf(mx[mi], fabsf(v));
            }
    }
    const bool marked = has_marks(a.inv[1], O, lane);
#pragma unroll
    for (int mi = 0; mi < MI; mi++) {
        mx[mi] = fmaxf(mx[mi], __shfl_xor(mx[mi], 32));
        if (G == 0) row_max[wave * TM + 32 * mi + m] = mx[mi];
    }
    __syncthreads();
#pragma unroll
    for (int mi = 0; mi < MI; mi++) {
        float top = 0.f;
        for (int w = 0; w < waves; w++) top = fmaxf(top, row_max[w * TM + 32 * mi + m]);
        const float scale = pow2_scale(top, &isx[mi]);
        odd[mi] = marked || beyond_split(top);
        if (wave == 0 && G == 0) row_inv[32 * mi + m] = isx[mi];
        auto each = [&](auto store) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float v[4] = {acc[mi][0][4 * t], acc[mi][0][4 * t + 1], acc[mi][0][4 * t + 2], acc[mi][0][4 * t + 3]};
                store(mi * 32 * O + piece_at(m, 32 * wave + 8 * t + 4 * G), v);
            }
        };
        each([&](int at, const float (&v)[4]) { store_pieces(xh, TM * O, at, v, scale); });
        if (__any(odd[mi]))                                        // (rare)
            each([&](int at, const float (&v)[4]) { if (odd[mi]) store_bits(xh, TM * O, at, v); });
    }
    __syncthreads();

    // second layer: lane = column 32 wave + m, register q = row 8 (q / 4) + 4 G + q % 4 of the block
    multiply<MI, 1, 1, true>(a.planes[1] + (long)wave * (O >> 5) * 1024, (long)pad256(O) * O, O, xh, 32 * O, TM * O, lane, acc);
    const int col = 32 * wave + m;
    const float iw = a.inv[1][col], b = a.bias[1] ? a.bias[1][col] : 0.f;
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const float4 f = *reinterpret_cast<const float4*>(row_inv + 32 * mi + 8 * t + 4 * G);
            const float inv[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int i = 0; i < 4; i++) acc[mi][0][4 * t + i] = acc[mi][0][4 * t + i] * inv[i] * iw + b;
        }
    if (__any(odd[0] || odd[1]))
        each_odd_row(1, O, [&](int mi, int r) {
            const float f = fixed[col] + b;
#pragma unroll
            for (int q = 0; q < 16; q++)
                if (8 * (q / 4) + 4 * G + q % 4 == r) acc[mi][0][q] = f;
        });
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(leaky(acc[0][0][q])), __float_as_uint(leaky(acc[1][0][q])), false, false);
        acc[0][0][q] = __uint_as_float(s[0]);                      // row 8 (q / 4) + q % 4 of block G
        acc[1][0][q] = __uint_as_float(s[1]);                      // row 8 (q / 4) + 4 + q % 4
    }
    const long left = a.R - r0 - 32 * G, block = 2 * (long)blockIdx.x + G;
    const int rows = left < 32 ? (int)left : 32;                   // of this half's block; none if <= 0
    const int my_seg = a.seg[row_of(lane)], before = __shfl_up(my_seg, 1);
    const unsigned long long starts = __ballot(m > 0 && my_seg != before);
    float* const slot = a.slots + (block < a.n_blocks ? block : 0) * O + col;
    float* to = slot;                                              // of a block's first run; later ones lie inside the block
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 32; r++) {
        if (r > 0 && (starts >> r & 0x100000001ull)) {
            const int s_lo = __builtin_amdgcn_readlane(my_seg, r), s_hi = __builtin_amdgcn_readlane(my_seg, 32 + r);
            if (starts >> (r + 32 * G) & 1) {                      // (never at a row past the end)
                *to = sum;
                sum = 0.f;
                to = a.out + (long)(G ? s_hi : s_lo) * a.out_stride + col;
            }
        }
        const float v = acc[r >> 2 & 1][0][4 * (r >> 3) + (r & 3)];
        sum += r < rows ? v : 0.f;
    }
    if (rows <= 0) return;
    if (to != slot && rows == 32) to = a.slots + (a.n_blocks + block) * O + col;
    *to = sum;
}

template <int MI, int NI, int MODE, bool DUAL, bool LEAKY = false>
int launch(const MlpArgs& a, hipStream_t st) {
    const auto kernel = mlp_f16x2_kernel<MI, NI, MODE, DUAL, LEAKY>;
    const int widest = a.K > a.O ? a.K : a.O;
    const size_t lds = (size_t)32 * MI * widest * 4 + (kMaxWaves / NI * 32 * MI + kMaxDim) * sizeof(float);
    // more than 64 KB of dynamic LDS has to be asked for (per device, so on every call)
    if (lds > 65536) MG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const long tiles = ceil_div(a.R, DUAL ? 16 : 32 * MI);
    MG_REQUIRE(tiles <= 0x7fffffffL, "mg_mlp_f16x2: grid too large (rows=%ld)", a.R);
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(2 * a.O / NI), lds, st, a);
    return check_launch("mg_mlp_f16x2");
}

// 32 rows a workgroup while the chip holds all of them at once, 64 beyond (the weights are read half as often):
// 128 -> 512 on 8192 rows 42 against 53 us, on 16 336 83 against 69; 128 -> 128 on 16 336 14.5 against 18.0
bool wide_tiles(const MlpArgs& a) { return ceil_div(a.R, 32) * (a.O / 32) > 256 * kMaxWaves; }

template <int MODE>
int choose(const MlpArgs& a, bool dual, hipStream_t st) {
    if constexpr (MODE == kInfer) {
        if (wide_tiles(a)) return launch<2, 1, MODE, false>(a, st);
        return launch<1, 1, MODE, false>(a, st);
    } else {
        // The passes over memory between the layers are longer here (z and h, or z and the gradients): from more tiles than CUs on two
        // workgroups of half as many waves share a CU, and one multiplies while the other writes.  128 -> 512, forward / adjoint, one
        // / two workgroups: 8192 rows 58 / 54 and 62 / 56 us, 12 000 96 / 96 and 94 / 88, 16 384 119 / 108 and 102 / 95,
        // 2 x 39 000 with tangents 576 / 554 and 528 / 501.
        const long tiles = ceil_div(a.R, dual ? 16 : 32);
        if (a.O > 256 && a.O % 64 == 0 && tiles > 256) return dual ? launch<1, 2, MODE, true>(a, st) : launch<1, 2, MODE, false>(a, st);
        return dual ? launch<1, 1, MODE, true>(a, st) : launch<1, 1, MODE, false>(a, st);
    }
}

template <int MI>
int launch_many(MlpMany& p, int jobs, hipStream_t st) {
    const int O = p.job[0].O;
    p.widest = O;
    long tiles = 0;
    for (int k = 0; k < jobs; k++) {
        p.widest = p.job[k].K > p.widest ? p.job[k].K : p.widest;
        p.first[k] = (unsigned)tiles;
        tiles += ceil_div(p.job[k].R, 32 * MI);
        MG_REQUIRE(tiles <= 0x7fffffffL, "mg_mlp_f16x2_forward_many: grid too large");
    }
    for (int k = jobs; k <= kMany; k++) p.first[k] = (unsigned)tiles;
    const size_t lds = (size_t)32 * MI * p.widest * 4 + (kMaxWaves * 32 * MI + kMaxDim) * sizeof(float);
    if (lds > 65536)
        MG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(mlp_many_f16x2_kernel<MI>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(mlp_many_f16x2_kernel<MI>, dim3((unsigned)tiles), dim3(2 * O), lds, st, p);
    return check_launch("mg_mlp_f16x2_forward_many");
}

// Two column blocks to a wave, so that two workgroups share a CU, where the width has them: by the width alone and not by the rows as
// above, since the slope at zero should not depend on how many rows a call has.  127 000 rows, 256 -> 512 -> 512 -> 256: 0.57 ms, the
// adjoint 0.72 (weights out of the L2 at 14 TB/s, 1.3 GB of kept rows); four linears, the activations, their derivatives and the row
// maxima in passes of their own took 0.4 ms more of a training step with two such MLPs each way.
template <int MODE>
int launch_leaky(const MlpArgs& a, hipStream_t st) {
    return a.O % 64 == 0 ? launch<1, 2, MODE, false, true>(a, st) : launch<1, 1, MODE, false, true>(a, st);
}

int fill(MlpArgs& a, const void* const* packed, int K, int O, int N) {
    for (int l = 0; l < 3; l++) {
        // (forward: K -> O -> O -> O; adjoint: O -> O -> O -> N)
        const int in = l == 0 ? K : O, out = l == 2 ? N : O;
        if (!packed[l]) continue;
        if (!aligned16(packed[l])) return 0;
        a.planes[l] = static_cast<const _Float16*>(packed[l]);
        a.inv[l] = reinterpret_cast<const float*>(a.planes[l] + 2L * ((out + 255) / 256 * 256) * in);
    }
    return 1;
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_mlp_f16x2_supported(int dim_in, int dim) {
    return dim_in >= 32 && dim_in <= kMaxDim && dim_in % 32 == 0 && dim >= 32 && dim <= kMaxDim && dim % 32 == 0;
}

int mg_mlp_f16x2_forward(const mg_mlp_f16x2* p, mg_stream_t stream) {
    MG_REQUIRE(p != nullptr && p->rows >= 0 && mg_mlp_f16x2_supported(p->dim_in, p->dim),
               "mg_mlp_f16x2_forward: dimensions must be multiples of 32 up to %d", kMaxDim);
    if (p->rows == 0) return MG_OK;
    MlpArgs a{};
    a.x = p->x;
    a.R = p->rows;
    a.K = p->dim_in;
    a.O = a.N = p->dim;
    a.y = p->y;
    a.x_max = p->x_rowmax;
    bool keep = false, keep_all = true;
    for (int l = 0; l < 2; l++) {
        a.z[l] = p->z[l];
        a.h[l] = p->h[l];
        a.h_max[l] = p->h_rowmax[l];
        keep |= p->z[l] || p->h[l] || p->h_rowmax[l];
        keep_all &= p->z[l] && p->h[l] && p->h_rowmax[l] && aligned16(p->z[l]) && aligned16(p->h[l]);
    }
    for (int l = 0; l < 3; l++) {
        a.bias[l] = p->bias[l];
        MG_REQUIRE(p->packed_W[l] && (!p->bias[l] || aligned16(p->bias[l])), "mg_mlp_f16x2_forward: null or unaligned weight or bias");
    }
    MG_REQUIRE(fill(a, p->packed_W, a.K, a.O, a.N) && a.x && a.y && aligned16(a.x) && aligned16(a.y) && keep == (keep && keep_all) &&
                   (keep || !p->dual),
               "mg_mlp_f16x2_forward: null or unaligned pointer");
    return keep ? choose<kTrain>(a, p->dual, (hipStream_t)stream) : choose<kInfer>(a, false, (hipStream_t)stream);
}

// kMany to a launch, each MLP in the tiles that it has alone: 64 rows leave no registers for the small products' own sums, so that a
// row would be less exact beside others (128 -> 512 2.25e-7 of the 2-norm from float64, 1.88e-7 in 32 rows)
static int forward_many(const mg_mlp_f16x2* const* in, int jobs, hipStream_t st) {
    MlpMany p[2] = {};
    int used[2] = {0, 0};
    auto send = [&](int wide) {
        const int count = used[wide];
        used[wide] = 0;
        return count == 0 ? MG_OK : wide ? launch_many<2>(p[1], count, st) : launch_many<1>(p[0], count, st);
    };
    for (int k = 0; k < jobs; k++) {
        const mg_mlp_f16x2& m = *in[k];
        MG_REQUIRE(m.rows >= 0 && mg_mlp_f16x2_supported(m.dim_in, m.dim) && m.dim == in[0]->dim && !m.dual && !m.z[0] && !m.h[0] && !m.x_rowmax,
                   "mg_mlp_f16x2_forward_many: inference only, one width, dimensions multiples of 32 up to %d", kMaxDim);
        MlpArgs a{};
        a.x = m.x;
        a.R = m.rows;
        a.K = m.dim_in;
        a.O = a.N = m.dim;
        a.y = m.y;
        for (int l = 0; l < 3; l++) {
            a.bias[l] = m.bias[l];
            MG_REQUIRE(m.packed_W[l] && (!m.bias[l] || aligned16(m.bias[l])), "mg_mlp_f16x2_forward_many: null or unaligned weight or bias");
        }
        MG_REQUIRE(fill(a, m.packed_W, a.K, a.O, a.N) && (m.rows == 0 || (a.x && a.y && aligned16(a.x) && aligned16(a.y))),
                   "mg_mlp_f16x2_forward_many: null or unaligned pointer");
        if (m.rows == 0) continue;
        const int wide = wide_tiles(a);
        p[wide].job[used[wide]++] = a;
        if (used[wide] == kMany)
            if (int code = send(wide)) return code;
    }
    if (int code = send(0)) return code;
    return send(1);
}

int mg_mlp_f16x2_forward_many(const mg_mlp_f16x2* const* args, int count, mg_stream_t stream) {
    MG_REQUIRE(count >= 0 && (count == 0 || args), "mg_mlp_f16x2_forward_many: null pointer");
    for (int k = 0; k < count; k++) MG_REQUIRE(args[k] && args[k]->dim == args[0]->dim, "mg_mlp_f16x2_forward_many: MLPs of one width");
    return count ? forward_many(args, count, (hipStream_t)stream) : MG_OK;
}

int mg_mlp_f16x2_forward_pair(const mg_mlp_f16x2* first, const mg_mlp_f16x2* second, mg_stream_t stream) {
    const mg_mlp_f16x2* in[2] = {first, second};
    return mg_mlp_f16x2_forward_many(in, 2, stream);
}

int mg_mlp_f16x2_adjoint(const mg_mlp_f16x2_grad* p, mg_stream_t stream) {
    MG_REQUIRE(p != nullptr && p->rows >= 0 && mg_mlp_f16x2_supported(p->dim_in, p->dim),
               "mg_mlp_f16x2_adjoint: dimensions must be multiples of 32 up to %d", kMaxDim);
    if (p->rows == 0) return MG_OK;
    MlpArgs a{};
    a.x = p->dy;
    a.R = p->rows;
    a.K = a.O = p->dim;
    a.N = p->dim_in;
    a.y = p->dx;
    a.x_max = p->dy_rowmax;
    for (int l = 0; l < 2; l++) {                                  // met in reverse
        a.z_in[l] = p->z[1 - l];
        a.h[l] = p->dz[1 - l];
        a.h_max[l] = p->dz_rowmax[1 - l];
        MG_REQUIRE(a.z_in[l] && a.h[l] && a.h_max[l] && aligned16(a.z_in[l]) && aligned16(a.h[l]),
                   "mg_mlp_f16x2_adjoint: null or unaligned pointer");
    }
    const void* packed[3] = {p->packed_Wt[2], p->packed_Wt[1], p->packed_Wt[0]};
    MG_REQUIRE(fill(a, packed, a.O, a.O, a.N) && packed[0] && packed[1] && (packed[2] || !a.y) && a.x && aligned16(a.x) && aligned16(a.y),
               "mg_mlp_f16x2_adjoint: null or unaligned pointer");
    return choose<kAdjoint>(a, p->dual, (hipStream_t)stream);
}

int mg_mlp_leaky_f16x2_supported(int dim_in, int dim, int dim_out) {
    return mg_mlp_f16x2_supported(dim_in, dim) && mg_mlp_f16x2_supported(dim_out, dim);
}

static int mlp_leaky_forward(const mg_mlp_leaky_f16x2* p, bool residual, mg_stream_t stream) {
    MG_REQUIRE(p != nullptr && p->rows >= 0 && mg_mlp_leaky_f16x2_supported(p->dim_in, p->dim, p->dim_out),
               "mg_mlp_leaky_f16x2_forward: dimensions must be multiples of 32 up to %d", kMaxDim);
    MG_REQUIRE(!residual || p->dim_in == p->dim_out, "mg_mlp_leaky_f16x2_residual_forward: dim_in == dim_out expected");
    if (p->rows == 0) return MG_OK;
    MlpArgs a{};
    a.residual = residual;
    a.x = p->x;
    a.R = p->rows;
    a.K = p->dim_in;
    a.O = p->dim;
    a.N = p->dim_out;
    a.y = p->y;
    a.x_max = p->x_rowmax;
    for (int l = 0; l < 3; l++) {
        a.bias[l] = p->bias[l];
        MG_REQUIRE(p->packed_W[l] && (!p->bias[l] || aligned16(p->bias[l])), "mg_mlp_leaky_f16x2_forward: null or unaligned weight or bias");
        if (l == 2) break;
        a.h[l] = p->h[l];
        a.h_max[l] = p->h_rowmax[l];
        MG_REQUIRE(a.h[l] && a.h_max[l] && aligned16(a.h[l]), "mg_mlp_leaky_f16x2_forward: null or unaligned pointer");
    }
    MG_REQUIRE(fill(a, p->packed_W, a.K, a.O, a.N) && a.x && a.y && aligned16(a.x) && aligned16(a.y),
               "mg_mlp_leaky_f16x2_forward: null or unaligned pointer");
    return launch_leaky<kTrain>(a, (hipStream_t)stream);
}

static int mlp_leaky_adjoint(const mg_mlp_leaky_f16x2_grad* p, bool residual, mg_stream_t stream) {
    MG_REQUIRE(p != nullptr && p->rows >= 0 && mg_mlp_leaky_f16x2_supported(p->dim_in, p->dim, p->dim_out),
               "mg_mlp_leaky_f16x2_adjoint: dimensions must be multiples of 32 up to %d", kMaxDim);
    MG_REQUIRE(!residual || p->dim_in == p->dim_out, "mg_mlp_leaky_f16x2_residual_adjoint: dim_in == dim_out expected");
    if (p->rows == 0) return MG_OK;
    MlpArgs a{};
    a.residual = residual;
    a.x = p->dy;
    a.R = p->rows;
    a.K = p->dim_out;
    a.O = p->dim;
    a.N = p->dim_in;
    a.y = p->dx;
    a.x_max = p->dy_rowmax;
    for (int l = 0; l < 2; l++) {                                  // met in reverse
        a.z_in[l] = p->h[1 - l];
        a.h[l] = p->dz[1 - l];
        a.h_max[l] = p->dz_rowmax[1 - l];
        MG_REQUIRE(a.z_in[l] && a.h[l] && a.h_max[l] && aligned16(a.z_in[l]) && aligned16(a.h[l]),
                   "mg_mlp_leaky_f16x2_adjoint: null or unaligned pointer");
    }
    const void* packed[3] = {p->packed_Wt[2], p->packed_Wt[1], p->packed_Wt[0]};
    MG_REQUIRE(fill(a, packed, a.K, a.O, a.N) && packed[0] && packed[1] && (packed[2] || !a.y) && a.x && aligned16(a.x) && aligned16(a.y),
               "mg_mlp_leaky_f16x2_adjoint: null or unaligned pointer");
    return launch_leaky<kAdjoint>(a, (hipStream_t)stream);
}

int mg_mlp_leaky_f16x2_forward(const mg_mlp_leaky_f16x2* p, mg_stream_t stream) { return mlp_leaky_forward(p, false, stream); }
int mg_mlp_leaky_f16x2_adjoint(const mg_mlp_leaky_f16x2_grad* p, mg_stream_t stream) { return mlp_leaky_adjoint(p, false, stream); }
int mg_mlp_leaky_f16x2_residual_forward(const mg_mlp_leaky_f16x2* p, mg_stream_t stream) { return mlp_leaky_forward(p, true, stream); }
int mg_mlp_leaky_f16x2_residual_adjoint(const mg_mlp_leaky_f16x2_grad* p, mg_stream_t stream) { return mlp_leaky_adjoint(p, true, stream); }

static int mlp_rowsum(const void* packed_W1, const float* b1, const void* packed_W2, const float* b2, const float* x, long rows, int dim_in,
                      int dim, const int* row_ptr, const int* seg, long n_out, void* workspace, float* out, long out_stride, float* row_max,
                      int max_stride, mg_stream_t stream) {
    MG_REQUIRE(mg_mlp_f16x2_supported(dim_in, dim), "mg_mlp_leaky_rowsum_f16x2: dimensions must be multiples of 32 up to %d", kMaxDim);
    MG_REQUIRE(rows >= 0 && n_out >= 0 && rows < (1L << 31) && n_out < (1L << 31), "mg_mlp_leaky_rowsum_f16x2: bad size");
    if (n_out == 0) return MG_OK;
    MG_REQUIRE(row_ptr && out && aligned16(out), "mg_mlp_leaky_rowsum_f16x2: null or unaligned output");
    hipStream_t st = (hipStream_t)stream;
    RowsumArgs a{};
    a.x = x;
    a.R = rows;
    a.K = dim_in;
    a.O = dim;
    a.seg = seg;
    a.n_blocks = ceil_div(rows, 32);
    a.slots = static_cast<float*>(workspace);
    a.out = out;
    a.out_stride = out_stride;
    if (rows > 0) {
        const void* packed[2] = {packed_W1, packed_W2};
        const float* bias[2] = {b1, b2};
        for (int l = 0; l < 2; l++) {
            MG_REQUIRE(packed[l] && aligned16(packed[l]) && (!bias[l] || aligned16(bias[l])), "mg_mlp_leaky_rowsum_f16x2: null or unaligned weight or bias");
            a.planes[l] = static_cast<const _Float16*>(packed[l]);
            a.inv[l] = reinterpret_cast<const float*>(a.planes[l] + 2L * ((dim + 255) / 256 * 256) * (l == 0 ? dim_in : dim));
            a.bias[l] = bias[l];
        }
        MG_REQUIRE(x && seg && workspace && aligned16(x) && aligned16(workspace), "mg_mlp_leaky_rowsum_f16x2: null or unaligned row operand");
        const int widest = dim_in > dim ? dim_in : dim;
        const size_t lds = (size_t)64 * widest * 4 + (kMaxWaves * 64 + 64 + kMaxDim) * sizeof(float);
        if (lds > 65536)
            MG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(mlp_rowsum_f16x2_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(mlp_rowsum_f16x2_kernel, dim3((unsigned)ceil_div(rows, 64)), dim3(2 * dim), lds, st, a);
        if (int code = check_launch("mg_mlp_leaky_rowsum_f16x2")) return code;
    }
    const dim3 finish((unsigned)ceil_div(n_out * (dim / 4), 256));
    if (row_max)
        rowsum_finish_into_kernel<<<finish, dim3(256), 0, st>>>(row_ptr, n_out, a.n_blocks, dim, a.slots, 1.f, out, out_stride, row_max,
                                                                max_stride, nullptr, nullptr, 0);
    else
        rowsum_finish_kernel<<<finish, dim3(256), 0, st>>>(row_ptr, n_out, a.n_blocks, dim, a.slots, 1.f, out);
    return check_launch("rowsum_finish_kernel");
}

int mg_mlp_leaky_rowsum_f16x2_workspace_bytes(long rows, int dim, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && rows >= 0 && dim >= 0, "mg_mlp_leaky_rowsum_f16x2_workspace_bytes: bad argument");
    *bytes = (size_t)(2 * ceil_div(rows, 32) * dim) * sizeof(float);
    return MG_OK;
}

int mg_mlp_leaky_rowsum_f16x2(const void* packed_W1, const float* b1, const void* packed_W2, const float* b2, const float* x,
                              long rows, int dim_in, int dim, const int* row_ptr, const int* seg, long n_out, void* workspace,
                              float* out, mg_stream_t stream) {
    return mlp_rowsum(packed_W1, b1, packed_W2, b2, x, rows, dim_in, dim, row_ptr, seg, n_out, workspace, out, dim, nullptr, 0, stream);
}

int mg_mlp_leaky_rowsum_f16x2_into(const void* packed_W1, const float* b1, const void* packed_W2, const float* b2, const float* x,
                                   long rows, int dim_in, int dim, const int* row_ptr, const int* seg, long n_out, void* workspace,
                                   float* out, long out_stride, float* row_max, int max_stride, mg_stream_t stream) {
    MG_REQUIRE(row_max && dim % 256 == 0 && out_stride >= dim && out_stride % 4 == 0 && max_stride >= dim / 256,
               "mg_mlp_leaky_rowsum_f16x2_into: rows of at least dim floats in fours, dim a multiple of 256, and their maxima");
    return mlp_rowsum(packed_W1, b1, packed_W2, b2, x, rows, dim_in, dim, row_ptr, seg, n_out, workspace, out, out_stride, row_max,
                      max_stride, stream);
}

}  // extern "C"
