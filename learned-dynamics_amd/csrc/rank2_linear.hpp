// The bias-free output linear of the rank-2 channel applied to a node's rank-2 sums (or products) while they are
// still in registers, shared by the edge kernel of Messages and the node kernel of SelfTensProds
// (archs/diffuser_atoms15.py:82-94, 244-252):
//     out[o][comp i] = sum over (label, channel) of s2[i][label][channel] Y2[o][label chan + channel],  o < dim_d <= 16.
// A workgroup is four waves, a wave holds one 64-channel chunk of one node (lane = channel, registers = the 45
// (comp, label) values), and the 4 / chunks nodes of a workgroup are whole.  The 9 components are the rows of 16-row matrix
// instructions, their k the labels and channels of the chunk: some labels at a time the wave's values go through rows of its own
// LDS, from which a lane takes one component at four channels (rows 9 .. 15 of the operand repeat others and are not used).  The
// waves' partial 9 x 16 results are added through LDS by the first wave of each node.
//
// The products are those of f16x2.hpp with the lo lo term (which the matrix cores have time for), scaled per wave by the largest of its
// values and per output by the weight: 40 instructions (16x16x32 in fp16) of 16 cycles.  On the fp32 matrix cores (16x16x4) it is 80 of
// 32 cycles, and those keep the vector instructions of the other waves waiting (an fp32 matrix instruction and eight multiply-adds
// beside it take 53 cycles, 34 and 24 by themselves): they remain for values or weights that the pieces cannot carry (pieces_fit) and
// where fp32 products are asked for.
// The edge kernel with 256 channels, 16 outputs and 20 edges a node: 2.30 -> 2.28 ms at 65 536 nodes, 69.6 -> 65.4 us at 2048.  Distance of
// a component from float64 (2-norm, normal values): 1.33e-7 for 1.63e-7 in fp32 in the node kernel, 1.38e-7 for 1.74e-7 in the edge
// kernel, and 1.64e-7 without the lo lo term.  A scale for each component, with no fp32 path for components of unlike size, takes 60
// instructions and 12 to 18 spilled registers more: 70.5 us for the edge kernel at 2048 nodes, 890 against 775 for the node kernel at 65 536.
#pragma once
#include "common.hpp"
#include "f16x2.hpp"
#include <type_traits>

namespace mg {

constexpr int kTrPitch = 68;   // dwords per LDS row of a wave's transposition buffer (16-byte aligned rows)
constexpr int kRank2Share = 2 * 9 * kTrPitch;   // floats of LDS per wave: the rows of hi and of lo pieces, and in their place its results
constexpr int kLinearF16x2 = 2;                 // the mode (mg_get_linear_mode) in which fp16 pieces may take the place of fp32 products
typedef float floatx4 __attribute__((ext_vector_type(4)));

// The packed weight of a chan: per chunk of 64 channels
//   fp32      [label][tq][lane = 16 kk + j][tr] = Y2[j][label chan + 64 chunk + 16 kk + 4 tq + tr], zero for j >= dim_d
// then of all chunks
//   pieces    [24 fragments][lane][8], scaled: labels (0, 1) and (2, 3), four steps t each, hi and lo: element 2 c + i is label 2 p + i at
//             channel 16 kk + 4 t + c; label 4, four steps, twice: (hi, hi) and (lo, lo) of channel 16 kk + 4 t + c
// and the 16 inverse scales of the outputs (mark_weight where an output's weights are not finite).
constexpr int kRank2Fp32 = 5 * 4 * 64 * 4, kRank2Pieces = 24 * 64 * 8;
inline size_t rank2_weight_bytes(int chan) {
    return (size_t)ceil_div(chan, 64) * (kRank2Fp32 * sizeof(float) + kRank2Pieces * sizeof(_Float16)) + 16 * sizeof(float);
}

// max over the wave of non-negative values (NaN counts as zero), valid in lane 63: six cross-lane VALU operations (shifts within
// rows of 16 lanes, then row broadcasts), no LDS traffic.  Such floats are ordered as their bits are, and an integer maximum
// takes the moved operand directly: as fmaxf each step was a move, a shift, a canonicalisation and the maximum.
__device__ __forceinline__ float wave_max_nonneg_last_lane(float v) {
    auto step = [](unsigned x, auto ctrl, auto row_mask) {
        const unsigned moved = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, decltype(row_mask)::value, 0xf, false);
        return x > moved ? x : moved;
    };
    unsigned x = __float_as_uint(fmaxf(v, 0.f));
    x = step(x, std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});   // row_shr:1
    x = step(x, std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});   // row_shr:2
    x = step(x, std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});   // row_shr:4
    x = step(x, std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});   // row_shr:8
    x = step(x, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});   // row_bcast:15
    x = step(x, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});   // row_bcast:31
    return __uint_as_float(x);
}

// Whether pieces under one scale can carry the wave's values: none beyond them, and each of the nine components, a sum of its own, no
// smaller than 2^-12 of the largest value, so that the last bit of a low piece is below 2^-26 of the component's largest.  It is
// enough that one lane has all nine of that size, which takes one comparison.  bound: the largest |s2| (NaN left out), the same in every lane.
__device__ __forceinline__ bool pieces_fit(const float (&s2)[45], float& bound) {
    float most = 0.f, least = __builtin_inff();
#pragma unroll
    for (int k = 0; k < 9; k++) {
        float v = 0.f;
#pragma unroll
        for (int lab = 0; lab < 5; lab++) v = fmaxf(v, fabsf(s2[5 * k + lab]));
        most = fmaxf(most, v);
        least = fminf(least, v);
    }
    bound = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(wave_max_nonneg_last_lane(most)), kWave - 1));
    return !beyond_split(bound) && __any(least >= 0x1p-12f * bound);
}

// a value that is uniform over the wave and never written while the kernel runs, as a scalar load
template <typename V>
__device__ __forceinline__ V scalar_at(const V* p) {
    return *(const __attribute__((address_space(4))) V*)(unsigned long)p;
}

// the wave's 9 x 16 sums over its chunk: lane (j = lane % 16, kk = lane / 16), register q: comp 4 kk + q of output j
__device__ __forceinline__ floatx4 rank2_sums_fp32(const float (&s2)[45], float* tr, int chunk, const float* __restrict__ y2_packed) {
    const int lane = threadIdx.x & (kWave - 1), ci = lane & 15, kk = lane >> 4;
    const float* a_src = tr + (ci < 9 ? ci : ci - 7) * kTrPitch + 16 * kk;
    const float4* yb = reinterpret_cast<const float4*>(y2_packed) + (long)chunk * 5 * 4 * 64 + lane;
    floatx4 d0 = {0.f, 0.f, 0.f, 0.f}, d1 = d0, d2 = d0, d3 = d0;   // four chains: a matrix instruction does not wait for the last one
    float4 b[2][4];
#pragma unroll
    for (int tq = 0; tq < 4; tq++) b[0][tq] = yb[tq * 64];
#pragma unroll
    for (int lab = 0; lab < 5; lab++) {
#pragma unroll
        for (int k = 0; k < 9; k++) tr[k * kTrPitch + lane] = s2[k * 5 + lab];
        wave_lds_fence();
        float4 a[4];
#pragma unroll
        for (int tq = 0; tq < 4; tq++) a[tq] = *reinterpret_cast<const float4*>(a_src + 4 * tq);
        if (lab < 4) {
#pragma unroll
            for (int tq = 0; tq < 4; tq++) b[(lab + 1) & 1][tq] = yb[((lab + 1) * 4 + tq) * 64];
        }
#pragma unroll
        for (int tq = 0; tq < 4; tq++) {
            d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tq].x, b[lab & 1][tq].x, d0, 0, 0, 0);
            d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tq].y, b[lab & 1][tq].y, d1, 0, 0, 0);
            d2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tq].z, b[lab & 1][tq].z, d2, 0, 0, 0);
            d3 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tq].w, b[lab & 1][tq].w, d3, 0, 0, 0);
        }
        wave_lds_fence();                                       // the rows are rewritten by the next label
    }
    return (d0 + d1) + (d2 + d3);
}
// pieces: those of the wave's chunk, of a pair of labels asked for before its rows are written (from memory, not LDS)
__device__ __forceinline__ floatx4 rank2_sums_f16x2(const float (&s2)[45], float scale, float* tr, const _Float16* __restrict__ pieces) {
    const int lane = threadIdx.x & (kWave - 1), ci = lane & 15, kk = lane >> 4;
    float* const hi_rows = tr;
    float* const lo_rows = tr + 9 * kTrPitch;
    const int from = (ci < 9 ? ci : ci - 7) * kTrPitch + 16 * kk;
    const halfx8* w = reinterpret_cast<const halfx8*>(pieces) + lane;
    floatx4 small[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, large[2] = {small[0], small[0]};
#pragma unroll
    for (int p = 0; p < 2; p++) {
        halfx8 ahead[8];
#pragma unroll
        for (int t = 0; t < 8; t++) ahead[t] = w[(8 * p + t) * 64];
#pragma unroll
        for (int k = 0; k < 9; k++) {
            halfx2 hi, lo;
            split_pair(s2[k * 5 + 2 * p], s2[k * 5 + 2 * p + 1], scale, scale, hi, lo);
            hi_rows[k * kTrPitch + lane] = __builtin_bit_cast(float, hi);
            lo_rows[k * kTrPitch + lane] = __builtin_bit_cast(float, lo);
        }
        wave_lds_fence();
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const halfx8 xh = *reinterpret_cast<const halfx8*>(hi_rows + from + 4 * t), xl = *reinterpret_cast<const halfx8*>(lo_rows + from + 4 * t);
            const halfx8 wh = ahead[2 * t], wl = ahead[2 * t + 1];
            small[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wh, small[0], 0, 0, 0);
            small[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wl, small[1], 0, 0, 0);
            large[t & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, wh, large[t & 1], 0, 0, 0);
            small[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, wl, small[0], 0, 0, 0);
        }
        wave_lds_fence();                                       // the rows are rewritten
    }
    halfx8 ahead[8];
#pragma unroll
    for (int t = 0; t < 8; t++) ahead[t] = w[(16 + t) * 64];
#pragma unroll
    for (int k = 0; k < 9; k++) {
        const float v = s2[k * 5 + 4];
        const _Float16 hi = (_Float16)(v * scale);
        hi_rows[k * kTrPitch + lane] = __builtin_bit_cast(float, halfx2{hi, (_Float16)__builtin_fmaf(v, scale, -(float)hi)});
    }
    wave_lds_fence();
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const halfx8 x = *reinterpret_cast<const halfx8*>(hi_rows + from + 4 * t);
        const halfx8 twice = ahead[2 * t], low = ahead[2 * t + 1];
        small[t & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, low, small[t & 1], 0, 0, 0);
        large[t & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, twice, large[t & 1], 0, 0, 0);
    }
    wave_lds_fence();
    return (small[0] + small[1]) + (large[0] + large[1]);
}

// The workgroup's waves meet over their LDS: unlike __syncthreads, without waiting for stores to memory
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Called by all four waves of the workgroup (it holds two barriers); valid = false: a wave without an item, whose s2
// must be zeros.  split: pieces may take the place of fp32 products.
// lds: kRank2Share floats for each wave, SHARE apart, 16-byte aligned.  out: this wave's node, (dim_d, 9);
// accumulate: the result is added to what out holds.
template <int SHARE = kRank2Share>
__device__ __forceinline__ void rank2_linear_of_node_sums(const float (&s2)[45], bool split, float* lds, int chunk, int chunks, bool valid,
                                                          const float* __restrict__ y2_packed, int dim_d,
                                                          float* __restrict__ out, bool accumulate = false) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    float* const tr = lds + wave * SHARE;
    const int ci = lane & 15, kk = lane >> 4;
    const _Float16* const pieces = reinterpret_cast<const _Float16*>(y2_packed + chunks * kRank2Fp32);
    const float iw = reinterpret_cast<const float*>(pieces + chunks * kRank2Pieces)[ci];
    floatx4 d;
    float bound;
    if (pieces_fit(s2, bound) && split && !__any(iw != iw)) {
        float inv;
        const float scale = pow2_scale(bound, &inv);
        d = rank2_sums_f16x2(s2, scale, tr, pieces + chunk * kRank2Pieces) * inv * iw;
    } else {
        d = rank2_sums_fp32(s2, tr, chunk, y2_packed);
    }
    // accumulator register q of lane l: comp 4 (l / 16) + q, output l % 16
#pragma unroll
    for (int q = 0; q < 4; q++) tr[(4 * kk + q) * 16 + ci] = d[q];
    lds_barrier();
    if (chunk == 0 && valid) {                                  // the first wave of a node adds up its chunks
        for (int idx = lane; idx < dim_d * 9; idx += kWave) {
            const int j = idx / 9, i = idx - 9 * j;
            float sum = 0.f;
            for (int wv = 0; wv < chunks; wv++) sum += tr[wv * SHARE + i * 16 + j];
            out[idx] = accumulate ? out[idx] + sum : sum;
        }
    }
    lds_barrier();                                            // before the workgroup's next use of lds
}

inline bool rank2_fusable(int chan, int dim_d) {
    const int chunks = chan / 64;
    return chan > 0 && chan % 64 == 0 && (chunks == 1 || chunks == 2 || chunks == 4) && dim_d >= 1 && dim_d <= 16;
}

}  // namespace mg
