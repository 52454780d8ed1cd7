// fp32-class GEMM on the fp16 matrix cores with two-piece operand splitting ("f16x2").
//
// Every fp32 operand is scaled by a per-row power of two (exact) and split into two fp16
// pieces, v = hi + lo with hi = RNE16(v) and lo = RNE16(v - hi): 11 + 11 significand bits, so
// |v - hi - lo| <= 2^-22 |v|.  A product is assembled from three piece products
//     a*b ~= a_lo*b_hi + a_hi*b_lo + a_hi*b_hi            (dropped: a_lo*b_lo <= 2^-22 |a||b|)
// accumulated in fp32 by v_mfma_f32_32x32x16_f16: half the matrix work of a three-piece bf16
// split, at an error of a few fp32 ulps per product (the rounding of an fp32 dot product of
// length K is of the same size).  The power-of-two scales put the largest element of an x row
// (a W row) into [2^14, 2^15), which removes fp16's narrow exponent range from the picture:
// an element e of a row with scaled maximum M carries an error of max(2^-22 |e|, 2^-25), i.e.
// the result is normwise as accurate as the fp32 dot product whenever M >= 1, and the scales
// are undone exactly in the epilogue.  Rows with an infinity or beyond 2^96, and columns whose weights hold an infinity or NaN,
// are summed in fp32 by the epilogue (row_in_fp32): the results are those of fp32 arithmetic there too.  The row maxima of x come from the kernel that produced
// x (this kernel's own epilogue can emit them for its output) or from row_absmax_kernel.
//
// Kernel shape (row streaming): a workgroup of WAVES waves owns a tile of 32 WAVES rows x 32 NI
// columns; wave w owns rows [32 w, 32 w + 32) of the tile and ALL its columns.
//   * x never touches LDS: a lane loads the 16 consecutive floats of ITS row that it will feed to
//     the matrix core (lane = row + 32 g holds k = 32 c + 16 g .. + 16 of chunk c: 64 contiguous
//     bytes, four 16-byte loads), two chunks ahead, and splits them in registers.  Every row is
//     loaded and split exactly once per tile, nothing about x is tied to a barrier, and the LDS
//     carries only W.
//   * W planes (already fp16, packed in fragment order: f16x2.hpp) go global -> registers -> LDS, double buffered, K
//     chunk 32, one barrier per chunk.
//   * the k order inside a chunk is a permutation (MFMA step s takes k = 16 g + 8 s .. + 8 from
//     lane group g); W is read from LDS with the same permutation, so the products pair up.
//   * loads are never predicated (rows past the end are clamped to the last row, whose
//     accumulators are simply not written): a loop body without branches lets every load stay in
//     flight until the chunk that needs it.  W (L2 resident, needed one chunk later) is requested
//     before x (HBM, needed two chunks later), because loads return in order.
//   * the epilogue runs once per tile with nothing to overlap it, so its instruction count is
//     what matters: one row pointer, row scale and bounds check per accumulator row, column
//     offsets as immediates, activation and accumulate chosen at compile time.
// v_mfma_f32_32x32x16_f16 layout: A[m][k]: lane = m + 32*(k/8), 8 consecutive k per lane;
// B[k][n] likewise; D[m][n]: n = lane%32, m = 8*(q/4) + 4*(lane/32) + q%4 for register q.
#include "common.hpp"
#include "f16x2.hpp"
#include <type_traits>

namespace mg {
namespace {

__device__ __forceinline__ float activate(float v, int act) {
    if (act == 1) return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    if (act == 2) return v > 0.f ? v : 0.1f * v;
    return v;
}

template <int ACT>
__device__ __forceinline__ float activate_c(float v) {
    // SiLU through the hardware exp2 and reciprocal (about 1 ulp each): far inside the fp32 tolerance
    if constexpr (ACT == 1) return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    if constexpr (ACT == 2) return v > 0.f ? v : 0.1f * v;
    return v;
}

// behind the inverse scales: per block of 32 output rows whether one of them is marked (mark_weight)
template <typename F>
__device__ __forceinline__ auto* marked_blocks(F* inv_scale, int O_pad) {
    return reinterpret_cast<std::conditional_t<std::is_const_v<F>, const int, int>*>(inv_scale + O_pad);
}

// Weight planes in fragment order (f16x2.hpp) + 1/scale per row: a workgroup takes a block of 32 output rows (rows past O
// are zeros), a thread pieces of 8 k of one row, kept in registers between the row maximum (LDS, max of the bit patterns
// of |w|: any order gives the same) and the split.  One pass over W for I <= kPackRegs * 256.  I_w <= I: columns of W, the
// others are zeros.  Rows with an infinity or NaN are scaled by their finite entries and marked.
constexpr int kPackThreads = 1024, kPackRegs = 4;
// A launch takes up to kPackJobs weights (a training step packs every weight of a layer and its transpose anew: one launch of
// 10 us per MLP instead of six of 6).
constexpr int kPackJobs = 8;
struct PackJob {
    const float* W;
    long so, si;
    int I_w, I, O, O_pad, first_block;
    _Float16* planes;
};
struct PackJobs {
    PackJob job[kPackJobs];
    int count;
};
__global__ void __launch_bounds__(kPackThreads) pack_weight_f16x2_kernel(const PackJobs jobs) {
    __shared__ unsigned row_max[32], row_odd[32];
    const int tid = threadIdx.x;
    int which = 0;
    while (which + 1 < jobs.count && (int)blockIdx.x >= jobs.job[which + 1].first_block) which++;     // (uniform)
    const PackJob& job = jobs.job[which];
    const float* __restrict__ W = job.W;
    const long so = job.so, si = job.si;
    const int I_w = job.I_w, I = job.I, O = job.O, O_pad = job.O_pad, block = blockIdx.x - job.first_block;
    _Float16* __restrict__ planes = job.planes;
    float* __restrict__ inv_scale = reinterpret_cast<float*>(planes + 2L * O_pad * I);
    const int m = tid & 31;
    const long o = 32L * block + m;
    const int pieces = I >> 3;                            // per row; thread t takes pieces t / 32, + 32, ...
    const long total = (long)O_pad * I;
    if (tid < 32) row_max[tid] = row_odd[tid] = 0;
    __syncthreads();
    const float* row = W + (o < O ? o : 0) * so;
    auto load = [&](float (&v)[8], int piece) {
        const float* p = row + (long)(8 * piece) * si;
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = o < O && 8 * piece + j < I_w ? p[j * si] : 0.f;
    };
    float keep[kPackRegs][8];
    unsigned mx = 0;
    bool odd = false;
    auto largest = [&](float v) {
        const unsigned b = __float_as_uint(fabsf(v));
        if (b >= 0x7f800000u) odd = true;
        else mx = b > mx ? b : mx;
    };
#pragma unroll
    for (int u = 0; u < kPackRegs; u++) {
        const int piece = (tid >> 5) + 32 * u;
        if (piece < pieces) {
            load(keep[u], piece);
#pragma unroll
            for (int j = 0; j < 8; j++) largest(keep[u][j]);
        }
    }
    for (int piece = (tid >> 5) + 32 * kPackRegs; piece < pieces; piece += 32) {
        float v[8];
        load(v, piece);
#pragma unroll
        for (int j = 0; j < 8; j++) largest(v[j]);
    }
    atomicMax(&row_max[m], mx);
    if (odd) row_odd[m] = 1;
    __syncthreads();
    float inv;
    const float s = pow2_scale(__uint_as_float(row_max[m]), &inv);
    if (tid < 32) {
        inv_scale[o] = row_odd[m] ? mark_weight(inv) : inv;
        const int marked = __any(row_odd[m]);
        if (tid == 0) marked_blocks(inv_scale, O_pad)[block] = marked;
    }
    auto store = [&](const float (&v)[8], int piece) {
        halfx8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float x = v[j] * s;
            const _Float16 h = (_Float16)x;
            hi[j] = h;
            lo[j] = (_Float16)(x - (float)h);
        }
        const long at = packed_index(o, 8 * piece, I);
        *reinterpret_cast<halfx8*>(planes + at) = hi;
        *reinterpret_cast<halfx8*>(planes + total + at) = lo;
    };
#pragma unroll
    for (int u = 0; u < kPackRegs; u++) {
        const int piece = (tid >> 5) + 32 * u;
        if (piece < pieces) store(keep[u], piece);
    }
    for (int piece = (tid >> 5) + 32 * kPackRegs; piece < pieces; piece += 32) {
        float v[8];
        load(v, piece);
        store(v, piece);
    }
}

// out[r] = max_i |x[r, i]|; a wave per row, 16-byte loads when the row length allows
__global__ void __launch_bounds__(256) row_absmax_kernel(const float* __restrict__ x, long R, int I,
                                                         float* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const long n_waves = ((long)gridDim.x * blockDim.x) >> 6;
    for (long r = wave; r < R; r += n_waves) {
        const float* row = x + r * I;
        float m = 0.f;
        if ((I & 3) == 0) {
            for (int i = lane * 4; i < I; i += 256) {
                const float4 v = *reinterpret_cast<const float4*>(row + i);
                m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
            }
        } else {
            for (int i = lane; i < I; i += 64) m = fmaxf(m, fabsf(row[i]));
        }
        for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
        if (lane == 0) out[r] = m;
    }
}


// x (rows, K, T) in the reference's tensor layout (channel, then components) -> xt (rows * T, K_pad): one plain
// GEMM row per (row, component), channels zero-padded to K_pad, and the maximum of |xt| per output row.
// A thread writes four consecutive channels of one output row; the K_pad / 4 threads of a row are neighbours.
__global__ void __launch_bounds__(256) components_to_rows_kernel(const float* __restrict__ x, long rows, int K, int T,
                                                                 int K_pad, float* __restrict__ xt,
                                                                 float* __restrict__ rowmax) {
    const int per_row = K_pad / 4;                            // 8, 16, ...: a power of two <= 64
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long out_row = idx / per_row;
    const int k0 = (int)(idx - out_row * per_row) * 4;
    const bool live = out_row < rows * T;
    const long r = live ? out_row / T : 0;
    const int t = live ? (int)(out_row - r * T) : 0;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = (live && k0 + j < K) ? x[(r * K + k0 + j) * T + t] : 0.f;
    if (live) *reinterpret_cast<float4*>(xt + out_row * K_pad + k0) = make_float4(v[0], v[1], v[2], v[3]);
    float mx = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
    for (int d = 1; d < per_row; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
    if (live && k0 == 0) rowmax[out_row] = mx;
}

// a barrier that orders LDS only: __syncthreads() would also wait for the stores to memory
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// (waves per SIMD that the registers of the narrow tiles are held to: the epilogue's rare paths would cost one otherwise)
constexpr int streaming_waves(int waves, int ni) { return waves == 4 && ni <= 2 ? 6 - ni : 1; }

// APART: the two small products of a step have an accumulator of their own, so that the large sum is rounded once per 16 k and not
// three times (apart_of)
template <int WAVES, int NI, bool APART>
__global__ void __launch_bounds__(64 * WAVES, APART ? 1 : streaming_waves(WAVES, NI))
linear_rows_f16x2_kernel(const _Float16* __restrict__ Wp, const float* __restrict__ w_inv, const float* __restrict__ X, long x_stride,
                         const float* __restrict__ xmax, int xmax_parts, long xmax_stride, long xmax_div, long R, int I,
                         int O, int O_pad, const float* __restrict__ bias, int act, int accumulate,
                         float* __restrict__ Y, float* __restrict__ ymax, int tiles_n, long tiles_total, int out_T,
                         float bound_mul, float bound_add, long bias_rows) {
    constexpr int TM = 32 * WAVES, TN = 32 * NI, THREADS = 64 * WAVES;
    constexpr int kPlaneW = TN * 64, kBufW = 2 * kPlaneW;
    constexpr int kPieces = 8 * TN;                          // 16-byte pieces of W per chunk (2 planes x TN rows x 4)
    constexpr int kPer = (kPieces + THREADS - 1) / THREADS;  // per thread
    // component rows of nine leave through LDS in this tile only (epilogue_runs): 32 columns of the tile's rows
    constexpr bool kRuns = WAVES == 4 && NI == 2;
    constexpr int kStage = kRuns ? 4 * 32 * (TM + 2 * 9) : 0;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kBufW > kStage ? 2 * kBufW : kStage];
    __shared__ float inv_sx[TM];

    const long bid = blockIdx.x;
    const long per_xcd = (tiles_total + 7) / 8;
    const long logical = (bid % 8) * per_xcd + bid / 8;
    if (logical >= tiles_total) return;
    const long tile_m = logical / tiles_n;
    const int tile_n = (int)(logical - tile_m * tiles_n);

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int m = lane & 31, g = lane >> 5;
    const long r0 = tile_m * TM;
    const int n0 = tile_n * TN;
    const long plane_elems = (long)O_pad * I;

    floatx16 acc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ni++)
#pragma unroll
        for (int q = 0; q < 16; q++) acc[ni][q] = 0.f;
    floatx16 apart[APART ? NI : 1];
    if constexpr (APART)
#pragma unroll
        for (int ni = 0; ni < NI; ni++) apart[ni] = acc[ni];

    // this lane's row of x (clamped past the end: those accumulators are never written)
    const long my_row = r0 + wave * 32 + m;
    const long ld_row = my_row < R ? my_row : R - 1;
    const float* xrow = X + ld_row * x_stride + 16 * g;
    float sx;
    bool odd;                                                // this wave has rows (columns: below) that the pieces cannot carry
    {
        float amax = 0.f;
        const float* xm = xmax + (ld_row / xmax_div) * xmax_stride;
        for (int p = 0; p < xmax_parts; p++) amax = fmaxf(amax, xm[p]);
        amax = fmaf(amax, bound_mul, bound_add);             // the caller's bound of |x| is bound_mul * xmax + bound_add
        float inv;
        sx = pow2_scale(amax, &inv);
        if (g == 0) inv_sx[wave * 32 + m] = beyond_split(amax) ? __builtin_nanf("") : inv;
        odd = __any(beyond_split(amax));
    }
    const _Float16* wsrc[kPer];
    int wdst[kPer];
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        int q = tid + THREADS * j;
        if (q >= kPieces) q = kPieces - 1;                    // surplus threads repeat the last piece
        const int plane = q / (4 * TN), i = q % (4 * TN);
        wsrc[j] = Wp + plane * plane_elems + packed_piece(n0, i, I);
        wdst[j] = plane * kPlaneW + 16 * i;
    }
    const int k_last = I - kCK;

    struct ARegs { float4 v[4]; };
    struct WRegs { halfx8 v[kPer]; };
    auto load_a = [&](ARegs& a, int k0) {
        k0 = k0 < I ? k0 : k_last;                            // surplus loads of the last trips are never used
#pragma unroll
        for (int j = 0; j < 4; j++) a.v[j] = *reinterpret_cast<const float4*>(xrow + k0 + 4 * j);
    };
    auto load_w = [&](WRegs& w, int k0) {
        k0 = k0 < I ? k0 : k_last;
#pragma unroll
        for (int j = 0; j < kPer; j++) w.v[j] = *reinterpret_cast<const halfx8*>(wsrc[j] + 32L * k0);
    };
    auto store_w = [&](const WRegs& w, unsigned char* buf) {
#pragma unroll
        for (int j = 0; j < kPer; j++) *reinterpret_cast<halfx8*>(buf + wdst[j]) = w.v[j];
    };
    const int b_off = 16 * lane;
    auto compute = [&](const ARegs& a, const unsigned char* buf, float scale) {
        halfx8 ah[2], al[2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const HalfSplit4 p0 = split(a.v[2 * s], scale), p1 = split(a.v[2 * s + 1], scale);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                ah[s][i] = p0.hi[i]; ah[s][4 + i] = p1.hi[i];
                al[s][i] = p0.lo[i]; al[s][4 + i] = p1.lo[i];
            }
        }
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                const halfx8 bh = *reinterpret_cast<const halfx8*>(buf + b_off + 2048 * ni + 1024 * s);
                const halfx8 bl = *reinterpret_cast<const halfx8*>(buf + kPlaneW + b_off + 2048 * ni + 1024 * s);
                // small terms first
                floatx16& small = APART ? apart[APART ? ni : 0] : acc[ni];
                small = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[s], bh, small, 0, 0, 0);
                small = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[s], bl, small, 0, 0, 0);
                acc[ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[s], bh, acc[ni], 0, 0, 0);
            }
        order_chunk<NI>();
    };

    unsigned char* buf0 = lds;
    unsigned char* buf1 = lds + kBufW;
    ARegs a0, a1;
    WRegs w;
    load_w(w, 0);
    load_a(a0, 0);
    int marked = 0;
#pragma unroll
    for (int ni = 0; ni < NI; ni++) marked |= marked_blocks(w_inv, O_pad)[n0 / 32 + ni];      // (scalar loads)
    store_w(w, buf0);
    load_w(w, kCK);
    load_a(a1, kCK);
    asm volatile("" : "+s"(marked));                         // (arrived by here, where W was waited for, and not in the epilogue)
    const bool odd_cols = marked != 0;
    odd |= odd_cols;
    __syncthreads();
    // chunks in pairs (even chunk: a0 / buf0, odd chunk: a1 / buf1); with an odd chunk count the
    // surplus chunk (a clamped reload of the last one) is scaled by zero instead of being branched
    // around, which keeps the loop body straight-line
    for (int k0 = 0; k0 < I; k0 += 2 * kCK) {
        compute(a0, buf0, sx);
        store_w(w, buf1);
        __builtin_amdgcn_sched_barrier(0);     // keep this issue order: the compiler would hoist the loads
        load_w(w, k0 + 2 * kCK);
        __builtin_amdgcn_sched_barrier(0);
        load_a(a0, k0 + 2 * kCK);
        __syncthreads();
        compute(a1, buf1, k0 + kCK < I ? sx : 0.f);
        store_w(w, buf0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(w, k0 + 3 * kCK);
        __builtin_amdgcn_sched_barrier(0);
        load_a(a1, k0 + 3 * kCK);
        __syncthreads();
    }
    if constexpr (APART)
#pragma unroll
        for (int ni = 0; ni < NI; ni++) acc[ni] += apart[ni];

    if constexpr (kRuns)
        if (out_T == 9) {                                    // (epilogue_runs has barriers: all waves go the same way)
            bool row = false;
            for (int r = lane; r < TM; r += 64) { const float isx = inv_sx[r]; row |= isx != isx; }
            odd |= __any(row);
        }
    const bool full_cols = n0 + TN <= O && !odd;
    // ---- fast path, plain rows: y (rows, O)
    auto epilogue_rows = [&](auto act_tag, auto acc_tag, auto some_tag) {
        constexpr int kAct = decltype(act_tag)::value;
        constexpr bool kAccumulate = decltype(acc_tag)::value;
        constexpr bool kSomeBias = decltype(some_tag)::value;      // only rows below bias_rows have the bias
        float bv[NI], iw[NI];
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            bv[ni] = bias ? bias[n0 + ni * 32 + m] : 0.f;
            iw[ni] = w_inv[n0 + ni * 32 + m];
        }
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int rl = wave * 32 + 8 * (q / 4) + 4 * g + (q % 4);
            const long r = r0 + rl;
            if (r < R) {
                float* yrow = Y + r * O + n0 + m;
                const float isx = inv_sx[rl];
                float mx = 0.f;
#pragma unroll
                for (int ni = 0; ni < NI; ni++) {
                    const float b = kSomeBias && r >= bias_rows ? 0.f : bv[ni];
                    float v = activate_c<kAct>(acc[ni][q] * isx * iw[ni] + b);
                    if constexpr (kAccumulate) v += yrow[ni * 32];
                    yrow[ni * 32] = v;
                    mx = fmaxf(mx, fabsf(v));
                }
                if (ymax) {
#pragma unroll
                    for (int d = 1; d < 32; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
                    if (m == 0) ymax[r * tiles_n + tile_n] = mx;
                }
            }
        }
    };
    // ---- fast path, rows are (row, comp) pairs and y is stored (row, chan, comp): no bias, no activation
    auto epilogue_comps = [&](auto t_tag) {
        constexpr int T = decltype(t_tag)::value;
        float iw[NI];
#pragma unroll
        for (int ni = 0; ni < NI; ni++) iw[ni] = w_inv[n0 + ni * 32 + m];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int rl = wave * 32 + 8 * (q / 4) + 4 * g + (q % 4);
            const long r = r0 + rl;
            if (r < R) {
                const long row = r / T;
                float* yp = Y + (row * O + n0 + m) * T + (r - row * T);
                const float isx = inv_sx[rl];
#pragma unroll
                for (int ni = 0; ni < NI; ni++) {
                    float v = acc[ni][q] * isx * iw[ni];
                    if (accumulate) v += yp[ni * 32 * T];
                    yp[ni * 32 * T] = v;
                }
            }
        }
    };
    // The same for nine components: a lane's values lie 36 bytes from its neighbours', so that every store of a wave would
    // write four bytes here and there of dozens of lines.  32 columns at a time are put in order in LDS (the W buffers are done
    // with) and leave in runs.  73 728 rows x 32 -> 256: 65 us stored directly, whatever the tile; 40 us in runs from this
    // tile, 62 from 256 x 256 (one workgroup per CU, whose passes wait for each other).  With three components direct stores
    // are faster: 15.6 against 17.7 us for 24 576 x 64 -> 256.
    auto epilogue_runs = [&](auto t_tag) {
        constexpr int T = decltype(t_tag)::value;
        float* stage = reinterpret_cast<float*>(lds);
        const long row_lo = r0 / T;
        const int first = (int)(r0 - row_lo * T);                    // the tile's rows are first .. first + TM - 1 of row_lo's
        const int count = ((first + TM - 1) / T + 1) * (32 * T);
        const int end = R - r0 < TM ? first + (int)(R - r0) : first + TM;
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            const float iw = w_inv[n0 + ni * 32 + m];
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int rl = wave * 32 + 8 * (q / 4) + 4 * g + (q % 4), row = (first + rl) / T;
                stage[row * (32 * T) + m * T + (first + rl - row * T)] = acc[ni][q] * inv_sx[rl] * iw;
            }
            lds_barrier();
            for (int e = tid; e < count; e += THREADS) {
                const int row = e / (32 * T), w = e - row * (32 * T), rr = row * T + w % T;
                if (rr >= first && rr < end) {
                    float* yp = Y + ((row_lo + row) * O + n0 + ni * 32) * T + w;
                    *yp = accumulate ? stage[e] + *yp : stage[e];
                }
            }
            lds_barrier();
        }
    };
    if (full_cols && out_T == 1) {
        constexpr std::integral_constant<int, 0> kNone{};
        constexpr std::integral_constant<int, 1> kSilu{};
        constexpr std::integral_constant<int, 2> kLeaky{};
        if (bias_rows < R) epilogue_rows(kNone, std::false_type{}, std::true_type{});   // (no activation, not accumulated)
        else if (accumulate) {
            if (act == 1) epilogue_rows(kSilu, std::true_type{}, std::false_type{});
            else if (act == 2) epilogue_rows(kLeaky, std::true_type{}, std::false_type{});
            else epilogue_rows(kNone, std::true_type{}, std::false_type{});
        } else {
            if (act == 1) epilogue_rows(kSilu, std::false_type{}, std::false_type{});
            else if (act == 2) epilogue_rows(kLeaky, std::false_type{}, std::false_type{});
            else epilogue_rows(kNone, std::false_type{}, std::false_type{});
        }
        return;
    }
    if (full_cols && act == 0 && bias == nullptr && out_T == 3) { epilogue_comps(std::integral_constant<int, 3>{}); return; }
    if (full_cols && act == 0 && bias == nullptr && out_T == 9) {
        if constexpr (kRuns) epilogue_runs(std::integral_constant<int, 9>{});
        else epilogue_comps(std::integral_constant<int, 9>{});
        return;
    }

    // ---- general path: partial column tiles, components with bias / activation, rows or columns beyond the pieces
    float rmax[16];
#pragma unroll
    for (int q = 0; q < 16; q++) rmax[q] = 0.f;
#pragma unroll
    for (int ni = 0; ni < NI; ni++) {
        const int n = n0 + ni * 32 + m;
        if (n >= O) continue;
        const float bv = bias ? bias[n] : 0.f;
        const float iw = w_inv[n];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int rl = wave * 32 + 8 * (q / 4) + 4 * g + (q % 4);
            const long r = r0 + rl;
            const float isx = inv_sx[rl];
            if (r < R && isx == isx && iw == iw) {
                const long row = r / out_T;
                const long addr = (row * O + n) * out_T + (r - row * out_T);
                float v = activate(acc[ni][q] * isx * iw + (r < bias_rows ? bv : 0.f), act);
                if (accumulate) v += Y[addr];
                Y[addr] = v;
                rmax[q] = fmaxf(rmax[q], fabsf(v));
            }
        }
    }
    if (odd) {
#pragma unroll 1
        for (int k = 0; k < 16 * NI; k++) {
            const int n = n0 + (k >> 4) * 32 + m, q = k & 15, rl = wave * 32 + 8 * (q / 4) + 4 * g + (q % 4);
            const long r = r0 + rl;
            if (n >= O || r >= R) continue;
            const float isx = inv_sx[rl], iw = w_inv[n];
            if (isx == isx && iw == iw) continue;
            const long row = r / out_T, addr = (row * O + n) * out_T + (r - row * out_T);
            const float v = activate(row_in_fp32(X + r * x_stride, Wp, plane_elems, n, I, iw) + (bias && r < bias_rows ? bias[n] : 0.f), act);
            Y[addr] = accumulate ? v + Y[addr] : v;
        }
    }
    if (ymax) {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const float isx = inv_sx[wave * 32 + 8 * (q / 4) + 4 * g + (q % 4)];
            float mx = odd_cols || isx != isx ? __builtin_inff() : rmax[q];        // (no bound: the next layer takes the row in fp32)
#pragma unroll
            for (int d = 1; d < 32; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
            const long r = r0 + wave * 32 + 8 * (q / 4) + 4 * g + (q % 4);
            if (m == 0 && r < R) ymax[r * tiles_n + tile_n] = mx;
        }
    }
}

// Few rows, few columns, long K (the output linears of one small system: 18 432 rows, K = 1280, 16 columns): the
// row-streaming kernel above gives such a problem a handful of workgroups that each walk 40 chunks one barrier at a
// time, about 1.3 us per chunk of load and LDS latency with nothing to overlap it.  Here a workgroup owns a tile of
// 32 rows x 32 NI columns and its WAVES waves split K: wave w takes chunks w, w + WAVES, ... with private
// accumulators, reads its W fragments straight from the packed planes (L2 resident; no LDS, no barrier in the loop),
// and the partial tiles are summed through LDS in wave order, so the result does not depend on timing.
// With a workgroup to a CU the reductions of several chunks a wave (ONE false) are bound by the chain bound of the row -> first chunk ->
// .. -> old value of y, and by the cache's lookups: the bounds (four parts at once) and the first chunk are requested together, the old
// values before the barrier, and a chunk of x is read eight lanes to a row, 128 bytes at a time, and handed to the lanes that multiply it
// through this wave's own part of LDS (a lane to a row, 16 bytes at a time, asks for 32 lines with every load, four times over).  6144 rows
// x 1280 -> 64 onto y 17.0 -> 14.3 us, 900 rows 12.1 -> 10.1; 9216 x 1280 -> 16 19.5 -> 16.2; 2048 x 768 -> 256 onto y 12.9 -> 11.4;
// 512 -> 512 at 337 rows 8.1 -> 7.6, at 3072 19.4 -> 18.0.  A wave with one chunk at most (ONE) has nothing to gain from either and keeps
// the straight order (2048 x 256 -> 256 8.0 against 8.3 us, 6144 x 64 -> 256 9.2 against 9.8).
template <int WAVES, int NI, bool ONE>
__global__ void __launch_bounds__(64 * WAVES)
linear_rows_splitk_f16x2_kernel(const _Float16* __restrict__ Wp, const float* __restrict__ w_inv,
                                const float* __restrict__ X, long x_stride, const float* __restrict__ xmax,
                                float* __restrict__ xmax_out, int xmax_parts,
                                long xmax_stride, long xmax_div, long R, int I, int O, int O_pad,
                                const float* __restrict__ bias, int act, int accumulate, float* __restrict__ Y,
                                float* __restrict__ ymax, int tiles_n, int out_T, float bound_mul, float bound_add,
                                long bias_rows) {
    constexpr int TN = 32 * NI, THREADS = 64 * WAVES;
    constexpr int kPitch = TN + 1;                            // floats per row of a partial tile
    constexpr int kTile = 32 * kPitch > 1024 ? 32 * kPitch : 1024;
    __shared__ __attribute__((aligned(16))) float partial[WAVES][kTile];
    __shared__ float inv_sx[32], wave_max[WAVES][32];

    // (choose_splitk: at most 49 152 rows, R O in 21 bits)
    const unsigned tile_m = blockIdx.x / (unsigned)tiles_n;
    const int tile_n = (int)(blockIdx.x - tile_m * tiles_n);
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int m = lane & 31, g = lane >> 5;
    const unsigned r0 = tile_m * 32;
    const int n0 = tile_n * TN;
    const long plane_elems = (long)O_pad * I;

    const unsigned my_row = r0 + m, n_rows = (unsigned)R;
    const unsigned ld_row = my_row < n_rows ? my_row : n_rows - 1;
    // Piece q (16 bytes) of a chunk's row r lies at q ^ (r / 2) % 8: 16 lanes read 16 different places of the 256 bytes that LDS delivers at once.
    float* const stage = partial[wave];
    unsigned piece_row[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const unsigned r = r0 + 8 * j + lane / 8;
        piece_row[j] = r < n_rows ? r : n_rows - 1;
    }
    float sx;
    auto set_scale = [&](float amax) {
        float inv;
        sx = pow2_scale(amax, &inv);
        if (wave == 0 && g == 0) inv_sx[m] = beyond_split(amax) ? __builtin_nanf("") : inv;
    };
    // lane's fragment of W for MFMA step s, column block ni: row n0 + 32 ni + m, k = k0 + 16 g + 8 s .. + 8
    const _Float16* wrow = Wp + packed_piece(n0, lane, I);

    floatx16 acc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ni++)
#pragma unroll
        for (int q = 0; q < 16; q++) acc[ni][q] = 0.f;

    struct Chunk {
        float4 a[4];
        halfx8 wh[NI][2], wl[NI][2];
    };
    auto load_pieces = [&](float4 (&a)[4], int k0) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            a[j] = ONE ? *reinterpret_cast<const float4*>(X + (long)ld_row * x_stride + k0 + 16 * g + 4 * j)
                       : *reinterpret_cast<const float4*>(X + (long)piece_row[j] * x_stride + k0 + 4 * (lane & 7));
    };
    auto load = [&](Chunk& c, int k0) {
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                c.wh[ni][s2] = *reinterpret_cast<const halfx8*>(wrow + (long)ni * 32 * I + 32L * k0 + 512 * s2);
                c.wl[ni][s2] = *reinterpret_cast<const halfx8*>(wrow + plane_elems + (long)ni * 32 * I + 32L * k0 + 512 * s2);
            }
        load_pieces(c.a, k0);
    };
    auto hand_over = [&](Chunk& c) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = 8 * j + lane / 8;
            *reinterpret_cast<float4*>(stage + 32 * r + 4 * ((lane & 7) ^ (r / 2 & 7))) = c.a[j];
        }
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; j++) c.a[j] = *reinterpret_cast<const float4*>(stage + 32 * m + 4 * ((4 * g + j) ^ (m / 2 & 7)));
        wave_lds_fence();                                     // (the place is written again)
    };
    auto compute = [&](const Chunk& c) {
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) {
            const HalfSplit4 p0 = split(c.a[2 * s2], sx), p1 = split(c.a[2 * s2 + 1], sx);
            halfx8 ah, al;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                ah[i] = p0.hi[i]; ah[4 + i] = p1.hi[i];
                al[i] = p0.lo[i]; al[4 + i] = p1.lo[i];
            }
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                acc[ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, c.wh[ni][s2], acc[ni], 0, 0, 0);
                acc[ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, c.wl[ni][s2], acc[ni], 0, 0, 0);
                acc[ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, c.wh[ni][s2], acc[ni], 0, 0, 0);
            }
        }
    };
    const int chunks = I / kCK;
    Chunk cur, nxt;
    const float* const xm = xmax ? xmax + (long)(ld_row / (unsigned)xmax_div) * xmax_stride : nullptr;
    if constexpr (ONE) {
        if (xmax) {                                           // (uniform)
            float amax = 0.f;
            for (int p = 0; p < xmax_parts; p++) amax = fmaxf(amax, xm[p]);
            set_scale(fmaf(amax, bound_mul, bound_add));
        }
        if (wave < chunks) load(cur, wave * kCK);
    } else {
        float part[4] = {0.f, 0.f, 0.f, 0.f};
        if (xmax) {
#pragma unroll
            for (int p = 0; p < 4; p++) part[p] = xm[p < xmax_parts ? p : 0];
        }
        if (wave < chunks) load(cur, wave * kCK);
        if (xmax) {
            float amax = fmaxf(fmaxf(fmaxf(0.f, part[0]), fmaxf(part[1], part[2])), part[3]);
            for (int p = 4; p < xmax_parts; p++) amax = fmaxf(amax, xm[p]);
            set_scale(fmaf(amax, bound_mul, bound_add));
        }
    }
    if (!xmax) {                                              // the rows' own maxima, as row_absmax_kernel takes them
        float mx[4] = {0.f, 0.f, 0.f, 0.f};
        auto largest = [&](const float4 (&a)[4]) {
#pragma unroll
            for (int j = 0; j < 4; j++) mx[j] = fmaxf(fmaxf(mx[j], fmaxf(fabsf(a[j].x), fabsf(a[j].y))), fmaxf(fabsf(a[j].z), fabsf(a[j].w)));
        };
        if (wave < chunks) largest(cur.a);
        for (int c = wave + WAVES; c < chunks; c += WAVES) {
            float4 a[4];
            load_pieces(a, c * kCK);
            largest(a);
        }
        if constexpr (ONE) {
            mx[0] = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
            mx[0] = fmaxf(mx[0], __shfl_xor(mx[0], 32));
            if (g == 0) wave_max[wave][m] = mx[0];
        } else
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) mx[j] = fmaxf(mx[j], __shfl_xor(mx[j], d));
            if ((lane & 7) == 0) wave_max[wave][8 * j + lane / 8] = mx[j];
        }
        __syncthreads();
        float amax = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) amax = fmaxf(amax, wave_max[w][m]);
        if (tile_n == 0 && wave == 0 && g == 0 && my_row < n_rows) xmax_out[my_row] = amax;
        set_scale(amax);
    }
    if constexpr (ONE) {
        if (wave < chunks) compute(cur);
    } else
    for (int c = wave; c < chunks; c += WAVES) {
        const bool more = c + WAVES < chunks;
        if (more) load(nxt, (c + WAVES) * kCK);
        hand_over(cur);
        compute(cur);
        if (more) cur = nxt;
    }
    // a thread finishes the elements e = tid, tid + THREADS, ...: row e / TN, column e % TN (the lanes of a row are neighbours, so its
    // maximum is a shuffle away)
    constexpr int kPer = 32 * TN / THREADS;
    static_assert(32 * TN % THREADS == 0 && THREADS % TN == 0 && TN <= 64, "whole rows per pass, a row within a wave");
    const int my_n = n0 + tid % TN;
    float iw = 0.f, my_bias = 0.f, was[kPer];
    unsigned at[kPer];
    auto request = [&] {
        if (my_n < O) {
            iw = w_inv[my_n];
            my_bias = bias ? bias[my_n] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < kPer; j++) {
            const unsigned r = r0 + (tid + THREADS * j) / TN;
            at[j] = r * O + my_n;
            if (out_T != 1) {                                 // (uniform)
                const unsigned row = r / (unsigned)out_T;
                at[j] = (row * O + my_n) * out_T + (r - row * out_T);
            }
            was[j] = accumulate && r < n_rows && my_n < O ? Y[at[j]] : 0.f;
        }
    };
    if (!ONE) request();
    // partial tiles -> LDS; accumulator register q of block ni is row 8 (q / 4) + 4 g + q % 4, column 32 ni + m
#pragma unroll
    for (int ni = 0; ni < NI; ni++)
#pragma unroll
        for (int q = 0; q < 16; q++)
            partial[wave][(8 * (q / 4) + 4 * g + (q % 4)) * kPitch + 32 * ni + m] = acc[ni][q];
    __syncthreads();
    if (ONE) request();
    bool odd = false;                                         // an element of a row or column that the pieces cannot carry
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int e = tid + THREADS * j;
        const int rl = e / TN, col = e - rl * TN;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) sum += partial[w][rl * kPitch + col];
        const unsigned r = r0 + rl;
        float v = 0.f;
        if (r < n_rows && my_n < O) {
            const float isx = inv_sx[rl];
            if (isx == isx && iw == iw) {
                v = activate(sum * isx * iw + ((long)r < bias_rows ? my_bias : 0.f), act);
                if (accumulate) v += was[j];
                Y[at[j]] = v;
            } else {
                odd = true;
                v = __builtin_inff();                         // (no bound: the next layer takes the row in fp32)
            }
        }
        if (ymax) {
            float mx = fabsf(v);
#pragma unroll
            for (int d = 1; d < TN; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
            if (col == 0 && r < n_rows) ymax[r * tiles_n + tile_n] = mx;
        }
    }
    if (odd) {
#pragma unroll 1
        for (int j = 0; j < kPer; j++) {
            const int rl = (tid + THREADS * j) / TN;
            const unsigned r = r0 + rl;
            if (r >= n_rows || my_n >= O) continue;
            const float isx = inv_sx[rl];
            if (isx == isx && iw == iw) continue;
            const unsigned row = r / (unsigned)out_T, addr = (row * O + my_n) * out_T + (r - row * out_T);
            const float v = activate(row_in_fp32(X + (long)r * x_stride, Wp, plane_elems, my_n, I, iw) + ((long)r < bias_rows ? my_bias : 0.f), act);
            Y[addr] = accumulate ? v + Y[addr] : v;
        }
    }
}

inline int o_pad_of(int dim_out) { return (dim_out + 255) / 256 * 256; }
inline int i_pad_of(int dim_in) { return (dim_in + 31) / 32 * 32; }

// The split-K kernel is for problems whose row-streaming tiles would leave most of the chip idle while a few workgroups walk
// K one barrier at a time.  The rule is the measured crossover (R = 337 .. 49152, K = 128 .. 1280, O = 64 .. 512) in units
// of 32 x 32 output blocks:
//   up to 256 blocks      one block per workgroup, eight waves on K     512 -> 512 at 337 rows  5.3 us (streaming 12.7)
//   up to 512 blocks      two column blocks per workgroup               512 -> 512 at 1024 rows 7.4 us (13.4)
//   up to 1536 blocks     two column blocks, four waves on K            512 -> 512 at 3072 rows 16.8 us (22.1)
//   more                  row streaming (W read once per 128 or 256 rows): 512 -> 512 at 4096 rows 22.5 us (23.0 split)
// K below 256 has fewer than eight chunks: four waves.  At most 64 column tiles (row maxima per tile).
struct SplitK {
    int waves, ni;       // waves = 0: the row-streaming kernel
};
inline SplitK choose_splitk(long R, int I, int O) {
    const long blocks = ceil_div(R, 32) * ceil_div(O, 32);
    if (blocks > 1536 || O > 2048) return SplitK{0, 0};
    if (I < 256) return SplitK{4, blocks <= 896 || O <= 32 ? 1 : 2};
    if (O <= 32) return SplitK{8, 1};
    if (blocks <= 256) return SplitK{8, 1};
    return SplitK{blocks <= 512 ? 8 : 4, 2};
}

struct Shape {
    int ni;      // 32-column blocks per tile
    int waves;   // waves per workgroup (32 rows each)
};
inline Shape choose_shape(long R, int I, int O) {
    Shape s;
    s.ni = O <= 32 ? 1 : (O <= 64 ? 2 : (O <= 128 ? 4 : 8));
    // column tiles that divide O: a partly filled tile takes the slow, bounds-checked epilogue (O = 384 with
    // 256-column tiles ran 4 times slower than with 128-column tiles)
    if (O % 32 == 0)
        while (s.ni > 1 && O % (32 * s.ni) != 0 && ceil_div(O, 16 * s.ni) <= 64) s.ni >>= 1;
    const long tiles_m = ceil_div(R, 256);
    if (tiles_m * ceil_div(O, 32 * s.ni) >= 1024 || O % 32 != 0) {
        s.waves = 8;                                       // many tiles: the widest tile, one 8-wave workgroup per CU
        return s;
    }
    // Few tiles (node-sized problems, the edges of one small system).  The chip takes 256 workgroups of 8 waves at
    // a time, and a workgroup's time was measured (33 392 rows, K = 256 .. 768, all tile widths) as about
    // 5 us + chunks x (1 + ni / 4) us: among the column tiles that divide O take the one with the least
    // (rounds of 256 workgroups) x (time per workgroup); ties go to the wider tile, which re-reads x less often.
    const long chunks = ceil_div(I, 32);
    long best = -1;
    for (int ni = s.ni; ni >= 1; ni >>= 1) {
        if (O % (32 * ni) != 0 || ceil_div(O, 32 * ni) > 64) continue;   // at most 64 column tiles (row maxima per tile)
        const long cost = ceil_div(tiles_m * (O / (32 * ni)), 256) * (20 + chunks * (4 + ni));
        if (best < 0 || cost < best) { best = cost; s.ni = ni; }
    }
    // fewer than two chips' worth of 8-wave workgroups: 4-wave workgroups (128 rows) double their number; not with
    // 256-column tiles, whose 4-wave variant keeps one wave per SIMD
    s.waves = (tiles_m * ceil_div(O, 32 * s.ni) >= 512 || (s.ni == 8 && tiles_m >= 32)) ? 8 : 4;
    return s;
}

// A reduction of more than 512 in tiles of at most 128 columns keeps the small products apart, in a second set of accumulators.
// K = 1280 (the five rank-1 or rank-2 products of a layer side by side, in inference) against float64: 2.7e-7 of the
// result's 2-norm; in one accumulator 4.3e-7, five linears of K = 256 and a sum 3.5e-7, in fp32 6.5e-7.  Sequential
// reductions take such a tile for every width; others keep the 256-column tile, which has no registers for the second set.
inline bool apart_of(int I, int ni) { return I > 512 && ni <= 4; }
inline Shape choose_sequential(long R, int I, int O) {
    Shape s = choose_shape(R, I, O);
    if (I > 512 && s.ni == 8) s.ni = 4;
    return s;
}

template <int WAVES, int NI, bool APART = false>
int launch(const _Float16* planes, const float* w_inv, const float* x, long x_stride, const float* xmax, int parts, long stride,
           long div, long rows, int I, int O, int O_pad, const float* bias, int act, int accumulate, float* y,
           float* ymax, int out_T, float bound_mul, float bound_add, long bias_rows, hipStream_t st) {
    const long tiles_m = ceil_div(rows, 32 * WAVES);
    const int tiles_n = (int)ceil_div(O, 32 * NI);
    const long total = tiles_m * tiles_n;
    const long grid = ceil_div(total, 8) * 8;
    MG_REQUIRE(grid <= 0x7fffffffL, "mg_tensor_linear_f16x2: grid too large (rows=%ld dim_out=%d)", rows, O);
    hipLaunchKernelGGL((linear_rows_f16x2_kernel<WAVES, NI, APART>), dim3((unsigned)grid), dim3(64 * WAVES), 0, st, planes,
                       w_inv, x, x_stride, xmax, parts, stride, div, rows, I, O, O_pad, bias, act, accumulate, y, ymax, tiles_n,
                       total, out_T, bound_mul, bound_add, bias_rows);
    return check_launch("mg_tensor_linear_f16x2");
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_linear_f16x2_packed_weight_bytes(int dim_in, int dim_out, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && dim_in >= 0 && dim_out >= 0, "mg_linear_f16x2_packed_weight_bytes: bad argument");
    const size_t o_pad = (size_t)o_pad_of(dim_out);
    *bytes = 2 * o_pad * (size_t)i_pad_of(dim_in) * sizeof(_Float16) + o_pad * sizeof(float) + o_pad / 32 * sizeof(int);
    return MG_OK;
}

int mg_linear_f16x2_pack_weights(const mg_f16x2_weight* weights, int count, mg_stream_t stream) {
    MG_REQUIRE(count >= 0 && (weights || count == 0), "mg_linear_f16x2_pack_weights: bad argument");
    PackJobs jobs;
    int blocks = 0;
    jobs.count = 0;
    auto flush = [&]() -> int {
        if (jobs.count == 0) return MG_OK;
        hipLaunchKernelGGL(pack_weight_f16x2_kernel, dim3((unsigned)blocks), dim3(kPackThreads), 0, (hipStream_t)stream, jobs);
        blocks = 0;
        jobs.count = 0;
        return check_launch("mg_linear_f16x2_pack_weight");
    };
    for (int k = 0; k < count; k++) {
        const mg_f16x2_weight& w = weights[k];
        MG_REQUIRE(w.dim_in >= 0 && w.dim_out >= 0 && w.dim_pad >= w.dim_in, "mg_linear_f16x2_pack_weight: bad size");
        if (w.dim_in == 0 || w.dim_out == 0) continue;
        MG_REQUIRE(w.W && w.packed && aligned16(w.packed), "mg_linear_f16x2_pack_weight: null or unaligned pointer");
        MG_REQUIRE(w.dim_pad % 32 == 0, "mg_linear_f16x2_pack_weight: dim_pad must be a multiple of 32");
        const int O_pad = o_pad_of(w.dim_out);
        jobs.job[jobs.count++] = PackJob{w.W, w.stride_o, w.stride_i, w.dim_in, w.dim_pad, w.dim_out, O_pad, blocks,
                                         static_cast<_Float16*>(w.packed)};
        blocks += O_pad / 32;
        if (jobs.count == kPackJobs)
            if (int code = flush()) return code;
    }
    return flush();
}

int mg_linear_f16x2_pack_weight_padded(const float* W, long w_stride_o, long w_stride_i, int dim_in, int dim_out, int dim_pad,
                                       void* packed, mg_stream_t stream) {
    const mg_f16x2_weight w{W, w_stride_o, w_stride_i, dim_in, dim_out, dim_pad, packed};
    return mg_linear_f16x2_pack_weights(&w, 1, stream);
}

int mg_linear_f16x2_pack_weight(const float* W, long w_stride_o, long w_stride_i, int dim_in, int dim_out,
                                void* packed, mg_stream_t stream) {
    MG_REQUIRE(dim_in % 8 == 0, "mg_linear_f16x2_pack_weight: dim_in must be a multiple of 8");
    return mg_linear_f16x2_pack_weight_padded(W, w_stride_o, w_stride_i, dim_in, dim_out, i_pad_of(dim_in), packed, stream);
}

int mg_row_absmax(const float* x, long rows, int dim, float* out, mg_stream_t stream) {
    MG_REQUIRE(rows >= 0 && dim >= 0, "mg_row_absmax: negative size");
    if (rows == 0) return MG_OK;
    MG_REQUIRE(out && (x || dim == 0), "mg_row_absmax: null pointer");
    MG_REQUIRE(dim % 4 != 0 || aligned16(x), "mg_row_absmax: x must be 16-byte aligned");
    long blocks = ceil_div(rows, 4);
    if (blocks > 256L * 32) blocks = 256L * 32;
    hipLaunchKernelGGL(row_absmax_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, x, rows, dim, out);
    return check_launch("mg_row_absmax");
}

int mg_components_to_rows(const float* x, long rows, int dim, int comps, int dim_pad, float* xt, float* rowmax,
                          mg_stream_t stream) {
    MG_REQUIRE(rows >= 0 && dim > 0 && comps > 0, "mg_components_to_rows: bad size");
    MG_REQUIRE(dim_pad >= dim && dim_pad % 32 == 0 && dim_pad <= 256 && (dim_pad & (dim_pad - 1)) == 0,
               "mg_components_to_rows: dim_pad must be a power of two in 32..256, at least dim (got %d for %d)", dim_pad, dim);
    if (rows == 0) return MG_OK;
    MG_REQUIRE(x && xt && rowmax && aligned16(xt), "mg_components_to_rows: null or unaligned pointer");
    const long threads = rows * comps * (dim_pad / 4);
    hipLaunchKernelGGL(components_to_rows_kernel, dim3((unsigned)ceil_div(threads, 256)), dim3(256), 0,
                       (hipStream_t)stream, x, rows, dim, comps, dim_pad, xt, rowmax);
    return check_launch("mg_components_to_rows");
}

int mg_tensor_linear_f16x2_rowmax_parts_sequential(long rows, int dim_in, int dim_out) {
    return (int)ceil_div(dim_out, 32 * choose_sequential(rows, dim_in, dim_out).ni);
}

int mg_tensor_linear_f16x2_rowmax_parts(long rows, int dim_in, int dim_out) {
    const SplitK sk = choose_splitk(rows, dim_in, dim_out);
    if (sk.waves) return (int)ceil_div(dim_out, 32 * sk.ni);
    return (int)ceil_div(dim_out, 32 * choose_shape(rows, dim_in, dim_out).ni);
}

int mg_tensor_linear_f16x2_splits_k(long rows, int dim_in, int dim_out) {
    return choose_splitk(rows, dim_in, dim_out).waves != 0;
}

int mg_tensor_linear_f16x2(const void* packed_W, const float* x, const float* x_rowmax, int x_rowmax_parts,
                           long x_rowmax_stride, long x_rows_per_bound, long rows, int dim_in, int dim_out,
                           const float* bias, int act, int accumulate, int out_comps, float* y, float* y_rowmax,
                           mg_stream_t stream) {
    return mg_tensor_linear_f16x2_scaled_bound(packed_W, x, x_rowmax, x_rowmax_parts, x_rowmax_stride, x_rows_per_bound,
                                               rows, dim_in, dim_out, bias, act, accumulate, out_comps, y, y_rowmax, 1.0f,
                                               0.0f, stream);
}

int mg_tensor_linear_f16x2_scaled_bound(const void* packed_W, const float* x, const float* x_rowmax, int x_rowmax_parts,
                                        long x_rowmax_stride, long x_rows_per_bound, long rows, int dim_in, int dim_out,
                                        const float* bias, int act, int accumulate, int out_comps, float* y,
                                        float* y_rowmax, float bound_mul, float bound_add, mg_stream_t stream) {
    const mg_f16x2_linear a{packed_W,  x,    x_rowmax, x_rowmax_parts, x_rowmax_stride, x_rows_per_bound, bound_mul, bound_add,
                            rows,      dim_in, dim_out, bias,          rows,            act,              accumulate, out_comps,
                            0,         y,    y_rowmax};
    return mg_tensor_linear_f16x2_run(&a, stream);
}

int mg_tensor_linear_f16x2_run(const mg_f16x2_linear* args, mg_stream_t stream) {
    MG_REQUIRE(args != nullptr, "mg_tensor_linear_f16x2: null pointer");
    return mg_tensor_linear_f16x2_run_strided(args, args->dim_in, stream);
}

// x_rowmax_out: where the row maxima of |x| go that this call is to find itself, or null with args->x_rowmax given.
// A reduction that is split over the waves of a workgroup has whole rows in it and finds them on the way: 337 rows 128 -> 512
// 5.1 us, and 4.8 behind a launch of 3.0 for them.
static int run_strided(const mg_f16x2_linear* args, long x_stride, float* x_rowmax_out, mg_stream_t stream) {
    MG_REQUIRE(args != nullptr, "mg_tensor_linear_f16x2: null pointer");
    mg_f16x2_linear a = *args;
    if (x_rowmax_out) {
        a.x_rowmax = x_rowmax_out;
        a.x_rowmax_parts = 1;
        a.x_rowmax_stride = a.x_rows_per_bound = 1;
        a.bound_mul = 1.f;
        a.bound_add = 0.f;
        MG_REQUIRE(x_stride == a.dim_in, "mg_tensor_linear_f16x2: row maxima are found of contiguous rows");
    }
    MG_REQUIRE(x_stride >= a.dim_in && x_stride % 4 == 0, "mg_tensor_linear_f16x2: x_stride must be a multiple of 4, at least dim_in");
    MG_REQUIRE(a.bound_mul >= 0.f && a.bound_add >= 0.f && a.bound_mul == a.bound_mul && a.bound_add == a.bound_add,
               "mg_tensor_linear_f16x2: the bound's factor and offset must be non-negative numbers");
    MG_REQUIRE(a.rows >= 0 && a.dim_in > 0 && a.dim_out >= 0, "mg_tensor_linear_f16x2: bad size");
    MG_REQUIRE(a.dim_in % 32 == 0, "mg_tensor_linear_f16x2: dim_in must be a multiple of 32");
    MG_REQUIRE(a.act >= 0 && a.act <= 2, "mg_tensor_linear_f16x2: unknown activation %d", a.act);
    MG_REQUIRE(a.out_comps == 1 || a.out_comps == 3 || a.out_comps == 9, "mg_tensor_linear_f16x2: out_comps must be 1, 3 or 9");
    MG_REQUIRE(a.x_rowmax_parts >= 1 && a.x_rowmax_parts <= 64, "mg_tensor_linear_f16x2: x_rowmax_parts must be in 1..64");
    MG_REQUIRE(a.x_rowmax_stride == 0 || a.x_rowmax_stride >= a.x_rowmax_parts,
               "mg_tensor_linear_f16x2: x_rowmax_stride must be 0 (one bound for all rows) or >= x_rowmax_parts");
    MG_REQUIRE(a.x_rows_per_bound >= 1, "mg_tensor_linear_f16x2: x_rows_per_bound must be positive");
    MG_REQUIRE(a.y_rowmax == nullptr || a.out_comps == 1, "mg_tensor_linear_f16x2: y_rowmax needs out_comps == 1");
    MG_REQUIRE(a.bias_rows >= a.rows || (a.bias_rows >= 0 && a.act == 0 && !a.accumulate && a.out_comps == 1),
               "mg_tensor_linear_f16x2: a bias for some rows only goes with plain rows, no activation, not accumulated");
    if (a.rows == 0 || a.dim_out == 0) return MG_OK;
    MG_REQUIRE(a.packed_W && a.x && a.y && a.x_rowmax && aligned16(a.x) && aligned16(a.packed_W),
               "mg_tensor_linear_f16x2: null or unaligned pointer");
    const int O_pad = o_pad_of(a.dim_out);
    const _Float16* planes = static_cast<const _Float16*>(a.packed_W);
    const float* w_inv = reinterpret_cast<const float*>(planes + 2L * O_pad * a.dim_in);
    hipStream_t st = (hipStream_t)stream;
    const SplitK sk = a.sequential ? SplitK{0, 0} : choose_splitk(a.rows, a.dim_in, a.dim_out);
    if (sk.waves) {
        const int tiles_n = (int)ceil_div(a.dim_out, 32 * sk.ni);
        const long tiles = ceil_div(a.rows, 32) * tiles_n;
        const float* given = x_rowmax_out ? nullptr : a.x_rowmax;
        MG_REQUIRE(tiles <= 0x7fffffffL, "mg_tensor_linear_f16x2: grid too large (rows=%ld)", a.rows);
#define MG_SPLITK(WV, N)                                                                                                   \
    if (sk.waves == WV && sk.ni == N)                                                                                      \
        hipLaunchKernelGGL((a.dim_in <= kCK * WV ? linear_rows_splitk_f16x2_kernel<WV, N, true>                            \
                                                 : linear_rows_splitk_f16x2_kernel<WV, N, false>),                         \
                           dim3((unsigned)tiles), dim3(64 * WV), 0, st, planes, w_inv, a.x, x_stride, given, x_rowmax_out,  \
                           a.x_rowmax_parts, a.x_rowmax_stride, a.x_rows_per_bound < 0x7fffffffL ? a.x_rows_per_bound : 0x7fffffffL, \
                           a.rows, a.dim_in, a.dim_out, O_pad, a.bias, a.act, a.accumulate, a.y, a.y_rowmax, tiles_n, a.out_comps, \
                           a.bound_mul, a.bound_add, a.bias_rows)
        MG_SPLITK(8, 1);
        MG_SPLITK(8, 2);
        MG_SPLITK(4, 1);
        MG_SPLITK(4, 2);
#undef MG_SPLITK
        return check_launch("mg_tensor_linear_f16x2");
    }
    if (x_rowmax_out)
        if (int code = mg_row_absmax(a.x, a.rows, a.dim_in, x_rowmax_out, stream)) return code;
    Shape sh = a.sequential ? choose_sequential(a.rows, a.dim_in, a.dim_out) : choose_shape(a.rows, a.dim_in, a.dim_out);
    // nine components and a short reduction: bound by the stores, in runs out of this tile (18 432 x 32 -> 256 17 against 19 us,
    // 73 728 rows 40 against 65); longer reductions keep the tile that re-reads x least
    if (a.out_comps == 9 && a.dim_in <= 64 && a.dim_out % 64 == 0 && a.act == 0 && a.bias == nullptr) sh = Shape{2, 4};
#define MG_F16X2_LAUNCH(WV, ...)                                                                                           \
    return launch<WV, __VA_ARGS__>(planes, w_inv, a.x, x_stride, a.x_rowmax, a.x_rowmax_parts, a.x_rowmax_stride, a.x_rows_per_bound, a.rows, \
                         a.dim_in, a.dim_out, O_pad, a.bias, a.act, a.accumulate, a.y, a.y_rowmax, a.out_comps,            \
                         a.bound_mul, a.bound_add, a.bias_rows, st)
    if (apart_of(a.dim_in, sh.ni)) {
        if (sh.waves == 8) {
            if (sh.ni == 1) MG_F16X2_LAUNCH(8, 1, true);
            if (sh.ni == 2) MG_F16X2_LAUNCH(8, 2, true);
            MG_F16X2_LAUNCH(8, 4, true);
        }
        if (sh.ni == 1) MG_F16X2_LAUNCH(4, 1, true);
        if (sh.ni == 2) MG_F16X2_LAUNCH(4, 2, true);
        MG_F16X2_LAUNCH(4, 4, true);
    }
    if (sh.waves == 8) {
        if (sh.ni == 1) MG_F16X2_LAUNCH(8, 1);
        if (sh.ni == 2) MG_F16X2_LAUNCH(8, 2);
        if (sh.ni == 4) MG_F16X2_LAUNCH(8, 4);
        MG_F16X2_LAUNCH(8, 8);
    }
    if (sh.ni == 1) MG_F16X2_LAUNCH(4, 1);
    if (sh.ni == 2) MG_F16X2_LAUNCH(4, 2);
    if (sh.ni == 4) MG_F16X2_LAUNCH(4, 4);
    MG_F16X2_LAUNCH(4, 8);
#undef MG_F16X2_LAUNCH
}

int mg_tensor_linear_f16x2_run_strided(const mg_f16x2_linear* args, long x_stride, mg_stream_t stream) {
    return run_strided(args, x_stride, nullptr, stream);
}

int mg_tensor_linear_f16x2_run_unbounded(const mg_f16x2_linear* args, float* x_rowmax_out, mg_stream_t stream) {
    MG_REQUIRE(args != nullptr && (x_rowmax_out || args->rows == 0), "mg_tensor_linear_f16x2_run_unbounded: null pointer");
    if (args->rows == 0) return MG_OK;
    return run_strided(args, args->dim_in, x_rowmax_out, stream);
}

}  // extern "C"
