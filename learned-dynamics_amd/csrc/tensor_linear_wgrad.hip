// Weight gradient of the channel-mixing linear:
//   dW[o, i] = sum_{r, t} dy[r, o, t] x[r, i, t]
// A GEMM whose reduction dimension (rows x components) is the long one, so the
// rows are split over workgroups (split-K); each workgroup reduces its slice
// for one 64x64 tile of dW in registers and writes it to its own plane of a
// workspace; a second kernel adds the planes in slice order.  No atomics: the
// result does not depend on the order in which workgroups finish.
// Plain rows (no tensor components) go through the matrix cores.  mg_tensor_linear_wgrad uses the fp32 ones:
// v_mfma_f32_32x32x2_f32 takes dy and x exactly as they lie in memory (for the reduction index r, lanes 0..31 supply
// 32 consecutive columns of row r and lanes 32..63 those of row r + 1), products and sums are fp32, nothing is
// rounded to a shorter format.  mg_tensor_linear_wgrad_f16x2 uses the fp16 ones with two-piece operands (three times
// the rate at an error of a few fp32 ulps of sum |dy| |x|) and also sums the columns of dy, the bias gradient.
// Training-side helper: not on the inference hot path.
#include "common.hpp"
#include "f16x2.hpp"
#include <type_traits>

namespace mg {
namespace {

constexpr int kTile = 64;      // dW tile edge
constexpr int kRowsPerStep = 4;

__global__ void __launch_bounds__(256) zero_f32_kernel(float* __restrict__ p, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0.f;
}

template <int T>
__global__ void __launch_bounds__(256) wgrad_kernel(const float* __restrict__ dy, const float* __restrict__ x, long R,
                                                    int I, int O, long rows_per_block, float* __restrict__ part) {
    __shared__ float dys[kRowsPerStep * T][kTile + 1];
    __shared__ float xs[kRowsPerStep * T][kTile + 1];
    const int o0 = blockIdx.x * kTile, i0 = blockIdx.y * kTile;
    const long r_lo = (long)blockIdx.z * rows_per_block;
    const long r_hi = r_lo + rows_per_block < R ? r_lo + rows_per_block : R;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;   // tx -> i, ty -> o
    float acc[4][4] = {};
    for (long r = r_lo; r < r_hi; r += kRowsPerStep) {
        __syncthreads();
        for (int idx = threadIdx.x; idx < kRowsPerStep * kTile * T; idx += 256) {
            const int rr = idx / (kTile * T), rem = idx % (kTile * T), c = rem / T, t = rem % T;
            const bool row_ok = r + rr < r_hi;
            dys[rr * T + t][c] = (row_ok && o0 + c < O) ? dy[((r + rr) * O + o0 + c) * T + t] : 0.f;
            xs[rr * T + t][c] = (row_ok && i0 + c < I) ? x[((r + rr) * I + i0 + c) * T + t] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kRowsPerStep * T; k++) {
            float a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) { a[q] = dys[k][ty + 16 * q]; b[q] = xs[k][tx + 16 * q]; }
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int q = 0; q < 4; q++) acc[p][q] += a[p] * b[q];
        }
    }
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int o = o0 + ty + 16 * p, i = i0 + tx + 16 * q;
            if (o < O && i < I) part[((long)blockIdx.z * O + o) * I + i] = acc[p][q];
        }
}

// Plain rows on the matrix cores.  A workgroup of 4 waves owns a 128 x 128 tile of dW over its slice of the rows;
// wave w owns the 64 x 64 quarter (w / 2, w % 2) as 2 x 2 accumulators of 32 x 32.  Columns past the matrix and rows
// past the slice are read from a clamped address and replaced by zero.
constexpr int kMTile = 128;
constexpr int kMRows = 8;       // rows per trip of the loop: 4 matrix steps of 2 rows

__global__ void __launch_bounds__(256) wgrad_mfma_kernel(const float* __restrict__ dy, const float* __restrict__ x,
                                                         long R, int I, int O, long rows_per_block,
                                                         float* __restrict__ part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 31, kk = lane >> 5;
    const int o_base = blockIdx.x * kMTile + (wave >> 1) * 64, i_base = blockIdx.y * kMTile + (wave & 1) * 64;
    const long r_lo = (long)blockIdx.z * rows_per_block;
    const long r_hi = r_lo + rows_per_block < R ? r_lo + rows_per_block : R;
    // this lane's two columns of dy and of x (clamped; `live` says whether the column exists)
    int oc[2], ic[2];
    bool o_live[2], i_live[2];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int o = o_base + 32 * p + m, i = i_base + 32 * p + m;
        o_live[p] = o < O; i_live[p] = i < I;
        oc[p] = o_live[p] ? o : O - 1;
        ic[p] = i_live[p] ? i : I - 1;
    }
    floatx16 acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int k = 0; k < 16; k++) acc[p][q][k] = 0.f;

    // the operands of the next trip are requested before the matrix instructions of this one
    float a[2][kMRows / 2][2], b[2][kMRows / 2][2];
    auto fetch = [&](float (&aa)[kMRows / 2][2], float (&bb)[kMRows / 2][2], long r) {
#pragma unroll
        for (int s = 0; s < kMRows / 2; s++) {
            const long row = r + 2 * s + kk;
            const bool row_live = row < r_hi;
            const long rc = row_live ? row : r_hi - 1;
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const float va = dy[rc * O + oc[p]], vb = x[rc * I + ic[p]];
                aa[s][p] = (row_live && o_live[p]) ? va : 0.f;
                bb[s][p] = (row_live && i_live[p]) ? vb : 0.f;
            }
        }
    };
    auto multiply = [&](const float (&aa)[kMRows / 2][2], const float (&bb)[kMRows / 2][2]) {
#pragma unroll
        for (int s = 0; s < kMRows / 2; s++)
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int q = 0; q < 2; q++)
                    acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x2f32(aa[s][p], bb[s][q], acc[p][q], 0, 0, 0);
    };
    fetch(a[0], b[0], r_lo);
    for (long r = r_lo; r < r_hi; r += 2 * kMRows) {
        fetch(a[1], b[1], r + kMRows);                 // (past the slice: clamped addresses, zeros)
        multiply(a[0], b[0]);
        fetch(a[0], b[0], r + 2 * kMRows);
        multiply(a[1], b[1]);
    }
    // D[o][i]: i = lane % 32, o = 8 (k / 4) + 4 (lane / 32) + k % 4 for register k
    float* plane = part + (long)blockIdx.z * O * I;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int i = i_base + 32 * q + m;
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const int o = o_base + 32 * p + 8 * (k / 4) + 4 * kk + (k % 4);
                if (o < O && i < I) plane[(long)o * I + i] = acc[p][q][k];
            }
        }
}

// The same with the operands staged through LDS, for dimensions that are multiples of 4: a lane of the kernel above
// loads one float per matrix operand, and the vector memory front end spends as long on such a load as on a 16-byte
// one (about a cycle per lane), four times the matrix time of the tile.  Here the workgroup loads 16 rows x 128
// columns of dy and of x with 16-byte loads into LDS (rows padded to 160 floats: the two rows that the two halves of a
// wave read lie 32 banks apart) and the lanes pick their operands out of LDS; the next 16 rows are on their way while
// the current ones are multiplied.
constexpr int kSRows = 16, kSPitch = 160;
__global__ void __launch_bounds__(256) wgrad_mfma_lds_kernel(const float* __restrict__ dy, const float* __restrict__ x,
                                                             long R, int I, int O, long rows_per_block,
                                                             float* __restrict__ part) {
    __shared__ __attribute__((aligned(16))) float dys[2][kSRows * kSPitch];
    __shared__ __attribute__((aligned(16))) float xs[2][kSRows * kSPitch];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 31, kk = lane >> 5;
    const int o_tile = blockIdx.x * kMTile, i_tile = blockIdx.y * kMTile;
    const int o_wave = (wave >> 1) * 64, i_wave = (wave & 1) * 64;
    const long r_lo = (long)blockIdx.z * rows_per_block;
    const long r_hi = r_lo + rows_per_block < R ? r_lo + rows_per_block : R;

    // staging: thread -> two 16-byte pieces per operand (piece = row * 32 + column quad)
    int st_row[2], st_col[2];
    bool o_ok[2], i_ok[2];
    const float* dy_src[2];
    const float* x_src[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int piece = threadIdx.x + 256 * u;
        st_row[u] = piece >> 5;
        st_col[u] = (piece & 31) * 4;
        o_ok[u] = o_tile + st_col[u] < O;
        i_ok[u] = i_tile + st_col[u] < I;
        dy_src[u] = dy + (o_ok[u] ? o_tile + st_col[u] : 0);
        x_src[u] = x + (i_ok[u] ? i_tile + st_col[u] : 0);
    }
    float4 ra[2], rb[2];
    auto fetch = [&](long r) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const long row = r + st_row[u];
            const long rc = row < r_hi ? row : r_hi - 1;            // (clamped: replaced by zeros when stored)
            ra[u] = *reinterpret_cast<const float4*>(dy_src[u] + rc * O);
            rb[u] = *reinterpret_cast<const float4*>(x_src[u] + rc * I);
        }
    };
    auto store = [&](long r, int buf) {
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const bool row_ok = r + st_row[u] < r_hi;
            *reinterpret_cast<float4*>(&dys[buf][st_row[u] * kSPitch + st_col[u]]) = (row_ok && o_ok[u]) ? ra[u] : zero;
            *reinterpret_cast<float4*>(&xs[buf][st_row[u] * kSPitch + st_col[u]]) = (row_ok && i_ok[u]) ? rb[u] : zero;
        }
    };

    floatx16 acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int k = 0; k < 16; k++) acc[p][q][k] = 0.f;

    fetch(r_lo);
    store(r_lo, 0);
    __syncthreads();
    int buf = 0;
    for (long r = r_lo; r < r_hi; r += kSRows) {
        const bool more = r + kSRows < r_hi;                          // uniform
        if (more) fetch(r + kSRows);
        const float* a_lds = &dys[buf][kk * kSPitch + o_wave + m];
        const float* b_lds = &xs[buf][kk * kSPitch + i_wave + m];
#pragma unroll
        for (int s = 0; s < kSRows / 2; s++) {
            float a[2], b[2];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                a[p] = a_lds[2 * s * kSPitch + 32 * p];
                b[p] = b_lds[2 * s * kSPitch + 32 * p];
            }
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int q = 0; q < 2; q++)
                    acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[p], b[q], acc[p][q], 0, 0, 0);
        }
        if (more) store(r + kSRows, buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
    // D[o][i]: i = lane % 32, o = 8 (k / 4) + 4 (lane / 32) + k % 4 for register k
    float* plane = part + (long)blockIdx.z * O * I;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int i = i_tile + i_wave + 32 * q + m;
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const int o = o_tile + o_wave + 32 * p + 8 * (k / 4) + 4 * kk + (k % 4);
                if (o < O && i < I) plane[(long)o * I + i] = acc[p][q][k];
            }
        }
}

// Plain rows on the fp16 matrix cores with two-piece operands: dy and x are scaled by one power of two each (taken
// from an upper bound of their magnitudes, so that nothing overflows fp16; an entry 2^17 times smaller than the bound
// still keeps 22 bits) and split into hi + lo fp16 pieces; dy^T x takes three v_mfma_f32_32x32x16_f16 per step
// (lo hi, hi lo, hi hi; the lo lo term is below fp32 rounding), accumulated in fp32 and unscaled on the way out.
//
// The matrix instruction wants, per lane, 8 consecutive values along the reduction index, which here is the row
// index: both operands are transposed on their way into LDS.  A stage is 32 rows x 128 columns of each operand.
// Waves 0-1 stage dy, waves 2-3 stage x: a thread loads 8 rows x 4 columns (eight 16-byte loads), splits the 32
// values and writes, for each of its 4 columns, the 8 row-consecutive halves of each piece with one 16-byte store.
// Column c of the tile lives in LDS row 32 (c % 4) + c / 4, so that the 32 column quads of a wave write 32
// consecutive LDS rows (as the matrix lanes read 32 consecutive rows); the epilogue undoes the permutation.  Two
// stage buffers: while one is multiplied the next stage is split into the other and the loads of the one after are
// in flight.
//
// With the splitting between the matrix instructions, three instructions a value instead of five, each load sent as soon as its
// registers are free, no bank conflicts and a slice's tiles on one XCD, against one after the other: 512 x 512 on 155 744
// rows 375 -> 342 us, 16 368 67 -> 59, 8192 40 -> 36; 1280 x 16 on 27 000 68 -> 61; 256 x 512 on 127 456 187 -> 168.  What bounds the
// large ones: the parts add up as energy does, not as time (without the loads 290 us, without the LDS writes too 230,
// reads and matrix instructions alone 218, a third of those 109); small ones a stage's chain at one wave a SIMD.
constexpr int kFTile = 128;                        // dW tile edge
constexpr int kFRows = 32;                         // rows per stage: two matrix steps of 16
constexpr int kFRowW = 64;                         // bytes per LDS row: 32 halves in four 16-byte pieces, piece k of
                                                   // row R at position k ^ swizzle(R)
// Rows R, R + 4, R + 8, R + 12 apart for the reads (sixteen lanes at once over 64 banks), R, R + 2, R + 4, R + 6 for the writes (eight
// lanes over 32): no conflicts counted, a third of the LDS cycles with (R >> 2) & 3
__device__ __forceinline__ int swizzle(int row) { return (row >> 1 & 2) | ((row >> 1 ^ row >> 3) & 1); }
constexpr int kFPlane = kFTile * kFRowW;           // bytes of one piece of one operand
constexpr int kFBuf = 4 * kFPlane;                 // one stage: two operands x two pieces
constexpr int kFParts = 1024;                      // partial maxima per operand
// rows per accumulation run (a multiple of kFRows).  Slices get longer the more tiles a product has: 27 000 rows of 16 x 1280 are
// 1080 a slice, whose weights' gradients were off by 4.8e-7 of their 2-norm in one run and are by 3.4e-7 in runs of 256 (as the
// five products of 16 x 256, 211 rows a slice, were).  Runs of 128 took 4096 x 512 x 512 from 2.0e-7 to 1.6e-7 and 5000 rows of 64 x 256
// beside two of 256 x 256 from 2.5e-7 to 2.3e-7, for half a percent of a training step at most.  The column sums go by the same runs: in one
// chain a slice, 78 000 rows of an MLP's three layers were off by 4.6e-7 of the 2-norm product by product, by 6.4e-7 together, whose slices are
// longer, and are by 1.8e-7.
constexpr int kFRun = 128;

// parts[b] = max |x| over the b-th share of n floats (n % 4 == 0, x 16-byte aligned)
__global__ void __launch_bounds__(256) absmax_parts_kernel(const float* __restrict__ x, long n,
                                                           float* __restrict__ parts) {
    float m = 0.f;
    const long n4 = n >> 2, stride = (long)gridDim.x * 256;
    const float4* x4 = reinterpret_cast<const float4*>(x);
    long k = (long)blockIdx.x * 256 + threadIdx.x;
    for (; k + 3 * stride < n4; k += 4 * stride) {
        const float4 a = x4[k], b = x4[k + stride], c = x4[k + 2 * stride], d = x4[k + 3 * stride];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
        m = fmaxf(m, fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w))));
        m = fmaxf(m, fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fmaxf(fabsf(c.z), fabsf(c.w))));
        m = fmaxf(m, fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fmaxf(fabsf(d.z), fabsf(d.w))));
    }
    for (; k < n4; k += stride) {
        const float4 a = x4[k];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
    }
    for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
    __shared__ float wave_max[4];
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) parts[blockIdx.x] = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
}
// the same for several arrays of any length and alignment (bounds handed in by the caller) in one launch: array k from workgroup
// first_block on
struct BoundArray {
    const float* data;
    long n;
    float* parts;
    int blocks, first_block;
};
struct BoundArrays {
    BoundArray array[2 * MG_WGRAD_F16X2_JOBS];
    int count;
};
__global__ void __launch_bounds__(256) absmax_parts_scalar_kernel(const BoundArrays arrays) {
    int which = 0;
    while (which + 1 < arrays.count && (int)blockIdx.x >= arrays.array[which + 1].first_block) which++;     // (uniform)
    const BoundArray& a = arrays.array[which];
    const float* __restrict__ x = a.data;
    const long n = a.n, stride = 256L * a.blocks;
    const int block = blockIdx.x - a.first_block;
    float* __restrict__ parts = a.parts;
    float m = 0.f;
    for (long k = (long)block * 256 + threadIdx.x; k < n; k += stride) m = fmaxf(m, fabsf(x[k]));
    for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
    __shared__ float wave_max[4];
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) parts[block] = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
}
// parts[g per + b] = max |x[.., g]| over the b-th share of the rows of x (rows, groups); a block (b, g)
__global__ void __launch_bounds__(256) absmax_columns_kernel(const float* __restrict__ x, long rows, int groups, float* __restrict__ parts) {
    float m = 0.f;
    for (long r = (long)blockIdx.x * 256 + threadIdx.x; r < rows; r += 256L * gridDim.x) m = fmaxf(m, fabsf(x[r * groups + blockIdx.y]));
    for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
    __shared__ float wave_max[4];
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) parts[blockIdx.y * gridDim.x + blockIdx.x] = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
}

// One product dW = dy^T x of several over the same R rows.  group_cols: columns of x that share a scale (I: all of them); part: where
// its partial sums lie in the plane of a slice; colsum: the same of the column sums of dy, or negative.
struct WgradJob {
    const float *dy, *x, *dy_parts, *x_parts;
    int n_dy_parts, n_x_parts, group_cols, I, O, first_tile;
    long part, colsum, bias_rows;
};
struct WgradJobs {
    WgradJob job[MG_WGRAD_F16X2_JOBS];
    int count, tiles;
    long R, rows_per_block, plane;                         // plane: floats of a slice
    float* parts;
};
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) wgrad_f16x2_kernel(const WgradJobs jobs) {
    // [stage buffer][operand: dy, x][piece: hi, lo][LDS row][64 bytes]
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kFBuf];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 31, g = lane >> 5;
    // Workgroup ids go round-robin over the 8 XCDs: XCD x takes the x-th eighth of the (slice, tile) pairs, slice by slice, so that the
    // tiles of a slice, which read the same rows four times over, find them in one L2
    // (the tiles of all products that a launch takes)
    const long R = jobs.R, rows_per_block = jobs.rows_per_block;
    const int tiles = jobs.tiles;
    const long slices = ceil_div(R, rows_per_block), per_xcd = ceil_div(slices * tiles, 8);
    const long item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per_xcd || item >= slices * tiles) return;
    const long slice = item / tiles;
    const int all_tile = (int)(item - slice * tiles);
    int which = 0;
    while (which + 1 < jobs.count && all_tile >= jobs.job[which + 1].first_tile) which++;     // (uniform)
    const WgradJob& job = jobs.job[which];
    const float *__restrict__ dy = job.dy, *__restrict__ x = job.x, *__restrict__ dy_parts = job.dy_parts, *__restrict__ x_parts = job.x_parts;
    const int n_dy_parts = job.n_dy_parts, n_x_parts = job.n_x_parts, group_cols = job.group_cols, I = job.I, O = job.O;
    const long bias_rows = job.bias_rows;
    const int tile = all_tile - job.first_tile, tiles_o = (int)ceil_div(O, kFTile);
    const int o_tile = tile % tiles_o * kFTile, i_tile = tile / tiles_o * kFTile;
    const long r_lo = slice * rows_per_block;
    const long r_hi = r_lo + rows_per_block < R ? r_lo + rows_per_block : R;

    float scale = 0.f, unscale[2] = {0.f, 0.f};            // (set by set_scales below; of this lane's two columns of dW)
    // staging role of this thread: operand (wave-uniform), 8 rows from row 8 * octet, columns 4 cq .. 4 cq + 3.
    // A stage is the 32 rows from `first`; the last stage of a slice starts at r_hi - 32, inside the matrix
    // (rows >= 32), and the rows it shares with the stage before, or with the slice before, are scaled by zero, as
    // are the columns past the matrix (read from column 0): every load is unconditional and in bounds, and its
    // address is a uniform row address plus a constant lane offset.
    const bool stage_x = wave >= 2;
    const int st = threadIdx.x & 127, octet = st >> 5, cq = st & 31;
    const int dim = stage_x ? I : O, tile0 = stage_x ? i_tile : o_tile;
    const bool col_ok = tile0 + 4 * cq < dim;
    const float* operand = stage_x ? x : dy;                                       // (uniform)
    const unsigned lane_off = (unsigned)(8 * octet * dim + (col_ok ? tile0 + 4 * cq : 0));
    // (the swizzle of LDS rows cq + 32 j does not depend on j)
    unsigned char* st_dst = lds + (stage_x ? 2 * kFPlane : 0) + cq * kFRowW + 16 * (octet ^ swizzle(cq));
    float4 v[8];
    auto first_row = [&](long r) { return r + kFRows <= r_hi ? r : r_hi - kFRows; };
    auto fetch = [&](long r) {
        const float* rows = operand + first_row(r) * dim;                          // (uniform)
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = *reinterpret_cast<const float4*>(rows + u * dim + lane_off);
    };
    // column sums of dy over the slice (the bias gradient), by the workgroups of the first column of tiles
    const bool sum_cols = job.colsum >= 0 && i_tile == 0;                          // (uniform)
    float4 colsum = make_float4(0.f, 0.f, 0.f, 0.f), colsums = colsum;             // (of a run of stages, of the runs before it)
    // One stage in eight parts: part g splits columns 2 (g % 2) and one more of rows 2 (g / 2) and one more of the stage at r, which
    // are in v or on their way there; every second part requests the same two rows of the stage at r_next.  finish writes the pieces.
    struct Pieces {
        union { halfx2 pair[4]; halfx8 all; } hi[4], lo[4];
    };
    auto split_part = [&](int g, Pieces& out, long r, long r_next, auto sums) {
        const int q = g / 2, first_live = (int)(r - first_row(r)) - 8 * octet;     // rows u >= first_live count
        const float4 v0 = v[2 * q], v1 = v[2 * q + 1];
        const bool live[2] = {2 * q >= first_live, 2 * q + 1 >= first_live};
        const float s0 = live[0] ? scale : 0.f, s1 = live[1] ? scale : 0.f;
        if (g % 2 == 0) {
            split_pair(v0.x, v1.x, s0, s1, out.hi[0].pair[q], out.lo[0].pair[q]);
            split_pair(v0.y, v1.y, s0, s1, out.hi[1].pair[q], out.lo[1].pair[q]);
        } else {
            split_pair(v0.z, v1.z, s0, s1, out.hi[2].pair[q], out.lo[2].pair[q]);
            split_pair(v0.w, v1.w, s0, s1, out.hi[3].pair[q], out.lo[3].pair[q]);
        }
        if constexpr (decltype(sums)::value) {                                     // (selected: 0 * inf would be NaN)
            const long last_live = r < r_hi ? bias_rows - first_row(r) - 8 * octet : 0;    // rows u < last_live have a bias
            const bool c0 = live[0] && 2 * q < last_live, c1 = live[1] && 2 * q + 1 < last_live;
            if (g % 2 == 0) {
                colsum.x += c0 ? v0.x : 0.f; colsum.y += c0 ? v0.y : 0.f;
                colsum.x += c1 ? v1.x : 0.f; colsum.y += c1 ? v1.y : 0.f;
            } else {
                colsum.z += c0 ? v0.z : 0.f; colsum.w += c0 ? v0.w : 0.f;
                colsum.z += c1 ? v1.z : 0.f; colsum.w += c1 ? v1.w : 0.f;
            }
        }
        if (g % 2 == 1) {
            const float* next = operand + first_row(r_next) * dim;                 // (uniform)
            v[2 * q] = *reinterpret_cast<const float4*>(next + 2 * q * dim + lane_off);
            v[2 * q + 1] = *reinterpret_cast<const float4*>(next + (2 * q + 1) * dim + lane_off);
        }
    };
    auto finish = [&](const Pieces& out, int buf_off) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            *reinterpret_cast<halfx8*>(st_dst + buf_off + 32 * j * kFRowW) = out.hi[j].all;
            *reinterpret_cast<halfx8*>(st_dst + buf_off + kFPlane + 32 * j * kFRowW) = out.lo[j].all;
        }
    };

    // the two scales, from the partial maxima
    auto set_scales = [&]() {
    // (16-byte loads, four of them requested before the first is used: up to 64 values per thread and array)
    auto absmax_of = [&](const float* __restrict__ p, int n) {
        float mx = 0.f;
        const int n4 = (reinterpret_cast<uintptr_t>(p) & 15) == 0 ? n / 4 : 0;
        const float4* p4 = reinterpret_cast<const float4*>(p);
        auto fold = [&](const float4 t) {
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(t.x), fabsf(t.y))), fmaxf(fabsf(t.z), fabsf(t.w)));
        };
        int k = threadIdx.x;
        for (; k + 3 * 256 < n4; k += 4 * 256) {
            const float4 t0 = p4[k], t1 = p4[k + 256], t2 = p4[k + 512], t3 = p4[k + 768];
            fold(t0); fold(t1); fold(t2); fold(t3);
        }
        for (; k < n4; k += 256) fold(p4[k]);
        for (int j = 4 * n4 + threadIdx.x; j < n; j += 256) mx = fmaxf(mx, fabsf(p[j]));
        return mx;
    };
    float ma = absmax_of(dy_parts, n_dy_parts);
    float* wave_max = reinterpret_cast<float*>(lds);
    // a scale for every group of group_cols columns of x that the tile has a part of (n_x_parts maxima each)
    const int last_col = i_tile + kFTile < I ? i_tile + kFTile - 1 : I - 1, my_col = i_tile + 4 * cq, out_col = i_tile + 4 * m + 2 * (wave & 1);
    for (int p = i_tile / group_cols; p <= last_col / group_cols; p++) {
        float mb = absmax_of(x_parts + (long)p * n_x_parts, n_x_parts);
        for (int d = 1; d < 64; d <<= 1) { ma = fmaxf(ma, __shfl_xor(ma, d)); mb = fmaxf(mb, __shfl_xor(mb, d)); }
        if (lane == 0) { wave_max[wave] = ma; wave_max[4 + wave] = mb; }
        __syncthreads();
        ma = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
        mb = fmaxf(fmaxf(wave_max[4], wave_max[5]), fmaxf(wave_max[6], wave_max[7]));
        __syncthreads();
        float inv_a, inv_b;
        const float scale_a = pow2_scale(ma, &inv_a), scale_b = pow2_scale(mb, &inv_b);
        if (!stage_x) scale = col_ok ? scale_a : 0.f;
        else if (col_ok && my_col / group_cols == p) scale = scale_b;
#pragma unroll
        for (int q = 0; q < 2; q++)
            if ((out_col + q) / group_cols == p) unscale[q] = inv_a * inv_b;
    }
    };

    floatx16 acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int k = 0; k < 16; k++) acc[p][q][k] = 0.f;

    // matrix lanes: LDS rows 64 (wave / 2) + 32 p + m of dy, 64 (wave % 2) + 32 q + m of x; 16-byte piece 2 step + g,
    // swizzled
    const int sw = swizzle(m);
    const unsigned char* a_lds = lds + ((wave >> 1) * 64 + m) * kFRowW;
    const unsigned char* b_lds = lds + 2 * kFPlane + ((wave & 1) * 64 + m) * kFRowW;
    halfx8 ah[2], al[2], bh[2], bl[2];
    auto read_a = [&](int p, int s, int buf_off) {
        const unsigned char* at = a_lds + buf_off + 16 * ((2 * s + g) ^ sw) + 32 * p * kFRowW;
        ah[p] = *reinterpret_cast<const halfx8*>(at);
        al[p] = *reinterpret_cast<const halfx8*>(at + kFPlane);
    };
    auto read_b = [&](int q, int s, int buf_off) {
        const unsigned char* at = b_lds + buf_off + 16 * ((2 * s + g) ^ sw) + 32 * q * kFRowW;
        bh[q] = *reinterpret_cast<const halfx8*>(at);
        bl[q] = *reinterpret_cast<const halfx8*>(at + kFPlane);
    };
    auto product = [&](int p, int q) {                     // small terms first
        acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[p], bh[q], acc[p][q], 0, 0, 0);
        acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[p], bl[q], acc[p][q], 0, 0, 0);
        acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[p], bh[q], acc[p][q], 0, 0, 0);
    };

    // The matrix instructions accumulate runs of kFRun rows; the runs are added in a second set of registers: the
    // rounding error of an fp32 sum grows with its length, and a slice of 50 000 rows in one chain was 1.7 times
    // less accurate than the same sum in chunks.
    floatx16 total[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int k = 0; k < 16; k++) total[p][q][k] = 0.f;
    // A stage is multiplied out of one buffer while the next one is split into the other and the loads of the one
    // after that are on their way; three matrix instructions and a part of the splitting in turn, in this order (left to itself the
    // compiler multiplies first and splits then, and every load is waited for as soon as it is sent).
    // (stages past the slice are fetched and stored like the others, scaled by zero and never multiplied: the loop
    // body has no branch)
    auto walk = [&](auto sums) {
        Pieces next;
#pragma unroll
        for (int k = 0; k < 8; k++) split_part(k, next, r_lo, r_lo + kFRows, sums);
        finish(next, 0);
        __syncthreads();
        int buf_off = 0;
        for (long r = r_lo; r < r_hi;) {
            const long run_hi = r + kFRun < r_hi ? r + kFRun : r_hi;
            for (; r < run_hi; r += kFRows) {
                read_a(0, 0, buf_off);
                read_b(0, 0, buf_off);
                read_b(1, 0, buf_off);
                read_a(1, 0, buf_off);
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    __builtin_amdgcn_sched_barrier(0);
                    split_part(k, next, r + kFRows, r + 2 * kFRows, sums);
                    __builtin_amdgcn_sched_barrier(0);
                    product(k >> 1 & 1, k & 1);
                    if (k == 1) read_a(0, 1, buf_off);
                    if (k == 2) read_b(0, 1, buf_off);
                    if (k == 3) {
                        read_b(1, 1, buf_off);
                        read_a(1, 1, buf_off);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                buf_off ^= kFBuf;
                finish(next, buf_off);
                __syncthreads();
            }
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int k = 0; k < 16; k++) { total[p][q][k] += acc[p][q][k]; acc[p][q][k] = 0.f; }
            if constexpr (decltype(sums)::value) {
                colsums.x += colsum.x; colsums.y += colsum.y; colsums.z += colsum.z; colsums.w += colsum.w;
                colsum = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    };
    fetch(r_lo);
    set_scales();                                          // (the first stage is on its way meanwhile)
    if (sum_cols) walk(std::true_type{});
    else walk(std::false_type{});
    float* plane = jobs.parts + slice * jobs.plane;
    if (sum_cols) {
        // the four row groups of a column quad, added in a fixed order
        float4* sums = reinterpret_cast<float4*>(lds);                             // [octet][cq]; the stage buffers are done with
        if (!stage_x) sums[octet * 32 + cq] = colsums;                             // (the stage behind the last run added nothing)
        __syncthreads();
        if (threadIdx.x < 32) {
            const float4 s0 = sums[cq], s1 = sums[32 + cq], s2 = sums[64 + cq], s3 = sums[96 + cq];
            const int o = o_tile + 4 * cq;
            if (o < O)
                *reinterpret_cast<float4*>(plane + job.colsum + o) =
                    make_float4((s0.x + s1.x) + (s2.x + s3.x), (s0.y + s1.y) + (s2.y + s3.y),
                                (s0.z + s1.z) + (s2.z + s3.z), (s0.w + s1.w) + (s2.w + s3.w));
        }
    }
    // D[row][col]: col = lane % 32, row = 8 (k / 4) + 4 (lane / 32) + k % 4 for register k; LDS row 32 j + c / 4 of
    // an operand is column 4 (c / 4) + j of the tile
    float* out = plane + job.part;
    const int i = i_tile + 4 * m + 2 * (wave & 1);         // (and i + 1: I is a multiple of four)
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const int o = o_tile + 4 * (8 * (k / 4) + 4 * g + (k % 4)) + 2 * (wave >> 1) + p;
            if (o < O && i < I)
                *reinterpret_cast<float2*>(out + (long)o * I + i) = make_float2(total[p][0][k] * unscale[0], total[p][1][k] * unscale[1]);
        }
}

// dW[k] = part[0][k] + part[1][k] + ... in this order
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float* __restrict__ part, long n, int splits,
                                                           float* __restrict__ dW) {
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
        float s = 0.f;
        int z = 0;
        for (; z + 8 <= splits; z += 8) {                  // eight loads in flight, added in slice order
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = part[(long)(z + u) * n + k];
#pragma unroll
            for (int u = 0; u < 8; u++) s += v[u];
        }
        for (; z < splits; z++) s += part[(long)z * n + k];
        dW[k] = s;
    }
}

// Sums of planes of few quads and many slices: 16 threads a quad, every sum in pairs (512 slices one after the other were a third
// of a narrow gradient's rounding): one thread a quad took 10 to 13 us for planes of 1000 quads and 192 to 512 slices, four workgroups, of which each load is waited for.
__device__ __forceinline__ float4 sum_of_slices(const float4* __restrict__ part, int quads, int splits, int k, float4* shared) {
    const int z = threadIdx.x >> 4;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    auto plus = [](const float4& a, const float4& b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); };
    auto add = [&](const float4& v) { s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w; };
    if (k < quads) {
        int j = z;
        for (; j + 48 < splits; j += 64) {
            const float4 v0 = part[(long)j * quads + k], v1 = part[(long)(j + 16) * quads + k], v2 = part[(long)(j + 32) * quads + k],
                         v3 = part[(long)(j + 48) * quads + k];
            add(plus(plus(v0, v1), plus(v2, v3)));
        }
        for (; j < splits; j += 16) add(part[(long)j * quads + k]);
    }
    shared[threadIdx.x] = s;
    __syncthreads();
    const float4* of = shared + (threadIdx.x & 15);
    float4 four[4];
#pragma unroll
    for (int j = 0; j < 4; j++) four[j] = plus(plus(of[64 * j], of[64 * j + 16]), plus(of[64 * j + 32], of[64 * j + 48]));
    return plus(plus(four[0], four[1]), plus(four[2], four[3]));
}
// the same for the planes of several products: quad k of a plane goes to the segment that holds it
struct WgradSegments {
    float* out[2 * MG_WGRAD_F16X2_JOBS];
    int first_quad[2 * MG_WGRAD_F16X2_JOBS];
    int count;
    bool aligned;                                          // every out is 16-byte aligned
};
template <bool MANY>
__global__ void __launch_bounds__(256) wgrad_reduce_f16x2_kernel(const float4* __restrict__ part, int quads, int splits,
                                                                 const WgradSegments seg) {
    __shared__ float4 shared[MANY ? 256 : 1];
    const int k = MANY ? 16 * blockIdx.x + (threadIdx.x & 15) : 256 * blockIdx.x + threadIdx.x;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (MANY) s = sum_of_slices(part, quads, splits, k, shared);
    if (k >= quads || (MANY && threadIdx.x >= 16)) return;
    if constexpr (!MANY) {
        auto plus = [](const float4& a, const float4& b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); };
        int z = 0;
        for (; z + 8 <= splits; z += 8) {                  // eight loads in flight, added in pairs
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = part[(long)(z + u) * quads + k];
            s = plus(s, plus(plus(plus(v[0], v[1]), plus(v[2], v[3])), plus(plus(v[4], v[5]), plus(v[6], v[7]))));
        }
        for (; z < splits; z++) s = plus(s, part[(long)z * quads + k]);
    }
    float* out = seg.out[0];
    int first = 0;
#pragma unroll
    for (int j = 1; j < 2 * MG_WGRAD_F16X2_JOBS; j++)
        if (j < seg.count && k >= seg.first_quad[j]) { out = seg.out[j]; first = seg.first_quad[j]; }
    out += 4L * (k - first);
    if (seg.aligned) *reinterpret_cast<float4*>(out) = s;
    else { out[0] = s.x; out[1] = s.y; out[2] = s.z; out[3] = s.w; }
}

// ---------------------------------------------------------------------------------------- one dimension of at most 16
// P[k, i] = sum_{r, t} narrow[r, k, t] wide[r, i, t] with k < n <= 16: two to thirty-two operations a float of the wide operand, which
// is read once, 16 bytes a lane, in whatever layout of components it has: nothing is transposed, and products and sums are fp32, so
// no bounds are needed either.
constexpr int kNarrow = 16, kNarrowRows = 64, kNarrowChains = 4;
enum NarrowBias { kNoBias, kOfWide, kOfNarrow };

// Plain rows, by matrix instructions: a wave takes 64 channels of every (4 / waves_c)-th step of four rows, a lane one row and four
// channels of the wide operand and one number of the narrow one, both as they lie in memory.  No LDS and no barrier until the end,
// so loads of kAhead steps are in flight while the steps before them are multiplied; the sums of every fourth step are a chain of
// their own (64 registers, and no longer chains than sixteen groups of lanes would have).
// Bound by memory: 1.5 M rows 16 -> 512 at 5.8 TB/s, 73 728 rows 1280 -> 16 at 5.0.  With the n results of four channels as
// multiply-adds of one lane, the narrow rows in LDS and two barriers for every 64 rows, loads and arithmetic took turns: 697 us against
// 545, 106 against 76, 73 728 rows 16 -> 256 32.5 against 25.5, 8192 rows 260 -> 16 15.5 against 10.3, level at 9.5 for 4096 rows
// 64 -> 1.  The split-fp16 product with its padding to 128 x 128 and its row maxima: 1242, 168 and 52 us.  Error against float64
// (2-norm, normal numbers): 73 728 rows 16 -> 256 1.4e-7 against 1.8e-7, 131 072 rows 8 -> 512 1.7e-7 against 2.0e-7.
// BIAS: the sums of the columns of dy as well, where dy is the wide operand or the narrow one; behind the plane (n, dim).
template <int BIAS>
__global__ void __launch_bounds__(256, 4) wgrad_narrow_rows_kernel(const float* __restrict__ narrow, int n, const float* __restrict__ wide,
                                                                int dim, long R, long rows_per_block, int waves_c, long plane,
                                                                float* __restrict__ part) {
    typedef float floatx4 __attribute__((ext_vector_type(4)));
    constexpr int kAhead = BIAS == kOfWide ? 4 : 8;             // (128 registers, four workgroups on a compute unit)
    __shared__ float4 shared[3 * 64 * 5];                      // of the row waves but the first: results, sums of columns
    __shared__ float shared_narrow[3 * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, sub = lane >> 4;
    const int shift = __builtin_ctz(waves_c), waves_r = 4 >> shift, wr = wave >> shift, wc = wave & (waves_c - 1);
    const int quad = (blockIdx.x * waves_c + wc) * 16 + c;
    const bool live = quad < dim / 4;
    const int own = live ? 4 * quad : 0, own_n = c < n ? c : 0;
    const long r_first = (long)blockIdx.y * rows_per_block, r_hi = r_first + rows_per_block < R ? r_first + rows_per_block : R;
    const int stride = 4 * waves_r;                            // rows between the steps of a wave
    floatx4 acc[kNarrowChains][4];
#pragma unroll
    for (int u = 0; u < kNarrowChains; u++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[u][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float column[4] = {0.f, 0.f, 0.f, 0.f};                    // BIAS: of the wide operand's four channels, or four chains of the narrow's
    float4 x[kAhead];
    float a[kAhead];
    auto load = [&](int u, long r) {                           // of rows r .. r + 3; those behind the last: the last, not counted
        const long row = r < r_hi ? r : r_hi - 1;
        const int past = r_hi - 1 - row < 3 ? (int)(r_hi - 1 - row) : 3, k = sub < past ? sub : past;
        x[u] = *reinterpret_cast<const float4*>(wide + row * dim + (unsigned)(k * dim + own));
        a[u] = (narrow + row * n)[(unsigned)(k * n + own_n)];
    };
    auto use = [&](int u, long r) {
        const bool in = sub < r_hi - r;                        // both operands are cleared: infinities of a row read twice stay out
        const float v[4] = {in ? x[u].x : 0.f, in ? x[u].y : 0.f, in ? x[u].z : 0.f, in ? x[u].w : 0.f};
        const float k = in && c < n ? a[u] : 0.f;
#pragma unroll
        for (int j = 0; j < 4; j++)
            acc[u % kNarrowChains][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, v[j], acc[u % kNarrowChains][j], 0, 0, 0);
        if constexpr (BIAS == kOfWide)
#pragma unroll
            for (int j = 0; j < 4; j++) column[j] += v[j];
        if constexpr (BIAS == kOfNarrow) column[u % 4] += k;
    };
    const long round = (long)kAhead * stride;
    const int rounds = (int)((r_hi - r_first + round - 1) / round);
    long r = r_first + 4 * wr;
#pragma unroll
    for (int u = 0; u < kAhead; u++) load(u, r + u * stride);
    for (int k = 1; k < rounds; k++, r += round) {
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            use(u, r + u * stride);
            load(u, r + round + u * stride);
        }
    }
#pragma unroll
    for (int u = 0; u < kAhead; u++)
        if (r + u * stride < r_hi) use(u, r + u * stride);      // (uniform)
    // the chains, then the waves of rows, added in their order; a lane has the results 4 sub + i of its four channels
    float4 sum[5];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = (acc[0][j][i] + acc[1][j][i]) + (acc[2][j][i] + acc[3][j][i]);
        sum[i] = make_float4(v[0], v[1], v[2], v[3]);
    }
    constexpr int kSums = BIAS == kOfWide ? 5 : 4;
    float of_narrow = 0.f;
    if constexpr (BIAS == kOfWide) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            column[j] += __shfl_xor(column[j], 16);
            column[j] += __shfl_xor(column[j], 32);
        }
        sum[4] = make_float4(column[0], column[1], column[2], column[3]);
    }
    if constexpr (BIAS == kOfNarrow) {
        of_narrow = (column[0] + column[1]) + (column[2] + column[3]);
        of_narrow += __shfl_xor(of_narrow, 16);
        of_narrow += __shfl_xor(of_narrow, 32);
    }
    if (wr > 0) {
        const int slot = (wr - 1) * waves_c + wc;
#pragma unroll
        for (int i = 0; i < kSums; i++) shared[(slot * 5 + i) * 64 + lane] = sum[i];
        if (BIAS == kOfNarrow && wc == 0 && lane < 16) shared_narrow[(wr - 1) * 16 + c] = of_narrow;
    }
    __syncthreads();
    if (wr > 0) return;
    for (int g = 0; g < waves_r - 1; g++) {
        const int slot = g * waves_c + wc;
#pragma unroll
        for (int i = 0; i < kSums; i++) {
            const float4 v = shared[(slot * 5 + i) * 64 + lane];
            sum[i].x += v.x; sum[i].y += v.y; sum[i].z += v.z; sum[i].w += v.w;
        }
        if constexpr (BIAS == kOfNarrow) of_narrow += shared_narrow[g * 16 + c];
    }
    float* out = part + blockIdx.y * plane;
    if (live) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (4 * sub + i < n) *reinterpret_cast<float4*>(out + (long)(4 * sub + i) * dim + 4 * quad) = sum[i];
        if (BIAS == kOfWide && sub == 0) *reinterpret_cast<float4*>(out + (long)n * dim + 4 * quad) = sum[4];
    }
    if (BIAS == kOfNarrow && blockIdx.x == 0 && wc == 0 && lane < 16) out[(long)n * dim + c] = of_narrow;
}

// Rows of T = 3 or 9 components: a lane holds the n results of four channels, L lanes a row, 256 / L rows at a time; the narrow
// operand's rows lie in LDS, where all lanes of a row read the same words.  8192 rows of three components 1 -> 128 and 128 -> 1 8 us,
// 128 -> 16 18, of nine 128 -> 1 11; the split-fp16 product with its padding to 128 x 128, its row maxima and transposed copies 42, 41, 68.
template <int T, int N>
__global__ void __launch_bounds__(256) wgrad_narrow_kernel(const float* __restrict__ narrow, int n, const float* __restrict__ wide,
                                                           int dim, long R, long rows_per_block, int L, long plane,
                                                           float* __restrict__ part) {
    constexpr int kAhead = T == 3 ? 4 : 1;                    // rows requested together
    __shared__ __attribute__((aligned(16))) float buf[kNarrowRows * N * T > 1024 ? kNarrowRows * N * T : 1024];
    const int l = threadIdx.x & (L - 1), group = threadIdx.x / L, groups = 256 / L;
    const int quad = blockIdx.x * L + l;
    const bool live = quad < dim / 4;
    const float* own = wide + (live ? quad : 0) * 4L * T;
    const long r_lo = (long)blockIdx.y * rows_per_block, r_hi = r_lo + rows_per_block < R ? r_lo + rows_per_block : R;
    float acc[N][4];
#pragma unroll
    for (int k = 0; k < N; k++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[k][j] = 0.f;
    for (long r = r_lo; r < r_hi; r += kNarrowRows) {
        const int rows = r_hi - r < kNarrowRows ? (int)(r_hi - r) : kNarrowRows;
        __syncthreads();
        // (what lies between n and N is never used)
        for (int at = threadIdx.x; at < rows * n * T; at += 256) {
            const int row = at / (n * T);
            buf[row * (N * T) + (at - row * (n * T))] = narrow[r * n * T + at];
        }
        __syncthreads();
        for (int first = group; first < rows; first += kAhead * groups) {
            union { float4 v[T]; float f[4 * T]; } x[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const int row = first + u * groups < rows ? first + u * groups : rows - 1;
                const float4* from = reinterpret_cast<const float4*>(own + (r + row) * ((long)dim * T));
#pragma unroll
                for (int t = 0; t < T; t++) x[u].v[t] = from[t];
            }
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const int row = first + u * groups;
                if (row < rows) {
                    const float* b = buf + row * (N * T);
#pragma unroll
                    for (int k = 0; k < N; k++)
#pragma unroll
                        for (int t = 0; t < T; t++)
#pragma unroll
                            for (int j = 0; j < 4; j++) acc[k][j] = fmaf(b[k * T + t], x[u].f[j * T + t], acc[k][j]);
                }
            }
        }
    }
    // the groups' sums, added in their order
    float4* sums = reinterpret_cast<float4*>(buf);
    auto combine = [&](int k, const float (&own_sum)[4]) {
        __syncthreads();
        sums[threadIdx.x] = make_float4(own_sum[0], own_sum[1], own_sum[2], own_sum[3]);
        __syncthreads();
        if (group == 0 && live) {
            float4 s = sums[l];
            for (int g = 1; g < groups; g++) {
                const float4 v = sums[g * L + l];
                s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
            }
            *reinterpret_cast<float4*>(part + blockIdx.y * plane + (long)k * dim + 4 * quad) = s;
        }
    };
#pragma unroll
    for (int k = 0; k < N; k++)
        if (k < n) combine(k, acc[k]);                        // (uniform)
}

// quad q of the plane (n, dim) to dW, transposed where x is the narrow operand, and those behind it to db (n_bias floats)
__global__ void __launch_bounds__(256) wgrad_narrow_reduce_kernel(const float4* __restrict__ part, int quads, int splits, int dim,
                                                                  int n, bool transposed, int n_bias, float* __restrict__ dW,
                                                                  float* __restrict__ db) {
    __shared__ float4 shared[256];
    const int q = 16 * blockIdx.x + (threadIdx.x & 15);
    const float4 s = sum_of_slices(part, quads, splits, q, shared);
    if (threadIdx.x >= 16 || q >= quads) return;
    const float v[4] = {s.x, s.y, s.z, s.w};
    const int k = q / (dim / 4), i = 4 * (q - k * (dim / 4));
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (k < n) dW[transposed ? (long)(i + j) * n + k : (long)k * dim + i + j] = v[j];
        else if (i + j < n_bias) db[i + j] = v[j];
    }
}

// lanes of a row (plain rows: waves that share one, 64 channels each), channel blocks, rows of a workgroup and their number: about four
// workgroups on each compute unit, of 64 rows at least
struct NarrowPlan {
    int lanes, waves_c, blocks, n, dim;
    long rows, splits, plane;
};
NarrowPlan narrow_plan(long R, int dim_in, int dim_out) {
    NarrowPlan p;
    p.n = dim_in < dim_out ? dim_in : dim_out;
    p.dim = dim_in < dim_out ? dim_out : dim_in;
    p.lanes = 16;
    while (p.lanes < 64 && 4 * p.lanes < p.dim) p.lanes *= 2;
    p.waves_c = p.lanes / 16;
    p.blocks = (int)ceil_div(p.dim, 4 * p.lanes);
    const long most = ceil_div(R, kNarrowRows), want = 1024 / p.blocks, s = want < most ? want : most;   // (no more than are resident at once)
    p.rows = ceil_div(ceil_div(R, s < 1 ? 1 : s), kNarrowRows) * kNarrowRows;
    p.splits = ceil_div(R, p.rows);
    p.plane = (long)p.n * p.dim;
    return p;
}
long narrow_bias_floats(int dim_in, int dim_out) { return dim_in < dim_out ? dim_out : kNarrow; }

// rows per slice and number of slices for a problem (the same on the sizing and the launching side)
// resident_groups = 0: aim at ~4 workgroups per CU; otherwise the number of workgroups the chip holds at once, which
// the grid then does not exceed (a second, partly filled round would cost a whole slice's time)
void wgrad_split_tiles(long rows, long tiles, long* rows_per_block, long* splits, long resident_groups = 0) {
    long s = resident_groups > 0 ? resident_groups / tiles : ceil_div(1024, tiles);
    const long max_splits = ceil_div(rows, 64);
    if (s > max_splits) s = max_splits;
    if (s < 1) s = 1;
    if (s > 65535) s = 65535;
    long rpb = ceil_div(rows, s);
    rpb = ceil_div(rpb, 32) * 32;                      // (a multiple of every kernel's rows per trip)
    *rows_per_block = rpb;
    *splits = rows > 0 ? ceil_div(rows, rpb) : 0;
}
void wgrad_split(long rows, int dim_in, int dim_out, int tile, long* rows_per_block, long* splits) {
    wgrad_split_tiles(rows, ceil_div(dim_out, tile) * ceil_div(dim_in, tile), rows_per_block, splits);
}
// plain rows take the matrix-core kernel and its 128 x 128 tiles
inline int wgrad_tile(int inds) { return inds == 0 ? kMTile : kTile; }

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_tensor_linear_wgrad_workspace_bytes(long rows, int dim_in, int dim_out, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && rows >= 0 && dim_in >= 0 && dim_out >= 0, "mg_tensor_linear_wgrad_workspace_bytes: bad argument");
    // (the number of tensor indices is not known here: room for either kernel's slices)
    long rpb, s_plain, s_comp;
    wgrad_split(rows, dim_in, dim_out, kMTile, &rpb, &s_plain);
    wgrad_split(rows, dim_in, dim_out, kTile, &rpb, &s_comp);
    const long splits = s_plain > s_comp ? s_plain : s_comp;
    // (+ the partial maxima and the column sums of the split-fp16 variant)
    *bytes = (size_t)splits * ((size_t)dim_in + 1) * (size_t)dim_out * sizeof(float) + 16 + 2 * kFParts * sizeof(float);
    return MG_OK;
}

int mg_tensor_linear_wgrad_f16x2_supported(long rows, int dim_in, int dim_out) {
    return rows >= 4096 && dim_in >= 4 && dim_out >= 4 && dim_in % 4 == 0 && dim_out % 4 == 0;
}

// How many of the first of `count` products over the same rows go together: while their tiles leave the chip's 256 compute units two
// slices.  What a launch costs beside its products, the bounds that every workgroup reads, the first loads, the partial results of
// as many workgroups as the chip holds and their sum, is then paid once, and the slices are longer: the three products of
// an MLP 128 -> 512 -> 512 -> 512 at 4096 rows 77 -> 39 us, at 8192 92 -> 56, at 32 768 242 -> 183, at 155 744 806 -> 758; four of
// 256 x 256 at 24 576 141 -> 76; 512 x 1024 and two of 1024 x 1024 at 8192 (two launches) 204 -> 194.  The longer slices cost
// up to 15 % in the error of a narrow product (128 -> 512 at 4096 rows 1.6e-7 of its 2-norm from float64, singly 1.4e-7) and 25 % in the column
// sums (1.7e-7, 1.4e-7 at 78 000 rows), in runs of kFRun rows both.
constexpr long kMergedTiles = 128;
static long job_tiles(const mg_wgrad_f16x2& j) { return ceil_div(j.dim_out, kFTile) * ceil_div(j.dim_in, kFTile); }
static int together(const mg_wgrad_f16x2* jobs, int count) {
    long tiles = 0;
    for (int k = 0; k < count && k < MG_WGRAD_F16X2_JOBS; k++) {
        tiles += job_tiles(jobs[k]);
        if (k > 0 && tiles > kMergedTiles) return k;
    }
    return count < MG_WGRAD_F16X2_JOBS ? count : MG_WGRAD_F16X2_JOBS;
}
static void slices_of(const mg_wgrad_f16x2* jobs, int count, long rows, long* rpb, long* splits, long* plane) {
    long tiles = 0;
    *plane = 0;
    for (int k = 0; k < count; k++) {
        tiles += job_tiles(jobs[k]);
        *plane += (long)jobs[k].dim_in * jobs[k].dim_out + (jobs[k].db ? jobs[k].dim_out : 0);
    }
    // Two workgroups per CU fit; where that leaves slices of fewer than some 320 rows, one per CU is faster (half the partial results to
    // write and add up; one against two: 4096 x 512 x 512 29, 35 us, four of 64 x 64 at 8192 19, 24, 64 x 256 and two of 256 x 256 at
    // 8192 28, 30; but 256 x 384 and two of 384 x 384 at 8192 47, 43, at 16 384 78, 70, 101 000 x 512 x 512 281, 238)
    constexpr long kShortSlices = 163840;
    wgrad_split_tiles(rows, tiles, rpb, splits, rows < 65536 && rows * tiles < kShortSlices ? 256 : 512);
}

// x_groups > 1: x_bound holds (rows, x_groups) maxima, one of each dim_in / x_groups columns
static int wgrad_f16x2(const mg_wgrad_f16x2* jobs, int count, int x_groups, long rows, void* workspace, mg_stream_t stream) {
    hipStream_t st = (hipStream_t)stream;
    WgradJobs all{};
    long rpb, splits, plane;
    slices_of(jobs, count, rows, &rpb, &splits, &plane);
    all.count = count;
    all.R = rows;
    all.rows_per_block = rpb;
    all.plane = plane;
    all.parts = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t(15));
    float* maxima = all.parts + splits * plane;              // per job [dy: kFParts][x: kFParts]
    constexpr long kDirectBounds = 16384;                    // a bound array this short is read by every workgroup itself
    auto blocks_for = [](long len) { return (int)(ceil_div(len, 4096) < kFParts ? ceil_div(len, 4096) : kFParts); };
    BoundArrays scan{};
    int scan_blocks = 0;
    // partial maxima of the caller's bounds, or of the data itself; an array that two products share is scanned once
    auto bound_parts = [&](const float* data, long n_data, const float* bound, long n_bound, float* parts, const float** from) -> int {
        *from = bound;
        if (bound && n_bound <= kDirectBounds) return (int)n_bound;
        *from = parts;
        const int blocks = blocks_for(bound ? n_bound : n_data);
        if (!bound) {
            hipLaunchKernelGGL(absmax_parts_kernel, dim3(blocks), dim3(256), 0, st, data, n_data, parts);
            return blocks;
        }
        for (int k = 0; k < scan.count; k++)
            if (scan.array[k].data == bound && scan.array[k].n == n_bound) {
                *from = scan.array[k].parts;
                return blocks;
            }
        scan.array[scan.count++] = BoundArray{bound, n_bound, parts, blocks, scan_blocks};
        scan_blocks += blocks;
        return blocks;
    };
    WgradSegments seg{};
    seg.aligned = true;
    long at = 0;
    auto segment = [&](float* out, long n) {
        seg.out[seg.count] = out;
        seg.first_quad[seg.count++] = (int)(at / 4);
        seg.aligned = seg.aligned && aligned16(out);
        at += n;
        return at - n;
    };
    for (int k = 0; k < count; k++) {
        const mg_wgrad_f16x2& j = jobs[k];
        WgradJob& to = all.job[k];
        to = WgradJob{j.dy, j.x, nullptr, nullptr, 0, 0, j.dim_in / x_groups, j.dim_in, j.dim_out, all.tiles, 0, -1, j.bias_rows};
        all.tiles += (int)job_tiles(j);
        float *dy_maxima = maxima + 2L * k * kFParts, *x_maxima = dy_maxima + kFParts;
        to.n_dy_parts = bound_parts(j.dy, rows * j.dim_out, j.dy_bound, j.n_dy_bound, dy_maxima, &to.dy_parts);
        if (x_groups > 1) {
            const long per = kFParts / x_groups;
            to.n_x_parts = (int)(ceil_div(rows, 1024) < per ? ceil_div(rows, 1024) : per);
            to.x_parts = x_maxima;
            hipLaunchKernelGGL(absmax_columns_kernel, dim3((unsigned)to.n_x_parts, (unsigned)x_groups), dim3(256), 0, st, j.x_bound, rows,
                               x_groups, x_maxima);
        } else {
            to.n_x_parts = bound_parts(j.x, rows * j.dim_in, j.x_bound, j.n_x_bound, x_maxima, &to.x_parts);
        }
        to.part = segment(j.dW, (long)j.dim_in * j.dim_out);
    }
    for (int k = 0; k < count; k++)
        if (jobs[k].db) all.job[k].colsum = segment(jobs[k].db, jobs[k].dim_out);
    if (scan.count > 0) hipLaunchKernelGGL(absmax_parts_scalar_kernel, dim3((unsigned)scan_blocks), dim3(256), 0, st, scan);
    const long items = all.tiles * splits;
    MG_REQUIRE(items < (1L << 31) - 8 && plane / 4 < (1L << 31), "mg_tensor_linear_wgrad_f16x2: grid too large");
    hipLaunchKernelGGL(wgrad_f16x2_kernel, dim3((unsigned)(8 * ceil_div(items, 8))), dim3(256), 0, st, all);
    const int quads = (int)(plane / 4);
    const bool many = splits > 32;
    hipLaunchKernelGGL(many ? wgrad_reduce_f16x2_kernel<true> : wgrad_reduce_f16x2_kernel<false>,
                       dim3((unsigned)ceil_div(quads, many ? 16 : 256)), dim3(256), 0, st,
                       reinterpret_cast<const float4*>(all.parts), quads, (int)splits, seg);
    return check_launch("mg_tensor_linear_wgrad_f16x2");
}

static int check_jobs(const mg_wgrad_f16x2* jobs, int count, long rows) {
    for (int k = 0; k < count; k++) {
        const mg_wgrad_f16x2& j = jobs[k];
        MG_REQUIRE(mg_tensor_linear_wgrad_f16x2_supported(rows, j.dim_in, j.dim_out),
                   "mg_tensor_linear_wgrad_f16x2: needs rows >= 4096 and dims that are multiples of 4");
        MG_REQUIRE(j.dy && j.x && j.dW, "mg_tensor_linear_wgrad_f16x2: null pointer");
        MG_REQUIRE(aligned16(j.dy) && aligned16(j.x), "mg_tensor_linear_wgrad_f16x2: dy and x must be 16-byte aligned");
        MG_REQUIRE((j.dy_bound == nullptr || j.n_dy_bound > 0) && (j.x_bound == nullptr || j.n_x_bound > 0),
                   "mg_tensor_linear_wgrad_f16x2: empty bound array");
    }
    return MG_OK;
}

int mg_tensor_linear_wgrad_f16x2_many_workspace_bytes(const mg_wgrad_f16x2* jobs, int count, long rows, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && count >= 0 && (jobs || count == 0) && rows >= 0,
               "mg_tensor_linear_wgrad_f16x2_many_workspace_bytes: bad argument");
    size_t most = 0;
    for (int k = 0; k < count;) {
        const int n = together(jobs + k, count - k);
        long rpb, splits, plane;
        slices_of(jobs + k, n, rows, &rpb, &splits, &plane);
        const size_t need = ((size_t)splits * (size_t)plane + 2 * (size_t)n * kFParts) * sizeof(float) + 16;
        most = need > most ? need : most;
        k += n;
    }
    *bytes = most;
    return MG_OK;
}

int mg_tensor_linear_wgrad_f16x2_many(const mg_wgrad_f16x2* jobs, int count, long rows, void* workspace, mg_stream_t stream) {
    MG_REQUIRE(count >= 0 && (jobs || count == 0), "mg_tensor_linear_wgrad_f16x2_many: bad argument");
    if (int code = check_jobs(jobs, count, rows)) return code;
    MG_REQUIRE(workspace || count == 0, "mg_tensor_linear_wgrad_f16x2: null pointer");
    for (int k = 0; k < count;) {
        const int n = together(jobs + k, count - k);
        if (int code = wgrad_f16x2(jobs + k, n, 1, rows, workspace, stream)) return code;
        k += n;
    }
    return MG_OK;
}

static int wgrad_f16x2_one(const mg_wgrad_f16x2& job, int x_groups, long rows, void* workspace, mg_stream_t stream) {
    if (int code = check_jobs(&job, 1, rows)) return code;
    MG_REQUIRE(workspace, "mg_tensor_linear_wgrad_f16x2: null pointer");
    return wgrad_f16x2(&job, 1, x_groups, rows, workspace, stream);
}

int mg_tensor_linear_wgrad_f16x2_rows(const float* dy, const float* x, const float* dy_bound, long n_dy_bound,
                                      const float* x_bound, long n_x_bound, long rows, long bias_rows, int dim_in, int dim_out,
                                      void* workspace, float* dW, float* db, mg_stream_t stream) {
    return wgrad_f16x2_one({dy, x, dy_bound, n_dy_bound, x_bound, n_x_bound, bias_rows, dim_in, dim_out, dW, db}, 1, rows, workspace,
                           stream);
}

int mg_tensor_linear_wgrad_f16x2_groups(const float* dy, const float* x, const float* dy_bound, long n_dy_bound,
                                        const float* x_rowmax, int groups, long rows, int dim_in, int dim_out, void* workspace,
                                        float* dW, mg_stream_t stream) {
    MG_REQUIRE(groups >= 1 && groups <= kFParts && dim_in % (4 * groups) == 0 && x_rowmax,
               "mg_tensor_linear_wgrad_f16x2_groups: groups of a multiple of four columns, and their row maxima");
    return wgrad_f16x2_one({dy, x, dy_bound, n_dy_bound, x_rowmax, rows * groups, rows, dim_in, dim_out, dW, nullptr}, groups, rows,
                           workspace, stream);
}

int mg_tensor_linear_wgrad_f16x2(const float* dy, const float* x, const float* dy_bound, long n_dy_bound,
                                 const float* x_bound, long n_x_bound, long rows, int dim_in, int dim_out,
                                 void* workspace, float* dW, float* db, mg_stream_t stream) {
    return mg_tensor_linear_wgrad_f16x2_rows(dy, x, dy_bound, n_dy_bound, x_bound, n_x_bound, rows, rows, dim_in, dim_out,
                                             workspace, dW, db, stream);
}

int mg_tensor_linear_wgrad_narrow_supported(int inds, long rows, int dim_in, int dim_out) {
    const int n = dim_in < dim_out ? dim_in : dim_out, dim = dim_in < dim_out ? dim_out : dim_in, T = inds == 0 ? 1 : inds == 1 ? 3 : 9;
    return inds >= 0 && inds <= 2 && rows >= 1 && rows < (1L << 31) && n >= 1 && n <= kNarrow && n * T <= 3 * kNarrow && dim % 4 == 0 &&
           dim >= 64 && dim >= 4 * n && dim <= 65536;
}

int mg_tensor_linear_wgrad_narrow_workspace_bytes(long rows, int dim_in, int dim_out, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && rows >= 0 && dim_in >= 1 && dim_out >= 1, "mg_tensor_linear_wgrad_narrow_workspace_bytes: bad argument");
    const NarrowPlan p = narrow_plan(rows > 0 ? rows : 1, dim_in, dim_out);
    *bytes = (size_t)p.splits * (p.plane + narrow_bias_floats(dim_in, dim_out)) * sizeof(float) + 16;
    return MG_OK;
}

int mg_tensor_linear_wgrad_narrow(int inds, const float* dy, const float* x, long rows, int dim_in, int dim_out, void* workspace,
                                  float* dW, float* db, mg_stream_t stream) {
    MG_REQUIRE(mg_tensor_linear_wgrad_narrow_supported(inds, rows, dim_in, dim_out),
               "mg_tensor_linear_wgrad_narrow: one dimension of at most 16 (5 in rank 2), the other of 64 or more, in fours");
    const bool of_x = dim_in < dim_out;                       // x is the narrow operand
    const float *narrow = of_x ? x : dy, *wide = of_x ? dy : x;
    MG_REQUIRE(dy && x && workspace && dW && aligned16(wide), "mg_tensor_linear_wgrad_narrow: null or unaligned pointer");
    hipStream_t st = (hipStream_t)stream;
    MG_REQUIRE(inds == 0 || db == nullptr, "mg_tensor_linear_wgrad_narrow: the bias gradient is defined for plain rows only");
    NarrowPlan p = narrow_plan(rows, dim_in, dim_out);
    if (db) p.plane += narrow_bias_floats(dim_in, dim_out);
    float* part = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t(15));
    const dim3 grid((unsigned)p.blocks, (unsigned)p.splits);
    const auto run = [&](auto kernel, int across) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, narrow, p.n, wide, p.dim, rows, p.rows, across, p.plane, part);
    };
    const auto of_width = [&](auto width) {
        constexpr int N = decltype(width)::value;
        if (inds == 1) run(wgrad_narrow_kernel<3, N>, p.lanes);
        else if constexpr (N <= 5) run(wgrad_narrow_kernel<9, N>, p.lanes);
    };
    if (inds == 0)
        run(db == nullptr ? wgrad_narrow_rows_kernel<kNoBias> : of_x ? wgrad_narrow_rows_kernel<kOfWide> : wgrad_narrow_rows_kernel<kOfNarrow>,
            p.waves_c);
    else if (p.n <= 1) of_width(std::integral_constant<int, 1>{});
    else if (p.n <= 2) of_width(std::integral_constant<int, 2>{});
    else if (p.n <= 4) of_width(std::integral_constant<int, 4>{});
    else if (p.n == 5) of_width(std::integral_constant<int, 5>{});
    else if (p.n <= 8) of_width(std::integral_constant<int, 8>{});
    else of_width(std::integral_constant<int, kNarrow>{});
    const int quads = (int)(p.plane / 4);
    hipLaunchKernelGGL(wgrad_narrow_reduce_kernel, dim3((unsigned)ceil_div(quads, 16)), dim3(256), 0, st,
                       reinterpret_cast<const float4*>(part), quads, (int)p.splits, p.dim, p.n, of_x, dim_out, dW, db);
    return check_launch("mg_tensor_linear_wgrad_narrow");
}

int mg_tensor_linear_wgrad(int inds, const float* dy, const float* x, long rows, int dim_in, int dim_out,
                           void* workspace, float* dW, mg_stream_t stream) {
    if (inds < 0 || inds > 2)
        return fail(MG_ERR_UNSUPPORTED, "tensor_linear currently only supports a number of indices up to 2.");
    MG_REQUIRE(rows >= 0 && dim_in >= 0 && dim_out >= 0, "mg_tensor_linear_wgrad: negative size");
    const long n = (long)dim_in * dim_out;
    if (n == 0) return MG_OK;
    MG_REQUIRE(dW != nullptr, "mg_tensor_linear_wgrad: dW is null");
    hipStream_t st = (hipStream_t)stream;
    const unsigned nblocks = (unsigned)(ceil_div(n, 256) < 1024 ? ceil_div(n, 256) : 1024);
    if (rows == 0) {
        hipLaunchKernelGGL(zero_f32_kernel, dim3(nblocks), dim3(256), 0, st, dW, n);
        return check_launch("mg_tensor_linear_wgrad");
    }
    MG_REQUIRE(dy && x && workspace, "mg_tensor_linear_wgrad: null pointer");
    long rpb, splits;
    const int tile = wgrad_tile(inds);
    wgrad_split(rows, dim_in, dim_out, tile, &rpb, &splits);
    float* part = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t(15));
    const int gx = (int)ceil_div(dim_out, tile), gy = (int)ceil_div(dim_in, tile);
    dim3 grid(gx, gy, (unsigned)splits), block(256);
    switch (inds) {
        case 0:
            if (dim_in % 4 == 0 && dim_out % 4 == 0 && aligned16(dy) && aligned16(x))
                hipLaunchKernelGGL(wgrad_mfma_lds_kernel, grid, block, 0, st, dy, x, rows, dim_in, dim_out, rpb, part);
            else
                hipLaunchKernelGGL(wgrad_mfma_kernel, grid, block, 0, st, dy, x, rows, dim_in, dim_out, rpb, part);
            break;
        case 1: hipLaunchKernelGGL(wgrad_kernel<3>, grid, block, 0, st, dy, x, rows, dim_in, dim_out, rpb, part); break;
        default: hipLaunchKernelGGL(wgrad_kernel<9>, grid, block, 0, st, dy, x, rows, dim_in, dim_out, rpb, part); break;
    }
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(nblocks), dim3(256), 0, st, (const float*)part, n, (int)splits, dW);
    return check_launch("mg_tensor_linear_wgrad");
}

}  // extern "C"
