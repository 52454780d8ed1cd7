// The per-edge chain of the rank-0/1/2 messages on bf16 storage (archs/diffuser_atoms15.py:98-110, 244-246),
// for the two sums over edges that the node-side layers need:
//     psi = Y P0                      (edges, 128)      -> sum over the edges of each node of bf16(psi)
//     h1  = act(W1 psi + b1)          (edges, 256)
//     h2  = act(W2 h1 + b2)           (edges, 256)      -> sum over the edges of each node of bf16(h2)
// in ONE kernel: psi and h1 stay in LDS, h2 in registers; each is rounded to bf16 exactly where the separate kernels round it when
// they store.  x = P0 is the only per-row tensor read, the sums the only output.  Weights are two bf16 planes (16 significand bits).
//
// A workgroup takes 128 rows through the three layers, two workgroups to a CU.  Activations lie in LDS in the order the matrix cores
// read them (fragment_at); a wave owns 32 output columns and reads the fragments of its weights straight from memory: a step of 16 k
// is two contiguous kilobytes of the L2 and feeds eight matrix instructions, and no barrier stands in the loop over k of the hidden
// layers.  Where rows are the first operand (psi, h2) a lane of the product holds rows of one column, which a segment's sum adds up in
// a register; where they are the second (h1) channels of one row, the next layer's operand sixteen bytes at a time.
//
// 5.9 M rows of 384 with 90 to a segment 3.59 ms, 180 000 rows 0.125 ms; with psi, h1 and h2 in the registers of one wave per 32 rows
// and the weights through LDS (two fragments read for two matrix instructions, a barrier for every 32 k) 4.11 and 0.134 ms.  What
// bounds it: the board's power.  It takes 22 % fewer cycles than that kernel, the matrix cores are busy for half of them (0.97 PFLOP/s,
// counting both planes), and the clock falls from 2.1 to 1.84 GHz.  64 columns to a wave and half the waves, a third less read for a
// matrix instruction: 3.85 ms.  Writers of a row meeting in one bank (fragment_at without its turn): 3.66 ms.
#include "common.hpp"
#include "rowsum_finish.hpp"

namespace mg {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kD = 128, kH = 256;
constexpr int kBlocks = 4, kRows = 32 * kBlocks, kThreads = 512;  // row blocks and rows of a workgroup
constexpr int kStage = 128, kStageBlock = 32 * kStage;            // k of x in LDS at a time; elements of a row block's part of it
constexpr int kStageElems = kRows * kStage;                       // (psi has the place of a stage, h1 that of both)
constexpr int kStep = 2 * 64 * 8;                                 // elements of a weight's fragments for 16 k: two planes
// Widest Y that the workspace has room for in fragments, 4 MB of it.  Read from its planes, a line for every row, Y takes 16 384 rows of
// 1056 54 us and 100 000 175, in fragments 47 and 134; of 2048 92 and 353, 66 and 231.  (From 3072 columns on the weights, read for every
// 128 rows, make some row counts slower than the kernel before, which read them for 256: 40 000 rows of 3072 143 us, there 130.)
constexpr int kPackedDimIn = 8192;

template <int ACT>
__device__ __forceinline__ float activate_c(float v) {
    if constexpr (ACT == 1) return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    if constexpr (ACT == 2) return v > 0.f ? v : 0.1f * v;
    return v;
}

// Element (row, k) of a row block: chunks of 32 k, in each two steps of 16, 8 consecutive k to a lane.  The four pieces of 8 k of a
// chunk lie 512 bytes apart: the last two bits of the row are turned by the piece, so that writers of one row meet different banks.
__device__ __forceinline__ int piece_of(int k) { return ((k >> 3) & 1) + 2 * ((k >> 4) & 1); }
__device__ __forceinline__ int fragment_at(int row, int k) {
    return (((k >> 5) * 2 + ((k >> 3) & 1)) * 64 + (row ^ piece_of(k)) + 32 * ((k >> 4) & 1)) * 8 + (k & 7);
}
// The k at which channel ch of psi and h1 stands, in the order that mg_mlp_chain_bf16 asks W1 and W2 for: a lane half of the matrix core
// holds channels 8 i + 4 G .. + 3 of a chunk, eight of which in a row are one piece of 16 bytes.
__device__ __forceinline__ int operand_k(int ch) { return (ch & ~31) + 16 * ((ch >> 2) & 1) + 4 * ((ch >> 3) & 3) + (ch & 3); }

// The two planes of a packed weight (rows of I) into fragments: [32 rows][16 k][plane][lane][8]
struct Repack {
    const __bf16* from;
    long plane;
    int rows, I;
    __bf16* to;
};
struct RepackAll {
    Repack w[3];
};
__global__ void __launch_bounds__(256) mlp_chain_repack_kernel(const RepackAll all) {
    const Repack w = all.w[blockIdx.y];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;           // of rows I / 4: eight elements each
    if (t >= (long)w.rows * w.I / 4) return;
    const int lane = (int)(t & 63), plane = (int)(t >> 6) & 1, steps = w.I / 16;
    const long step = t >> 7;
    const int row = 32 * (int)(step / steps) + (lane & 31), s = (int)(step % steps);
    const __bf16* from = w.from + plane * w.plane + (long)row * w.I + 32 * (s >> 1) + 16 * (lane >> 5) + 8 * (s & 1);
    *reinterpret_cast<bf16x8*>(w.to + 8 * t) = *reinterpret_cast<const bf16x8*>(from);
}

// acc[mi] += rows of block mi (from LDS) times 32 weight rows, a step of 16 k at a time; the weights of two steps are in flight.
// ROWS_FIRST: a lane of acc is a column and its registers are rows 8 (q / 4) + 4 (lane / 32) + q % 4; else a row and its channels.
// PLANES: the weight is read from its planes of rows, a line for every row: Y where the workspace has no room for its fragments.
template <int MI, bool ROWS_FIRST, bool PLANES = false>
struct Product {
    floatx16 acc[MI];
    const __bf16* w;
    int steps, next;
    unsigned lane_at;
    long low;
    bf16x8 wh[2], wl[2];
    __device__ __forceinline__ void load_w(int u) {
        const int s = next < steps ? next : steps - 1;             // (surplus loads at the end are never used)
        const __bf16* p = w + (PLANES ? 32L * (s >> 1) + 8 * (s & 1) : (long)kStep * s);
        wh[u] = *reinterpret_cast<const bf16x8*>(p + lane_at);
        wl[u] = *reinterpret_cast<const bf16x8*>(p + low + lane_at);
        next++;
    }
    // block: which 32 rows of the weight
    __device__ __forceinline__ void start(const __bf16* weight, long plane, int block, int K) {
        const int lane = threadIdx.x & 63;
        steps = K / 16;
        next = 0;
        w = weight + (long)block * (PLANES ? 32 * K : kStep * steps);
        lane_at = PLANES ? (unsigned)((lane & 31) * K + 16 * (lane >> 5)) : 8u * lane;
        low = PLANES ? plane : kStep / 2;
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int q = 0; q < 16; q++) acc[mi][q] = 0.f;
        load_w(0);
        load_w(1);
    }
    __device__ __forceinline__ void run(const __bf16* x, int block_elems, int n) {      // n steps, an even number
        const int lane = threadIdx.x & 63;
        const __bf16* const at[2] = {x + fragment_at(lane & 31, 16 * (lane >> 5)), x + fragment_at(lane & 31, 16 * (lane >> 5) + 8)};   // of even and odd steps
        bf16x8 b[MI];
#pragma unroll
        for (int mi = 0; mi < MI; mi++) b[mi] = *reinterpret_cast<const bf16x8*>(at[0] + mi * block_elems);
        for (int s = 0; s < n; s += 2) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int chunk = u && s + 2 < n ? s + 2 : s;          // (the last trip reads its own chunk again)
#pragma unroll
                for (int pair = 0; pair < MI; pair += 2) {
                    __builtin_amdgcn_sched_barrier(0);             // keep this issue order
#pragma unroll
                    for (int mi = pair; mi < pair + 2; mi++) acc[mi] = product(wl[u], b[mi], acc[mi]);   // small terms first
#pragma unroll
                    for (int mi = pair; mi < pair + 2; mi++) acc[mi] = product(wh[u], b[mi], acc[mi]);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int mi = pair; mi < pair + 2; mi++)
                        b[mi] = *reinterpret_cast<const bf16x8*>(at[1 - u] + mi * block_elems + 512 * chunk);
                }
                load_w(u);
            }
        }
    }
    static __device__ __forceinline__ floatx16 product(const bf16x8& w, const bf16x8& x, const floatx16& c) {
        return ROWS_FIRST ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, w, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, c, 0, 0, 0);
    }
};

// The sums over the rows of each segment, column `col`: v[half][q] are the lane's rows of two blocks as Product has them with
// ROWS_FIRST.  Two partial slots per block of 32 rows (rowsum_finish.hpp); runs strictly inside a block are written to `out`.
// After the halves have changed places lanes 0 .. 31 hold all rows of the first block and lanes 32 .. 63 those of the second, and a
// segment's rows add up in row order.
__device__ __forceinline__ void sum_segments(float (&v)[2][16], long first_block, long R, const int* __restrict__ seg, int O, int col,
                                             float* __restrict__ slots, long n_blocks, float* __restrict__ out) {
    const int lane = threadIdx.x & 63, m = lane & 31, G = lane >> 5;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0][q]), __float_as_uint(v[1][q]), false, false);
        v[0][q] = __uint_as_float(s[0]);                           // row 8 (q / 4) + q % 4 of block G
        v[1][q] = __uint_as_float(s[1]);                           // row 8 (q / 4) + 4 + q % 4
    }
    const long r0 = 32 * first_block, left = R - r0 - 32 * G, block = first_block + G;
    const int rows = left < 32 ? (int)left : 32;                   // of this half's block; none if <= 0
    if (r0 + 64 > R) {
#pragma unroll
        for (int r = 0; r < 32; r++) v[r >> 2 & 1][4 * (r >> 3) + (r & 3)] = r < rows ? v[r >> 2 & 1][4 * (r >> 3) + (r & 3)] : 0.f;
    }
    const int my_seg = seg[r0 + lane < R ? r0 + lane : R - 1], before = __shfl_up(my_seg, 1);
    const unsigned long long starts = __ballot(m > 0 && my_seg != before);
    float* const slot = slots + (block < n_blocks ? block : 0) * O + col;
    float* to = slot;                                              // of a block's first run; later ones lie inside the block
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 32; r++) {
        if (r > 0 && (starts >> r & 0x100000001ull)) {
            const int s_lo = __builtin_amdgcn_readlane(my_seg, r), s_hi = __builtin_amdgcn_readlane(my_seg, 32 + r);
            if (starts >> (r + 32 * G) & 1) {                      // (never at a row past the end: those repeat the last one)
                *to = sum;
                sum = 0.f;
                to = out + (long)(G ? s_hi : s_lo) * O + col;
            }
        }
        sum += v[r >> 2 & 1][4 * (r >> 3) + (r & 3)];
    }
    if (rows <= 0) return;
    if (to != slot && rows == 32) to = slots + (n_blocks + block) * O + col;
    *to = sum;
}

template <int ACT, bool Y_PLANES>
__global__ void __launch_bounds__(kThreads, 4)
mlp_chain_bf16_kernel(const __bf16* __restrict__ X, long R, int I, const __bf16* __restrict__ Wa, long plane_a,
                      const __bf16* __restrict__ Wb, const float* __restrict__ bias_b, const __bf16* __restrict__ Wc,
                      const float* __restrict__ bias_c, const int* __restrict__ seg, float* __restrict__ slots_x,
                      float* __restrict__ slots_h, long n_blocks, float* __restrict__ out_x, float* __restrict__ out_h,
                      long tiles_total) {
    __shared__ __attribute__((aligned(16))) __bf16 lds[2 * kStageElems];
    static_assert(kRows * kH == 2 * kStageElems && kRows * kD == kStageElems, "the layers' places");

    const long bid = blockIdx.x;
    const long per_xcd = (tiles_total + 7) / 8;
    const long tile = (bid % 8) * per_xcd + bid / 8;
    if (tile >= tiles_total) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 31, G = lane >> 5;
    const long block0 = tile * kBlocks;

    // ---- psi = Y x: wave = 32 columns of two row blocks; x by stages of 128 k, the next one in registers
    const int cb = wave & 3, half = wave >> 2;
    {
        Product<2, true, Y_PLANES> y;
        y.start(Wa, plane_a, cb, I);
        // a quarter of a row's pieces of 8 k to a thread; two rows of eight threads are four apart (fragment_at)
        const int row = (tid >> 2 & 0x78) + (tid >> 2 & 1) * 4 + (tid >> 3 & 3);
        const long my_row = block0 * 32 + row;
        const __bf16* from = X + (my_row < R ? my_row : R - 1) * I + 8 * (tid & 3);
        __bf16* to = lds + (row >> 5) * kStageBlock + fragment_at(row & 31, 8 * (tid & 3));
        bf16x8 piece[4];
        auto load = [&](int k0) {                                  // chunk j of the stage (past the end: the last one again)
#pragma unroll
            for (int j = 0; j < 4; j++) piece[j] = *reinterpret_cast<const bf16x8*>(from + (k0 + 32 * j < I ? k0 + 32 * j : I - 32));
        };
        load(0);
        for (int k0 = 0, at = 0; k0 < I; k0 += kStage, at = kStageElems - at) {
#pragma unroll
            for (int j = 0; j < 4; j++) *reinterpret_cast<bf16x8*>(to + at + 1024 * j) = piece[j];
            if (k0 + kStage < I) load(k0 + kStage);
            __syncthreads();
            const int left = I - k0;
            y.run(lds + at + 2 * half * kStageBlock, kStageBlock, (left < kStage ? left : kStage) / 16);
        }
        __syncthreads();                                           // (the last stage may lie where psi goes)
        __bf16* psi[4];                                            // of rows q % 4
#pragma unroll
        for (int i = 0; i < 4; i++) psi[i] = lds + 2 * half * kStageBlock + fragment_at(4 * G + i, operand_k(32 * cb + m));
        float v[2][16];
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const __bf16 r = (__bf16)y.acc[mi][q];
                psi[q % 4][mi * kStageBlock + 64 * (q / 4)] = r;
                v[mi][q] = (float)r;
            }
        sum_segments(v, block0 + 2 * half, R, seg, kD, 32 * cb + m, slots_x, n_blocks, out_x);
    }
    __syncthreads();

    // ---- h1 = act(W1 psi + b1): wave = 32 columns of all rows
    {
        Product<kBlocks, false> h;
        h.start(Wb, 0, wave, kD);
        h.run(lds, kStageBlock, kD / 16);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; t++) {                              // channels 16 t + 8 (j / 4) + 4 G + j % 4 of the wave's 32
            const int col = 32 * wave + 16 * t + 4 * G;
            float b[8];
#pragma unroll
            for (int j = 0; j < 8; j++) b[j] = bias_b[col + 8 * (j / 4) + j % 4];
#pragma unroll
            for (int mi = 0; mi < kBlocks; mi++) {
                bf16x8 v;
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = (__bf16)activate_c<ACT>(h.acc[mi][8 * t + j] + b[j]);
                *reinterpret_cast<bf16x8*>(lds + mi * 32 * kH + fragment_at(m, operand_k(col))) = v;
            }
        }
    }
    __syncthreads();

    // ---- h2 = act(W2 h1 + b2), only its sums per node leave the kernel
    Product<kBlocks, true> h;
    h.start(Wc, 0, wave, kH);
    h.run(lds, 32 * kH, kH / 16);
    const int col = 32 * wave + m;
    const float b = bias_c[col];
#pragma unroll
    for (int pair = 0; pair < kBlocks; pair += 2) {
        float v[2][16];
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int q = 0; q < 16; q++) v[mi][q] = (float)(__bf16)activate_c<ACT>(h.acc[pair + mi][q] + b);
        sum_segments(v, block0 + pair, R, seg, kH, col, slots_h, n_blocks, out_h);
    }
}

}  // namespace
}  // namespace mg

using namespace mg;

// fragments of W1, W2 and, where it is no wider than kPackedDimIn, Y
static long chain_weight_elems(int dim_in) { return 2L * kH * kD + 2L * kH * kH + (dim_in <= kPackedDimIn ? 2L * kD * dim_in : 0); }

extern "C" {

int mg_mlp_chain_bf16_workspace_bytes(long rows, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && rows >= 0, "mg_mlp_chain_bf16_workspace_bytes: bad argument");
    *bytes = (size_t)(2L * (ceil_div(rows, 32) + 1) * (kD + kH)) * sizeof(float) + chain_weight_elems(kPackedDimIn) * sizeof(__bf16);
    return MG_OK;
}

int mg_mlp_chain_bf16(const void* x, long rows, int dim_in, const void* packed_Y, const void* packed_W1,
                      const float* b1, const void* packed_W2, const float* b2, int act, const int* row_ptr,
                      const int* seg, long n_out, void* workspace, float* sum_psi, float* sum_h2, mg_stream_t stream) {
    MG_REQUIRE(dim_in >= 32 && dim_in % 32 == 0, "mg_mlp_chain_bf16: dim_in must be a multiple of 32 (got %d)", dim_in);
    MG_REQUIRE(rows >= 0 && n_out >= 0 && rows < (1L << 31) && n_out < (1L << 31), "mg_mlp_chain_bf16: bad size");
    MG_REQUIRE(act >= 0 && act <= 2, "mg_mlp_chain_bf16: unknown activation %d", act);
    if (n_out == 0) return MG_OK;
    MG_REQUIRE(packed_Y && packed_W1 && packed_W2 && row_ptr && sum_psi && sum_h2 && workspace && aligned16(packed_Y) &&
                   aligned16(packed_W1) && aligned16(packed_W2) && aligned16(workspace) && aligned16(sum_psi) &&
                   aligned16(sum_h2),
               "mg_mlp_chain_bf16: null or unaligned operand");
    hipStream_t st = (hipStream_t)stream;
    const long n_blocks = ceil_div(rows, 32);
    __bf16* const w1 = static_cast<__bf16*>(workspace);
    __bf16* const w2 = w1 + 2L * kH * kD;
    __bf16* const y = w2 + 2L * kH * kH;
    float* slots_x = reinterpret_cast<float*>(w1 + chain_weight_elems(kPackedDimIn));
    float* slots_h = slots_x + 2L * (n_blocks + 1) * kD;
    if (rows > 0) {
        MG_REQUIRE(x && seg && b1 && b2 && aligned16(x), "mg_mlp_chain_bf16: null or unaligned row operand");
        const long tiles = ceil_div(rows, kRows);
        const long grid = ceil_div(tiles, 8) * 8;
        MG_REQUIRE(grid <= 0x7fffffffL, "mg_mlp_chain_bf16: grid too large");
        // packed weights: planes of ceil(dim_out / 128) * 128 rows.  Their fragments are formed on every call: 5 us
        const bool planes = dim_in > kPackedDimIn;
        const __bf16 *from_y = static_cast<const __bf16*>(packed_Y), *from_1 = static_cast<const __bf16*>(packed_W1),
                     *from_2 = static_cast<const __bf16*>(packed_W2);
        const RepackAll all{{{from_1, (long)kH * kD, kH, kD, w1}, {from_2, (long)kH * kH, kH, kH, w2}, {from_y, (long)kD * dim_in, kD, dim_in, y}}};
        const long most = planes || dim_in < 2 * kH ? (long)kH * kH / 4 : (long)kD * dim_in / 4;
        mlp_chain_repack_kernel<<<dim3((unsigned)ceil_div(most, 256), planes ? 2 : 3), dim3(256), 0, st>>>(all);
        if (int code = check_launch("mlp_chain_repack_kernel")) return code;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kThreads), 0, st, static_cast<const __bf16*>(x), rows, dim_in,
                               planes ? from_y : y, (long)kD * dim_in, w1, b1, w2, b2, seg, slots_x, slots_h, n_blocks, sum_psi,
                               sum_h2, tiles);
        };
        if (act == 1) planes ? launch(mlp_chain_bf16_kernel<1, true>) : launch(mlp_chain_bf16_kernel<1, false>);
        else if (act == 2) planes ? launch(mlp_chain_bf16_kernel<2, true>) : launch(mlp_chain_bf16_kernel<2, false>);
        else planes ? launch(mlp_chain_bf16_kernel<0, true>) : launch(mlp_chain_bf16_kernel<0, false>);
        if (int code = check_launch("mlp_chain_bf16_kernel")) return code;
    }
    rowsum_finish_kernel<<<dim3((unsigned)ceil_div(n_out * (kD / 4), 256)), dim3(256), 0, st>>>(
        row_ptr, n_out, n_blocks, kD, slots_x, 1.0f, sum_psi);
    if (int code = check_launch("rowsum_finish_kernel")) return code;
    rowsum_finish_kernel<<<dim3((unsigned)ceil_div(n_out * (kH / 4), 256)), dim3(256), 0, st>>>(
        row_ptr, n_out, n_blocks, kH, slots_h, 1.0f, sum_h2);
    return check_launch("rowsum_finish_kernel");
}

}  // extern "C"
