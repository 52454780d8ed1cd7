// The 13 Cartesian products on node rows in component-major layout (node, comp, chan), for the
// self-interaction block (archs/diffuser_atoms15.py:59-95) of the bf16-storage configuration.
//
// Inputs  l0/r0 (N, chan), l1/r1 (N, 3, chan), l2/r2 (N, 9, chan)
// Outputs P0 (N, 3, chan)      labels 000, 110, 220
//         P1 (N, 3, 5, chan)   labels 011, 101, 121, 211, 111 per vector component
//         P2 (N, 9, 5, chan)   labels 022, 202, 112, 222, 212 per rank-2 component (xy -> 3x+y)
// i.e. the layout the edge kernel uses for its per-node sums, so the output linears of a rank are
// one GEMM with K = 3*chan or 5*chan.  A lane owns one (node, channel): every access of a wave is
// unit stride.  Bound by HBM: 26 values in, 63 out per (node, channel).
#include "common.hpp"
#include "rank2_linear.hpp"

namespace mg {
namespace {

template <typename T>
__global__ void __launch_bounds__(256) node_products_kernel(long n_nodes, int chan, const T* __restrict__ l0,
                                                            const T* __restrict__ l1, const T* __restrict__ l2,
                                                            const T* __restrict__ r0, const T* __restrict__ r1,
                                                            const T* __restrict__ r2, T* __restrict__ P0,
                                                            T* __restrict__ P1, T* __restrict__ P2,
                                                            float* __restrict__ node_max) {
    const long total = n_nodes * chan;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const long node = t / chan;
        const int c = (int)(t - node * chan);
        const float a = (float)l0[t], b = (float)r0[t];
        float u[3], v[3], L[9], R[9];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            u[x] = (float)l1[(node * 3 + x) * chan + c];
            v[x] = (float)r1[(node * 3 + x) * chan + c];
        }
#pragma unroll
        for (int k = 0; k < 9; k++) {
            L[k] = (float)l2[(node * 9 + k) * chan + c];
            R[k] = (float)r2[(node * 9 + k) * chan + c];
        }
        float dot = 0.f, ddot = 0.f;
#pragma unroll
        for (int x = 0; x < 3; x++) dot += u[x] * v[x];
#pragma unroll
        for (int k = 0; k < 9; k++) ddot += L[k] * R[k];
        T* p0 = P0 + (node * 3) * chan + c;
        p0[0] = (T)(a * b);
        p0[chan] = (T)dot;
        p0[2 * chan] = (T)ddot;
        float mx = fmaxf(fabsf(a * b), fmaxf(fabsf(dot), fabsf(ddot)));

        const float cr[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]};
#pragma unroll
        for (int x = 0; x < 3; x++) {
            T* p1 = P1 + ((node * 3 + x) * 5) * chan + c;
            p1[0] = (T)(a * v[x]);                                                      // 011
            p1[chan] = (T)(u[x] * b);                                                   // 101
            p1[2 * chan] = (T)(u[0] * R[3 * x] + u[1] * R[3 * x + 1] + u[2] * R[3 * x + 2]);   // 121: sum_k l_k r_{x k}
            p1[3 * chan] = (T)(L[3 * x] * v[0] + L[3 * x + 1] * v[1] + L[3 * x + 2] * v[2]);   // 211
            p1[4 * chan] = (T)cr[x];                                                    // 111
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(a * v[x]), fabsf(u[x] * b)), fabsf(cr[x])));
            mx = fmaxf(mx, fabsf(u[0] * R[3 * x] + u[1] * R[3 * x + 1] + u[2] * R[3 * x + 2]));
            mx = fmaxf(mx, fabsf(L[3 * x] * v[0] + L[3 * x + 1] * v[1] + L[3 * x + 2] * v[2]));
        }
#pragma unroll
        for (int x = 0; x < 3; x++) {
            // 212: row x of L crossed with v
            const float rc[3] = {L[3 * x + 1] * v[2] - L[3 * x + 2] * v[1], L[3 * x + 2] * v[0] - L[3 * x] * v[2],
                                 L[3 * x] * v[1] - L[3 * x + 1] * v[0]};
#pragma unroll
            for (int z = 0; z < 3; z++) {
                const int k = 3 * x + z;
                T* p2 = P2 + ((node * 9 + k) * 5) * chan + c;
                p2[0] = (T)(a * R[k]);                                                  // 022
                p2[chan] = (T)(L[k] * b);                                               // 202
                p2[2 * chan] = (T)(u[x] * v[z]);                                        // 112
                p2[3 * chan] = (T)(L[3 * x] * R[3 * z] + L[3 * x + 1] * R[3 * z + 1] + L[3 * x + 2] * R[3 * z + 2]);  // 222
                p2[4 * chan] = (T)rc[z];                                                // 212
                mx = fmaxf(mx, fmaxf(fmaxf(fabsf(a * R[k]), fabsf(L[k] * b)), fmaxf(fabsf(u[x] * v[z]), fabsf(rc[z]))));
                mx = fmaxf(mx, fabsf(L[3 * x] * R[3 * z] + L[3 * x + 1] * R[3 * z + 1] + L[3 * x + 2] * R[3 * z + 2]));
            }
        }
        if (node_max) {
            // chan is a multiple of 64 here, so a wave lies inside one node: one partial maximum
            // per (node, 64-channel chunk), a row bound for the GEMMs that read P0 / P1 / P2
            for (int d = 1; d < kWave; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
            if ((threadIdx.x & (kWave - 1)) == 0) node_max[node * (chan / kWave) + c / kWave] = mx;
        }
    }
}

// The adjoint on the same rows: both operands' gradients in one pass, a lane per (node, channel), 26 operand and 63 gradient values
// in, 26 out: bound by HBM (8192 rows, 256 channels: 0.21 ms, 4.6 TB/s).  With a kernel an operand on (row, chan, comp) arrays 0.32 ms,
// and the gradients of 13 linears to transpose before and after.  WITH_P2 false: the rank-2 products lead nowhere (the last block of a
// denoiser, whose rank-2 features are not read), and 45 of the 63 gradients are no zeros to be written first and read here (8192 rows with the writing of the zeros 270 -> 110 us).
template <bool WITH_P2>
__global__ void __launch_bounds__(256) node_products_grad_kernel(long n_nodes, int chan, const float* __restrict__ l0,
                                                                 const float* __restrict__ l1, const float* __restrict__ l2,
                                                                 const float* __restrict__ r0, const float* __restrict__ r1,
                                                                 const float* __restrict__ r2, const float* __restrict__ dP0,
                                                                 const float* __restrict__ dP1, const float* __restrict__ dP2,
                                                                 float* __restrict__ g_l0, float* __restrict__ g_l1,
                                                                 float* __restrict__ g_l2, float* __restrict__ g_r0,
                                                                 float* __restrict__ g_r1, float* __restrict__ g_r2) {
    const long total = n_nodes * chan;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const long node = t / chan;
        const int c = (int)(t - node * chan);
        const float a = l0[t], b = r0[t];
        float u[3], v[3], L[9], R[9];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            u[x] = l1[(node * 3 + x) * chan + c];
            v[x] = r1[(node * 3 + x) * chan + c];
        }
#pragma unroll
        for (int k = 0; k < 9; k++) {
            L[k] = l2[(node * 9 + k) * chan + c];
            R[k] = r2[(node * 9 + k) * chan + c];
        }
        const float* p0 = dP0 + (node * 3) * chan + c;
        const float g000 = p0[0], g110 = p0[chan], g220 = p0[2 * chan];
        float ga = g000 * b, gb = g000 * a, gu[3], gv[3], gL[9], gR[9], q111[3];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            gu[x] = g110 * v[x];
            gv[x] = g110 * u[x];
        }
#pragma unroll
        for (int k = 0; k < 9; k++) {
            gL[k] = g220 * R[k];
            gR[k] = g220 * L[k];
        }
#pragma unroll
        for (int x = 0; x < 3; x++) {
            const float* p1 = dP1 + ((node * 3 + x) * 5) * chan + c;
            const float q011 = p1[0], q101 = p1[chan], q121 = p1[2 * chan], q211 = p1[3 * chan];
            q111[x] = p1[4 * chan];
            ga += q011 * v[x];
            gv[x] += q011 * a;
            gb += q101 * u[x];
            gu[x] += q101 * b;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                gu[k] += q121 * R[3 * x + k];
                gR[3 * x + k] += q121 * u[k];
                gv[k] += q211 * L[3 * x + k];
                gL[3 * x + k] += q211 * v[k];
            }
        }
        // (l x r) . g: v x g for l, g x u for r
        gu[0] += v[1] * q111[2] - v[2] * q111[1];
        gu[1] += v[2] * q111[0] - v[0] * q111[2];
        gu[2] += v[0] * q111[1] - v[1] * q111[0];
        gv[0] += q111[1] * u[2] - q111[2] * u[1];
        gv[1] += q111[2] * u[0] - q111[0] * u[2];
        gv[2] += q111[0] * u[1] - q111[1] * u[0];
        if constexpr (WITH_P2)
#pragma unroll
        for (int x = 0; x < 3; x++) {
            float h[3];
#pragma unroll
            for (int z = 0; z < 3; z++) {
                const int k = 3 * x + z;
                const float* p2 = dP2 + ((node * 9 + k) * 5) * chan + c;
                const float q022 = p2[0], q202 = p2[chan], q112 = p2[2 * chan], q222 = p2[3 * chan];
                h[z] = p2[4 * chan];
                ga += q022 * R[k];
                gR[k] += q022 * a;
                gb += q202 * L[k];
                gL[k] += q202 * b;
                gu[x] += q112 * v[z];
                gv[z] += q112 * u[x];
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    gL[3 * x + j] += q222 * R[3 * z + j];
                    gR[3 * z + j] += q222 * L[3 * x + j];
                }
            }
            const float* l = L + 3 * x;                                                     // 212: row x of L crossed with v
            gL[3 * x] += v[1] * h[2] - v[2] * h[1];
            gL[3 * x + 1] += v[2] * h[0] - v[0] * h[2];
            gL[3 * x + 2] += v[0] * h[1] - v[1] * h[0];
            gv[0] += h[1] * l[2] - h[2] * l[1];
            gv[1] += h[2] * l[0] - h[0] * l[2];
            gv[2] += h[0] * l[1] - h[1] * l[0];
        }
        g_l0[t] = ga;
        g_r0[t] = gb;
#pragma unroll
        for (int x = 0; x < 3; x++) {
            g_l1[(node * 3 + x) * chan + c] = gu[x];
            g_r1[(node * 3 + x) * chan + c] = gv[x];
        }
#pragma unroll
        for (int k = 0; k < 9; k++) {
            g_l2[(node * 9 + k) * chan + c] = gL[k];
            g_r2[(node * 9 + k) * chan + c] = gR[k];
        }
    }
}

// The five rank-2 products of a node (labels 022, 202, 112, 222, 212) and the rank-2 output linear of SelfTensProds
// in one pass: a wave owns (node, 64-channel chunk), a lane one channel; the 45 product values stay in registers
// and go through rank2_linear_of_node_sums.  Reads the 26 operand rows of a node once (unit stride), writes
// (node, dim_d, 9); the products themselves are never stored.  For chan = 64, 128 or 256 and dim_d <= 16.
// 256 channels, 16 outputs, x_d of 16 channels: 775 us at 65 536 nodes, 85 at 8192, 24 at 2048 (870, 114 and 32 where the linear goes the
// way of fp32); with the linear on the fp32 matrix cores, x_d through LDS (a broadcast read costs as much as any other) and the scalar
// and vector products stored before the linear 860, 112 and 31.  What bounds it: a wave's chain of loads (of 775 us the linear takes
// 330, the rank-2 operands 180, the stores 175, and 300 are left without all three), beside 9 GB of weights from the L2.  A chunk's
// weights in LDS for eight nodes, the chunks of a node in turn: 753 us, but 31 at 2048 nodes, and 1030 with the stores at the end of a
// chunk, for want of registers; five waves a SIMD 994 us (35 spilled).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4)))
node_rank2_linear_kernel(long n_nodes, int chan, const float* __restrict__ l0,
                                                                const float* __restrict__ l1, const float* __restrict__ l2,
                                                                const float* __restrict__ r0, const float* __restrict__ r1,
                                                                const float* __restrict__ r2,
                                                                const float* __restrict__ y2_packed, int dim_d,
                                                                float* __restrict__ out, float* __restrict__ P0,
                                                                float* __restrict__ P1, float* __restrict__ node_max,
                                                                const float* __restrict__ x_d,
                                                                const float* __restrict__ L2t,
                                                                const float* __restrict__ R2t, int dim_in2, int split) {
    __shared__ __attribute__((aligned(16))) float rank2_lds[4 * kRank2Share];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int chunks = chan / kWave;
    const long items = n_nodes * chunks;
    long item = (long)blockIdx.x * 4 + wave;
    const bool valid = item < items;                           // uniform over the wave
    item = valid ? item : items - 1;
    const long node = item >> (chunks >> 1);                   // (1, 2 or 4 of them)
    const int chunk = (int)item & (chunks - 1);
    const int c = chunk * kWave + lane;
    float s2[45], lower[18];
    if (valid) {
        // x_d is read as scalars below, some lines at a time: all of them are asked for here, beside the other operands
        float touched[9];
        if (x_d) {
            const float* src = x_d + node * (long)(dim_in2 * 9);
#pragma unroll
            for (int t = 0; t < 9; t++) touched[t] = scalar_at(src + (16 * t < dim_in2 * 9 ? 16 * t : dim_in2 * 9 - 1));
        }
        const float a = l0[node * chan + c], b = r0[node * chan + c];
        float u[3], v[3], L[9], R[9];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            u[x] = l1[(node * 3 + x) * chan + c];
            v[x] = r1[(node * 3 + x) * chan + c];
        }
        if (x_d) {
            // the rank-2 operands are formed here: l2[k] = sum_i L2[c, i] x_d[node, i, k] (dim_in2 <= 16 input
            // channels; the node's 9 dim_in2 values are scalars of the wave, the weights come
            // transposed, (dim_in2, chan), one coalesced row per input channel).  Two GEMMs that would each write
            // (node, 9, chan) and this kernel's read of both are not needed.
            const float* src = x_d + node * (long)(dim_in2 * 9);
#pragma unroll
            for (int k = 0; k < 9; k++) { L[k] = 0.f; R[k] = 0.f; }
            // four input channels at a time, the weights of the next four requested before these are used (past the end: the last one's)
            float wl[4], wr[4];
            auto weights = [&](int i0) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int i = i0 + j < dim_in2 ? i0 + j : dim_in2 - 1;
                    wl[j] = L2t[(long)i * chan + c];
                    wr[j] = R2t[(long)i * chan + c];
                }
            };
            auto add = [&](int i, float w_l, float w_r) {
#pragma unroll
                for (int k = 0; k < 9; k++) {
                    const float xv = scalar_at(src + i * 9 + k);
                    L[k] = fmaf(w_l, xv, L[k]);
                    R[k] = fmaf(w_r, xv, R[k]);
                }
            };
            weights(0);
#pragma unroll
            for (int t = 0; t < 9; t++) asm volatile("" ::"s"(touched[t]));
            for (int i0 = 0; i0 < dim_in2; i0 += 4) {
                const float l[4] = {wl[0], wl[1], wl[2], wl[3]}, r[4] = {wr[0], wr[1], wr[2], wr[3]};
                weights(i0 + 4);
                if (i0 + 4 <= dim_in2) {
#pragma unroll
                    for (int j = 0; j < 4; j++) add(i0 + j, l[j], r[j]);
                } else {
#pragma unroll
                    for (int j = 0; j < 3; j++)
                        if (i0 + j < dim_in2) add(i0 + j, l[j], r[j]);
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < 9; k++) {
                L[k] = l2[(node * 9 + k) * chan + c];
                R[k] = r2[(node * 9 + k) * chan + c];
            }
        }
        // the scalar and vector products as well (stored below)
        lower[0] = a * b;
        lower[1] = u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
        lower[2] = 0.f;
#pragma unroll
        for (int k = 0; k < 9; k++) lower[2] += L[k] * R[k];
        const float cr[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]};
#pragma unroll
        for (int x = 0; x < 3; x++) {                          // 011 101 121 211 111
            lower[3 + 5 * x] = a * v[x];
            lower[4 + 5 * x] = u[x] * b;
            lower[5 + 5 * x] = u[0] * R[3 * x] + u[1] * R[3 * x + 1] + u[2] * R[3 * x + 2];
            lower[6 + 5 * x] = L[3 * x] * v[0] + L[3 * x + 1] * v[1] + L[3 * x + 2] * v[2];
            lower[7 + 5 * x] = cr[x];
        }
#pragma unroll
        for (int x = 0; x < 3; x++) {
            // 212: row x of L crossed with v
            const float rc[3] = {L[3 * x + 1] * v[2] - L[3 * x + 2] * v[1], L[3 * x + 2] * v[0] - L[3 * x] * v[2],
                                 L[3 * x] * v[1] - L[3 * x + 1] * v[0]};
#pragma unroll
            for (int z = 0; z < 3; z++) {
                const int k = 3 * x + z;
                s2[k * 5 + 0] = a * R[k];                                                                       // 022
                s2[k * 5 + 1] = L[k] * b;                                                                       // 202
                s2[k * 5 + 2] = u[x] * v[z];                                                                    // 112
                s2[k * 5 + 3] = L[3 * x] * R[3 * z] + L[3 * x + 1] * R[3 * z + 1] + L[3 * x + 2] * R[3 * z + 2];  // 222
                s2[k * 5 + 4] = rc[z];                                                                          // 212
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < 45; k++) s2[k] = 0.f;
#pragma unroll
        for (int k = 0; k < 18; k++) lower[k] = 0.f;
    }
    rank2_linear_of_node_sums<>(s2, split != 0, rank2_lds, chunk, chunks, valid, y2_packed, dim_d, out + node * (long)dim_d * 9);
    if (P0 && valid) {
        // In the layout of mg_bee_node_products with their maximum per (node, chunk): the operands are in registers once, and the
        // two GEMMs that follow read 18 chan floats per node instead of gathering 26 chan through their operand loads.  Behind everything
        // that loads: the queue of a wave completes in order, and a load behind these stores waits for memory to take them.
        float mx = 0.f;
#pragma unroll
        for (int k = 0; k < 18; k++) {
            float* to = k < 3 ? P0 + (node * 3 + k) * chan + c : P1 + (node * 15 + k - 3) * chan + c;
            __builtin_nontemporal_store(lower[k], to);
            mx = fmaxf(mx, fabsf(lower[k]));
        }
        if (node_max) {
            mx = wave_max_nonneg_last_lane(mx);
            if (lane == kWave - 1) node_max[node * chunks + chunk] = mx;
        }
    }
}

template <typename T>
int launch(const char* what, long n_nodes, int chan, const void* l0, const void* l1, const void* l2, const void* r0,
           const void* r1, const void* r2, void* P0, void* P1, void* P2, float* node_max, mg_stream_t stream) {
    MG_REQUIRE(n_nodes >= 0 && chan >= 0, "%s: negative size", what);
    MG_REQUIRE(node_max == nullptr || chan % kWave == 0, "%s: node_max needs chan to be a multiple of 64", what);
    if (n_nodes == 0 || chan == 0) return MG_OK;
    MG_REQUIRE(l0 && l1 && l2 && r0 && r1 && r2 && P0 && P1 && P2, "%s: null pointer", what);
    long blocks = ceil_div(n_nodes * chan, 256);
    if (blocks > 256L * 32) blocks = 256L * 32;
    hipLaunchKernelGGL(node_products_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, n_nodes,
                       chan, static_cast<const T*>(l0), static_cast<const T*>(l1), static_cast<const T*>(l2),
                       static_cast<const T*>(r0), static_cast<const T*>(r1), static_cast<const T*>(r2),
                       static_cast<T*>(P0), static_cast<T*>(P1), static_cast<T*>(P2), node_max);
    return check_launch(what);
}

}  // namespace
}  // namespace mg

using namespace mg;

namespace {
template <bool WITH_P2>
int node_products_grad(long n_nodes, int chan, const float* l0, const float* l1, const float* l2, const float* r0, const float* r1,
                       const float* r2, const float* d_P0, const float* d_P1, const float* d_P2, float* g_l0, float* g_l1, float* g_l2,
                       float* g_r0, float* g_r1, float* g_r2, mg_stream_t stream) {
    MG_REQUIRE(n_nodes >= 0 && chan > 0, "mg_bee_node_products_grad: bad size");
    if (n_nodes == 0) return MG_OK;
    MG_REQUIRE(l0 && l1 && l2 && r0 && r1 && r2 && d_P0 && d_P1 && g_l0 && g_l1 && g_l2 && g_r0 && g_r1 && g_r2,
               "mg_bee_node_products_grad: null pointer");
    const long blocks = ceil_div(n_nodes * chan, 256);
    hipLaunchKernelGGL(node_products_grad_kernel<WITH_P2>, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0,
                       (hipStream_t)stream, n_nodes, chan, l0, l1, l2, r0, r1, r2, d_P0, d_P1, d_P2, g_l0, g_l1, g_l2, g_r0, g_r1, g_r2);
    return check_launch("mg_bee_node_products_grad");
}
}  // namespace

extern "C" {

int mg_bee_node_products(long n_nodes, int chan, const float* l0, const float* l1, const float* l2, const float* r0,
                         const float* r1, const float* r2, float* P0, float* P1, float* P2, float* node_max,
                         mg_stream_t stream) {
    return launch<float>("mg_bee_node_products", n_nodes, chan, l0, l1, l2, r0, r1, r2, P0, P1, P2, node_max, stream);
}

int mg_bee_node_products_grad(long n_nodes, int chan, const float* l0, const float* l1, const float* l2, const float* r0,
                              const float* r1, const float* r2, const float* d_P0, const float* d_P1, const float* d_P2,
                              float* g_l0, float* g_l1, float* g_l2, float* g_r0, float* g_r1, float* g_r2, mg_stream_t stream) {
    MG_REQUIRE(n_nodes <= 0 || d_P2, "mg_bee_node_products_grad: null pointer");
    return node_products_grad<true>(n_nodes, chan, l0, l1, l2, r0, r1, r2, d_P0, d_P1, d_P2, g_l0, g_l1, g_l2, g_r0, g_r1, g_r2, stream);
}

int mg_bee_node_products_grad_lower(long n_nodes, int chan, const float* l0, const float* l1, const float* l2, const float* r0,
                                    const float* r1, const float* r2, const float* d_P0, const float* d_P1, float* g_l0, float* g_l1,
                                    float* g_l2, float* g_r0, float* g_r1, float* g_r2, mg_stream_t stream) {
    return node_products_grad<false>(n_nodes, chan, l0, l1, l2, r0, r1, r2, d_P0, d_P1, nullptr, g_l0, g_l1, g_l2, g_r0, g_r1, g_r2, stream);
}

int mg_bee_node_products_rank2(long n_nodes, int chan, const float* l0, const float* l1, const float* l2,
                               const float* r0, const float* r1, const float* r2, const float* packed_Y2, int dim_d,
                               float* out_d, float* P0, float* P1, float* node_max, const float* x_d,
                               const float* L2t, const float* R2t, int dim_in2, mg_stream_t stream) {
    MG_REQUIRE((P0 == nullptr) == (P1 == nullptr) && (node_max == nullptr || P0 != nullptr),
               "mg_bee_node_products_rank2: P0 and P1 go together, node_max with them");
    MG_REQUIRE(x_d == nullptr || (L2t && R2t && dim_in2 >= 1 && dim_in2 <= 16),
               "mg_bee_node_products_rank2: x_d needs both transposed weights and 1 .. 16 input channels");

    MG_REQUIRE(n_nodes >= 0, "mg_bee_node_products_rank2: negative size");
    MG_REQUIRE(rank2_fusable(chan, dim_d), "mg_bee_node_products_rank2: needs chan = 64, 128 or 256 and dim_d <= 16");
    if (n_nodes == 0) return MG_OK;
    MG_REQUIRE(l0 && l1 && r0 && r1 && packed_Y2 && out_d && aligned16(packed_Y2),
               "mg_bee_node_products_rank2: null or unaligned pointer");
    MG_REQUIRE(x_d != nullptr || (l2 && r2), "mg_bee_node_products_rank2: l2 and r2, or x_d and the weights");
    const long blocks = ceil_div(n_nodes * (chan / kWave), 4);
    MG_REQUIRE(blocks < (1L << 31), "mg_bee_node_products_rank2: too many nodes for one launch");
    hipLaunchKernelGGL(node_rank2_linear_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, n_nodes,
                       chan, l0, l1, l2, r0, r1, r2, packed_Y2, dim_d, out_d, P0, P1, node_max, x_d, L2t, R2t, dim_in2,
                       mg_get_linear_mode() == kLinearF16x2);
    return check_launch("mg_bee_node_products_rank2");
}

int mg_bee_node_products_bf16(long n_nodes, int chan, const void* l0, const void* l1, const void* l2, const void* r0,
                              const void* r1, const void* r2, void* P0, void* P1, void* P2, mg_stream_t stream) {
    return launch<__bf16>("mg_bee_node_products_bf16", n_nodes, chan, l0, l1, l2, r0, r1, r2, P0, P1, P2, nullptr, stream);
}

}  // extern "C"
