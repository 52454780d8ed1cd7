// The three maps l, r, v of PaiNN's Update (archs/meanflow_painn8.py:63-75) and what is made of the first two, in one kernel, in the
// split-fp16 arithmetic of f16x2.hpp: ip = l . r and |r| per channel, [x_a | |r|] with its row maxima, and v.
//
// A workgroup takes the 96 (node, component) rows of 32 nodes, one block of 32 rows a component, so that in the product (weight as
// the A operand) a lane holds all three components of the same channels of one node: the sums over components need no exchange,
// and l and r, two thirds of the maps' output, are not stored.  Wave w owns channels [32 w, + 32) of the three maps, l and r
// together and then v: 96 sums in two sets of accumulators (the small products apart) within 256 registers.
// Bound by memory in part (16 336 nodes of 128 channels: 83 MB, 18 us) and by what a workgroup does in turn: loads, split, products,
// stores.  Transposition to rows, a linear with component rows and a pass over (rows, 3, 3n) / this kernel, us: 128 channels 1280
// nodes 17.2 / 14.9, 5120 31 / 18, 16 336 65 / 30, 40 000 147 / 71; 64 channels 12.0 / 12.1, 21 / 13, 39 / 19, 73 / 37; 256 channels
// 29 / 30, 51 / 39, 143 / 85, 343 / 222.  Up to 128 channels the kernel for few nodes, below, takes up to 8192 of them.  Of wider rows a
// kernel of ten workgroups takes longer than three launches (320 nodes 16 / 28): the caller's line is at 1280 nodes, and at 2304 for 256
// channels, whose workgroups are alone on a CU.  The whole update, both ways: 224 channels 87.5 / 84.6 at 1280; 256 channels 85 / 92 at 1280,
// 102.5 / 104 at 2048, 136.2 / 136.0 at 2304, 146 / 143.5 at 3072.
#include "common.hpp"
#include "rows_in_lds.hpp"

namespace mg {
namespace {

constexpr int kNodes = 32, kMaxN = 256;

struct UpdateMaps {
    const float *x_v, *x_a;
    long rows;
    int n;
    const _Float16* planes;        // of the three maps below one another, (3n, n)
    const float* inv;
    float *ip, *cat, *cat_max, *v;
};

__global__ void __launch_bounds__(64 * kMaxN / 32, 2) painn_update_maps_kernel(const UpdateMaps a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int n = a.n, x_lo = 3 * kNodes * n, waves = n / 32;
    _Float16* const xh = reinterpret_cast<_Float16*>(lds);
    float* const row_max = reinterpret_cast<float*>(lds + (size_t)3 * kNodes * n * 4);   // [3][32]
    float* const top = row_max + 3 * kNodes;                                              // [1 + waves][32], of x_a and |r|
    float* const fixed = top + (1 + kMaxN / 32) * kNodes;                                 // [3 n]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 31, G = lane >> 5;
    const long r0 = (long)blockIdx.x * kNodes;
    const bool marked = has_marks(a.inv, 3 * n, lane);
    // rows past the end repeat the last one and are not written
    auto row_of = [&](int mm) { return r0 + mm < a.rows ? r0 + mm : a.rows - 1; };

    for (int grp = wave; grp < kNodes / 8; grp += waves) {         // eight lanes to a node, four channels at a time
        const int mm = grp * 8 + (lane >> 3), p = lane & 7;
        const long row = row_of(mm);
        const bool live = r0 + mm < a.rows;
        float f[kMaxN / 32][12], mx[3] = {0.f, 0.f, 0.f}, ma = 0.f;
#pragma unroll
        for (int j = 0; j < kMaxN / 32; j++)
            if (32 * j < n) {
                const float4* src = reinterpret_cast<const float4*>(a.x_v + (row * n + 32 * j + 4 * p) * 3);
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const float4 t = src[k];
                    f[j][4 * k] = t.x; f[j][4 * k + 1] = t.y; f[j][4 * k + 2] = t.z; f[j][4 * k + 3] = t.w;
                }
            }
#pragma unroll
        for (int j = 0; j < kMaxN / 32; j++)
            if (32 * j < n) {
                const float4 t = *reinterpret_cast<const float4*>(a.x_a + row * n + 32 * j + 4 * p);
                if (live) *reinterpret_cast<float4*>(a.cat + row * 2 * n + 32 * j + 4 * p) = t;
                ma = fmaxf(fmaxf(fmaxf(ma, fabsf(t.x)), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w)));
#pragma unroll
                for (int k = 0; k < 12; k++) mx[k % 3] = fmaxf(mx[k % 3], fabsf(f[j][k]));
            }
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) {
            ma = fmaxf(ma, __shfl_xor(ma, d));
#pragma unroll
            for (int x = 0; x < 3; x++) mx[x] = fmaxf(mx[x], __shfl_xor(mx[x], d));
        }
        if (p == 0) top[mm] = ma;
#pragma unroll
        for (int x = 0; x < 3; x++) {
            float inv;
            const float scale = pow2_scale(mx[x], &inv);
            const bool bits = marked || beyond_split(mx[x]);
#pragma unroll
            for (int j = 0; j < kMaxN / 32; j++)
                if (32 * j < n) {
                    const float v[4] = {f[j][x], f[j][3 + x], f[j][6 + x], f[j][9 + x]};
                    const int at = x * kNodes * n + piece_at(mm, 32 * j + 4 * p);
                    if (bits) store_bits(xh, x_lo, at, v);
                    else store_pieces(xh, x_lo, at, v, scale);
                }
            if (p == 0) row_max[x * kNodes + mm] = mx[x];
        }
    }
    __syncthreads();
    float isx[3];
    bool odd[3], any_odd = false;
#pragma unroll
    for (int x = 0; x < 3; x++) {
        const float mx = row_max[x * kNodes + m];
        pow2_scale(mx, &isx[x]);
        odd[x] = marked || beyond_split(mx);
        any_odd |= __any(odd[x]);
    }
    const long w_lo = (long)pad256(3 * n) * n;
    const long row = row_of(m);
    const bool live = r0 + m < a.rows;
    const _Float16* w = a.planes + (long)wave * (n >> 5) * 1024;
    // rows that the pieces cannot carry (all waves see the same ones): their sums for maps [first, first + NI)
    auto finish = [&](auto& acc, int first) {
        constexpr int NI = sizeof(acc[0]) / sizeof(floatx16);
#pragma unroll
        for (int x = 0; x < 3; x++) {
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const float4 w4 = *reinterpret_cast<const float4*>(a.inv + (first + ni) * n + 32 * wave + 8 * t + 4 * G);
                    const float iw[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[x][ni][4 * t + i] = acc[x][ni][4 * t + i] * isx[x] * iw[i];
                }
            if (!any_odd) continue;
            unsigned rows = (unsigned)__ballot(odd[x]);
            while (rows) {
                const int r = __builtin_ctz(rows);
                rows &= rows - 1;
                for (int c = tid; c < NI * n; c += blockDim.x)
                    fixed[c] = lds_row_in_fp32(xh + x * kNodes * n, x_lo, r, a.planes, w_lo, first * n + c, n, a.inv[first * n + c]);
                __syncthreads();
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
#pragma unroll
                    for (int q = 0; q < 16; q++) {
                        const float f = fixed[ni * n + 32 * wave + 8 * (q / 4) + 4 * G + q % 4];
                        if (m == r) acc[x][ni][q] = f;
                    }
                __syncthreads();
            }
        }
    };
    {
        floatx16 acc[3][2];
        multiply<3, 2, 1>(w, w_lo, n, xh, kNodes * n, x_lo, lane, acc, waves);
        finish(acc, 0);
        float mr = 0.f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int c = 32 * wave + 8 * t + 4 * G;
            float ip[4], nr[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int q = 4 * t + i;
                const float x = acc[0][1][q], y = acc[1][1][q], z = acc[2][1][q];
                ip[i] = acc[0][0][q] * x + acc[1][0][q] * y + acc[2][0][q] * z;
                nr[i] = sqrtf(x * x + y * y + z * z);
                mr = fmaxf(mr, nr[i]);
            }
            if (live) {
                *reinterpret_cast<float4*>(a.ip + row * n + c) = make_float4(ip[0], ip[1], ip[2], ip[3]);
                *reinterpret_cast<float4*>(a.cat + row * 2 * n + n + c) = make_float4(nr[0], nr[1], nr[2], nr[3]);
            }
        }
        mr = fmaxf(mr, __shfl_xor(mr, 32));
        if (G == 0) top[(1 + wave) * kNodes + m] = mr;
    }
    {
        floatx16 acc[3][1];
        multiply<3, 1, 1>(w + 2L * waves * (n >> 5) * 1024, w_lo, n, xh, kNodes * n, x_lo, lane, acc);
        finish(acc, 2);
        if (live)
#pragma unroll
            for (int x = 0; x < 3; x++)
#pragma unroll
                for (int t = 0; t < 4; t++)
                    *reinterpret_cast<float4*>(a.v + (row * 3 + x) * n + 32 * wave + 8 * t + 4 * G) =
                        make_float4(acc[x][0][4 * t], acc[x][0][4 * t + 1], acc[x][0][4 * t + 2], acc[x][0][4 * t + 3]);
    }
    __syncthreads();
    if (tid < kNodes && r0 + tid < a.rows) {
        float mx = top[tid];
        for (int k = 1; k <= waves; k++) mx = fmaxf(mx, top[k * kNodes + tid]);
        a.cat_max[r0 + tid] = mx;
    }
}

// Few nodes: tiles of 16 nodes in 16 x 16 x 32 matrix instructions, a wave owning 16 channels of all three maps, n = 32 C channels.  What a
// workgroup does in turn is then half as long, and what it waits for is asked for at once: its nodes, and its share of the weights,
// which all fit in registers (up to 128 channels: wider workgroups have half as many registers to a lane).
//
// The whole update in us, in a graph: three launches in this one's place / the kernel above / this one.  128 channels, 16 nodes 41 / 35 /
// 29, 337 35.7 / 38.8 / 32.7, 1000 49 / 49 / 42, 4096 66 / 58 / 51, 8192 88 / 70.8 / 70.2; 64 channels 36 / 33 / 27, 31.5 / 33.8 / 28.2,
// 34 / 34 / 29, 50 / 43 / 37, 59 / 49 / 44.  Called eagerly on 337 nodes 46.4 / 40.5 / 37.6, where the host is what is waited for.  Bound by
// the way from the loads through LDS and the products to the stores, up to two tiles to a CU: on 14 000 nodes of 128 channels the update
// takes 104 where the kernel above, which reads the weights half as often, takes 98 (10 000 nodes 97.7 and 96.5, of 64 channels 53.2
// and 53.7).
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kFewNodes = 16, kFewMaxN = 128;
constexpr long kFewRows = 512 * kFewNodes;
// x . w of one component of a node, in fp32 and k in order, as lds_row_in_fp32 has it
__device__ __noinline__ float component_in_fp32(const float* x, const _Float16* planes, long plane_elems, int o, int n, float iw) {
    const float inv = unmark_weight(iw);
    float sum = 0.f;
#pragma unroll 1
    for (int k = 0; k < n; k++) {
        const long at = packed_index(o, k, n);
        const float h = (float)planes[at], l = (float)planes[plane_elems + at];
        sum = fmaf(x[3 * k], (fabsf(h) < __builtin_inff() ? h + l : h) * inv, sum);
    }
    return sum;
}

template <int C>
__global__ void __launch_bounds__(128 * C) painn_update_maps_few_kernel(const UpdateMaps a) {
    constexpr int n = 32 * C, waves = 2 * C, kPairs = kFewNodes / 2, kTrips = (kPairs + waves - 1) / waves;
    constexpr int x_stride = kFewNodes * n, x_lo = 3 * x_stride;
    // [piece][component][chunk of 32 k][8 k][node][k % 8]: a fragment is one contiguous kilobyte
    __shared__ __attribute__((aligned(16))) _Float16 xh[2 * x_lo];
    __shared__ float row_max[3][kFewNodes], top[1 + waves][kFewNodes];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, kk = lane >> 4, p = lane & 31, quad = p < n / 4 ? p : 0;
    const long r0 = (long)blockIdx.x * kFewNodes;
    // rows past the end repeat the last one and are not written
    auto row_of = [&](int node) { return r0 + node < a.rows ? r0 + node : a.rows - 1; };

    // 32 lanes to a node, four channels to a lane
    float4 f[kTrips][3], xa[kTrips];
#pragma unroll
    for (int t = 0; t < kTrips; t++) {
        const long at = row_of(2 * (wave + t * waves < kPairs ? wave + t * waves : wave) + (lane >> 5)) * n + 4 * quad;
#pragma unroll
        for (int k = 0; k < 3; k++) f[t][k] = reinterpret_cast<const float4*>(a.x_v + 3 * at)[k];
        xa[t] = *reinterpret_cast<const float4*>(a.x_a + at);
    }
    const long w_lo = (long)pad256(3 * n) * n;
    const _Float16* const w = a.planes + packed_index(16 * wave + m, 8 * kk, n);
    halfx8 wh[3][C], wl[3][C];
#pragma unroll
    for (int map = 0; map < 3; map++)
#pragma unroll
        for (int c = 0; c < C; c++) {
            wh[map][c] = *reinterpret_cast<const halfx8*>(w + 1024 * (map * C * C + c));
            wl[map][c] = *reinterpret_cast<const halfx8*>(w + w_lo + 1024 * (map * C * C + c));
        }
    float iw[3][4];
#pragma unroll
    for (int map = 0; map < 3; map++) {
        const float4 w4 = *reinterpret_cast<const float4*>(a.inv + map * n + 16 * wave + 4 * kk);
        iw[map][0] = w4.x; iw[map][1] = w4.y; iw[map][2] = w4.z; iw[map][3] = w4.w;
    }
    const bool marked = has_marks(a.inv, 3 * n, lane);
    __builtin_amdgcn_sched_barrier(0);                             // (all of it is asked for before any is waited for)

#pragma unroll
    for (int t = 0; t < kTrips; t++) {
        if (wave + t * waves >= kPairs) break;                     // (uniform)
        const int node = 2 * (wave + t * waves) + (lane >> 5);
        const float g[12] = {f[t][0].x, f[t][0].y, f[t][0].z, f[t][0].w, f[t][1].x, f[t][1].y,
                             f[t][1].z, f[t][1].w, f[t][2].x, f[t][2].y, f[t][2].z, f[t][2].w};
        float mx[3] = {0.f, 0.f, 0.f}, ma = fmaxf(fmaxf(fabsf(xa[t].x), fabsf(xa[t].y)), fmaxf(fabsf(xa[t].z), fabsf(xa[t].w)));
#pragma unroll
        for (int k = 0; k < 12; k++) mx[k % 3] = fmaxf(mx[k % 3], fabsf(g[k]));
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) {
            ma = fmaxf(ma, __shfl_xor(ma, d));
#pragma unroll
            for (int x = 0; x < 3; x++) mx[x] = fmaxf(mx[x], __shfl_xor(mx[x], d));
        }
#pragma unroll
        for (int x = 0; x < 3; x++) {
            float inv;
            const float v[4] = {g[x], g[3 + x], g[6 + x], g[9 + x]};
            if (p < n / 4)
                store_pieces(xh, x_lo, x * x_stride + (p >> 3) * 512 + (p >> 1 & 3) * 128 + node * 8 + (p & 1) * 4, v, pow2_scale(mx[x], &inv));
            if (p == 0) row_max[x][node] = mx[x];
        }
        if (p == 0) top[0][node] = ma;
    }
    __syncthreads();

    floatx4 large[3][3], small[3][3];                              // [component][map]
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int map = 0; map < 3; map++) large[x][map] = small[x][map] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int x = 0; x < 3; x++) {
            const _Float16* at = xh + x * x_stride + 512 * c + 8 * lane;
            const halfx8 bh = *reinterpret_cast<const halfx8*>(at), bl = *reinterpret_cast<const halfx8*>(at + x_lo);
#pragma unroll
            for (int map = 0; map < 3; map++) small[x][map] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[map][c], bh, small[x][map], 0, 0, 0);
#pragma unroll
            for (int map = 0; map < 3; map++) large[x][map] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[map][c], bh, large[x][map], 0, 0, 0);
#pragma unroll
            for (int map = 0; map < 3; map++) small[x][map] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[map][c], bl, small[x][map], 0, 0, 0);
        }
    // lane: node m, channels o .. o + 3
    const int o = 16 * wave + 4 * kk;
    const long row = row_of(m);
    const bool live = r0 + m < a.rows;
    float y[3][3][4];
#pragma unroll
    for (int x = 0; x < 3; x++) {
        float isx;
        pow2_scale(row_max[x][m], &isx);
#pragma unroll
        for (int map = 0; map < 3; map++)
#pragma unroll
            for (int i = 0; i < 4; i++) y[x][map][i] = (small[x][map][i] + large[x][map][i]) * isx * iw[map][i];
        if (marked || beyond_split(row_max[x][m]))                 // (a row or a weight that the pieces cannot carry)
#pragma unroll
            for (int map = 0; map < 3; map++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    y[x][map][i] = component_in_fp32(a.x_v + row * n * 3 + x, a.planes, w_lo, map * n + o + i, n, iw[map][i]);
    }
    float ip[4], nr[4], mr = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float x = y[0][1][i], yy = y[1][1][i], z = y[2][1][i];
        ip[i] = y[0][0][i] * x + y[1][0][i] * yy + y[2][0][i] * z;
        nr[i] = sqrtf(x * x + yy * yy + z * z);
        mr = fmaxf(mr, nr[i]);
    }
    mr = fmaxf(mr, __shfl_xor(mr, 16));
    mr = fmaxf(mr, __shfl_xor(mr, 32));
    if (kk == 0) top[1 + wave][m] = mr;
    __syncthreads();
    if (live) {
        *reinterpret_cast<float4*>(a.ip + row * n + o) = make_float4(ip[0], ip[1], ip[2], ip[3]);
        *reinterpret_cast<float4*>(a.cat + row * 2 * n + n + o) = make_float4(nr[0], nr[1], nr[2], nr[3]);
#pragma unroll
        for (int x = 0; x < 3; x++)
            *reinterpret_cast<float4*>(a.v + (row * 3 + x) * n + o) = make_float4(y[x][2][0], y[x][2][1], y[x][2][2], y[x][2][3]);
    }
#pragma unroll
    for (int t = 0; t < kTrips; t++) {
        const int node = 2 * (wave + t * waves) + (lane >> 5);
        if (node < kFewNodes && p < n / 4 && r0 + node < a.rows) *reinterpret_cast<float4*>(a.cat + (r0 + node) * 2 * n + 4 * p) = xa[t];
    }
    if (tid < kFewNodes && r0 + tid < a.rows) {
        float mx = top[0][tid];
#pragma unroll
        for (int k = 1; k <= waves; k++) mx = fmaxf(mx, top[k][tid]);
        a.cat_max[r0 + tid] = mx;
    }
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_painn_update_maps_supported(int n) { return n >= 64 && n <= kMaxN && n % 32 == 0; }

int mg_painn_update_maps(const float* x_v, const float* x_a, long rows, int n, const void* packed_W, float* ip, float* cat,
                         float* cat_rowmax, float* v, mg_stream_t stream) {
    MG_REQUIRE(rows >= 0 && mg_painn_update_maps_supported(n), "mg_painn_update_maps: n must be a multiple of 32 from 64 to %d", kMaxN);
    if (rows == 0) return MG_OK;
    MG_REQUIRE(x_v && x_a && packed_W && ip && cat && cat_rowmax && v && aligned16(x_v) && aligned16(x_a) && aligned16(packed_W) &&
                   aligned16(ip) && aligned16(cat) && aligned16(v),
               "mg_painn_update_maps: null or unaligned pointer");
    const long tiles = ceil_div(rows, kNodes);
    MG_REQUIRE(tiles <= 0x7fffffffL, "mg_painn_update_maps: too many rows");
    UpdateMaps a{x_v, x_a, rows, n, static_cast<const _Float16*>(packed_W), nullptr, ip, cat, cat_rowmax, v};
    a.inv = reinterpret_cast<const float*>(a.planes + 2L * ((3 * n + 255) / 256 * 256) * n);
    if (n <= kFewMaxN && rows <= kFewRows) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(rows, kFewNodes)), dim3(4 * n), 0, (hipStream_t)stream, a);
            return check_launch("mg_painn_update_maps");
        };
        return n == 64 ? launch(painn_update_maps_few_kernel<2>) : n == 96 ? launch(painn_update_maps_few_kernel<3>)
                                                                          : launch(painn_update_maps_few_kernel<4>);
    }
    const size_t lds = (size_t)3 * kNodes * n * 4 + ((3 + 1 + kMaxN / 32) * kNodes + 3 * kMaxN) * sizeof(float);
    if (lds > 65536)
        MG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(painn_update_maps_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(painn_update_maps_kernel, dim3((unsigned)tiles), dim3(2 * n), lds, (hipStream_t)stream, a);
    return check_launch("mg_painn_update_maps");
}

}  // extern "C"
