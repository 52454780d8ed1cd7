// Gradients of the PaiNN message whose filter is interpolated from its grid (painn.hip, painn_table_message_lds_kernel), for
// edge vectors that are not differentiated.  With f the filter of an edge (4 blocks of n columns), a and v the rows of its
// destination, u its direction, and (g, ga) the gradient rows of its source:
//   d_actv[r] = (v . M0, v . M1, S2, S3),  d_v[r] = a0 M0 + a1 M1   with the sums over the edges that read row r
//   M0 = sum f0 g,  M1 = sum f1 (u x g),  S2 = sum f2 (u . g),  S3 = sum f3 ga
//   d_grid[i, k] = sum over edges and taps of w (dp_k a_k),  dp = (g . v, v . (u x g), u . g, ga)
// The first line needs only the 8 sums per channel: a and v of the row come in once at the end, an edge reads its source's g and
// ga (2 KB at n = 128; the pass it replaces also read four grid rows from the caches, 8 KB, and wrote the edge's 2 KB of
// d_filter).  The second takes the edges in the order of their grid rows, so that the 4 taps x 4 blocks of a row are sums in
// registers, and forms d_filter itself from the node rows: no per-edge array is written or read (3.3 GB each way at 1.6 M
// edges).  16384 nodes, 1.6 M edges, n = 128: see the figures at the two kernels.
#include "common.hpp"
#include "lane_sums.hpp"
#include <algorithm>

namespace mg {
namespace {

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }

// |r| / h and 1 / sqrt(eps + |r|^2).  (The fused multiply-adds are spelled out: every kernel here that puts an edge into a grid
// row must find the same one.)
typedef float floatx4 __attribute__((ext_vector_type(4)));
struct EdgePlace { float u, inv; };
__device__ __forceinline__ EdgePlace place(float x, float y, float z, float inv_h, float eps) {
    const float r2 = fmaf(x, x, fmaf(y, y, z * z));
    return {sqrtf(r2) * inv_h, 1.0f / sqrtf(eps + r2)};
}
__device__ __forceinline__ void lagrange(float t, float (&w)[4]) {
    const float tp = t + 1.0f, tm = t - 1.0f, tq = t - 2.0f;
    w[0] = -(1.0f / 6.0f) * t * tm * tq;
    w[1] = 0.5f * tp * tm * tq;
    w[2] = -0.5f * tp * t * tq;
    w[3] = (1.0f / 6.0f) * tp * t * tm;
}

// ------------------------------------------------------------------------------------------------ records
// Per position of the order by destination: (float offset of the first grid row in LDS as int bits, w0, w1, w2), (w3, u), and
// the source.
__global__ void __launch_bounds__(256) node_records_kernel(const float* __restrict__ r_ij, const int* __restrict__ order,
                                                           const int* __restrict__ src, long E, int mask, float inv_h, float eps,
                                                           float4* __restrict__ rec, int* __restrict__ from) {
    const long p = (long)blockIdx.x * 256 + threadIdx.x;
    if (p >= E) return;
    const long e = order ? min(max((long)order[p], 0L), E - 1) : p;
    const float x = r_ij[3 * e], y = r_ij[3 * e + 1], z = r_ij[3 * e + 2];
    const EdgePlace q = place(x, y, z, inv_h, eps);
    const float fl = floorf(q.u);
    float w[4];
    lagrange(q.u - fl, w);
    const int first = ((int)fl - 1) & mask;
    rec[2 * p] = make_float4(__int_as_float(first * kSliceRowF), w[0], w[1], w[2]);
    rec[2 * p + 1] = make_float4(w[3], x * q.inv, y * q.inv, z * q.inv);
    from[p] = src[e];
}
// Per position of the order by grid row: (source, destination as int bits, t, ux), (uy, uz, 0, 0)
__global__ void __launch_bounds__(256) row_records_kernel(const float* __restrict__ r_ij, const int* __restrict__ order,
                                                          const int* __restrict__ src, const int* __restrict__ dst, long E,
                                                          float inv_h, float eps, float4* __restrict__ rec) {
    const long p = (long)blockIdx.x * 256 + threadIdx.x;
    if (p >= E) return;
    const long e = min(max((long)order[p], 0L), E - 1);
    const float x = r_ij[3 * e], y = r_ij[3 * e + 1], z = r_ij[3 * e + 2];
    const EdgePlace q = place(x, y, z, inv_h, eps);
    rec[2 * p] = make_float4(__int_as_float(src[e]), __int_as_float(dst[e]), q.u - floorf(q.u), x * q.inv);
    rec[2 * p + 1] = make_float4(y * q.inv, z * q.inv, 0.f, 0.f);
}
__global__ void __launch_bounds__(256) grid_row_kernel(const float* __restrict__ r_ij, long E, int mask, float inv_h, float eps,
                                                       int* __restrict__ row) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e < E) row[e] = (int)floorf(place(r_ij[3 * e], r_ij[3 * e + 1], r_ij[3 * e + 2], inv_h, eps).u) & mask;
}

// The same with the edges taken in the order of their sources in node_order (cells of the neighbour search): row and edge per
// position.  Neighbours in space then stay neighbours inside a grid row's bucket, and so do the node rows its kernel gathers.
// first[slot]: position of a slot's first edge inside its block of 256 slots, block_edges: the block's edges.
constexpr int kSlotBlock = 256, kTailBlocks = 64;
__global__ void __launch_bounds__(kSlotBlock) slot_starts_kernel(const int* __restrict__ row_ptr, const int* __restrict__ node_order,
                                                                 long n_nodes, int* __restrict__ first, int* __restrict__ block_edges) {
    __shared__ int wave_sum[kSlotBlock / kWave];
    const long slot = (long)blockIdx.x * kSlotBlock + threadIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int own = 0;
    if (slot < n_nodes) {
        const long node = min(max((long)node_order[slot], 0L), n_nodes - 1);
        own = max(row_ptr[node + 1] - row_ptr[node], 0);
    }
    int sum = own;
    for (int d = 1; d < kWave; d <<= 1) {
        const int up = __shfl_up(sum, d);
        if (lane >= d) sum += up;
    }
    if (lane == kWave - 1) wave_sum[wave] = sum;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kSlotBlock / kWave; w++) {
        if (w < wave) before += wave_sum[w];
        total += wave_sum[w];
    }
    if (slot < n_nodes) first[slot] = before + sum - own;
    if (threadIdx.x == 0) block_edges[blockIdx.x] = total;
}
// a wave per slot; the last kTailBlocks blocks take edges behind the last row, as they come
__global__ void __launch_bounds__(256) grid_row_by_node_kernel(const float* __restrict__ r_ij, const int* __restrict__ row_ptr,
                                                               const int* __restrict__ node_order, long n_nodes, long E,
                                                               const int* __restrict__ first, const int* __restrict__ block_edges,
                                                               int mask, float inv_h, float eps, int* __restrict__ row,
                                                               int* __restrict__ edge) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    auto put = [&](long p, long e) {
        row[p] = (int)floorf(place(r_ij[3 * e], r_ij[3 * e + 1], r_ij[3 * e + 2], inv_h, eps).u) & mask;
        edge[p] = (int)e;
    };
    const long slot_blocks = gridDim.x - kTailBlocks;
    if (blockIdx.x >= slot_blocks) {
        for (long p = max(row_ptr[n_nodes], 0) + (blockIdx.x - slot_blocks) * 256 + threadIdx.x; p < E; p += 256 * kTailBlocks) put(p, p);
        return;
    }
    const long slot = (long)blockIdx.x * 4 + wave;
    if (slot >= n_nodes) return;
    int base = 0;
    for (int b = lane; b < slot / kSlotBlock; b += kWave) base += block_edges[b];
    for (int d = 1; d < kWave; d <<= 1) base += __shfl_xor(base, d);
    const long node = min(max((long)node_order[slot], 0L), n_nodes - 1);
    const long lo = max(row_ptr[node], 0), hi = min((long)row_ptr[node + 1], E), at = (long)base + first[slot];
    for (long e = lo + lane; e < hi; e += kWave)
        if (at + e - lo < E) put(at + e - lo, e);
}

// ------------------------------------------------------------------------------------------------ gradients of actv and v
// The mapping of painn_table_message_lds_kernel: a workgroup holds one slice of 16 channels of the grid in LDS, a wave takes 16
// edges of its node per step, 4 lanes x 4 channels each.  Bound by vector issue, like that kernel.
__global__ void __launch_bounds__(1024) grid_node_grad_kernel(
    const int* __restrict__ row_ptr, const int* __restrict__ from, const int* __restrict__ node_order, long n_nodes, long E,
    const float4* __restrict__ rec, const float* __restrict__ table, int tab_rows, const float* __restrict__ g_v,
    const float* __restrict__ g_a, const float* __restrict__ actv, const float* __restrict__ v, int n,
    const float* __restrict__ add_v, float* __restrict__ d_actv, float* __restrict__ d_v) {
    extern __shared__ float tab[];                            // (tab_rows + 3) x kSliceRowF
    const int n_slices = n / kSliceChan;
    const int slice = blockIdx.x % n_slices;
    const int group = blockIdx.x / n_slices, groups = gridDim.x / n_slices;
    for (int q = threadIdx.x; q < (tab_rows + kSliceExtraRows) * (kSliceCols / 4); q += blockDim.x) {
        const int row = q / (kSliceCols / 4), piece = q % (kSliceCols / 4), k = piece / 4, c4 = piece % 4;
        st4(tab + row * kSliceRowF + 4 * piece,
            ld4(table + (long)(row & (tab_rows - 1)) * 4 * n + k * n + slice * kSliceChan + 4 * c4));
    }
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, waves = blockDim.x / kWave;
    const int l4 = lane & 3, sub = lane >> 2;
    constexpr int kPerIter = kWave / 4;
    const float* gv_base = g_v + (slice * kSliceChan + 4 * l4) * 3;
    const float* ga_base = g_a + slice * kSliceChan + 4 * l4;
    const unsigned v_stride = 3u * (unsigned)n, a_stride = (unsigned)n;
    const float* tab_l = tab + 4 * l4;
    for (long slot = (long)group * waves + wave; slot < n_nodes; slot += (long)groups * waves) {
        const long node = node_order ? node_order[slot] : slot;
        const int lo = max(row_ptr[node], 0), hi = min(row_ptr[node + 1], (int)E);
        // value 4 c + q of channel c: (M0, S2) and (M1, S3)
        float A[16], B[16];
#pragma unroll
        for (int k = 0; k < 16; k++) { A[k] = 0.f; B[k] = 0.f; }
        int e = lo + sub;
        unsigned j = 0;
        float4 ra = make_float4(0.f, 0.f, 0.f, 0.f), rb = ra;
        if (e < hi) { j = (unsigned)from[e]; ra = rec[2 * (long)e]; rb = rec[2 * (long)e + 1]; }
        while (e < hi) {
            const float* gv = gv_base + (long)j * v_stride;
            const float4 g0 = ld4(gv), g1 = ld4(gv + 4), g2 = ld4(gv + 8), ga = ld4(ga_base + (long)j * a_stride);
            e += kPerIter;
            unsigned j_next = 0;
            float4 na = ra, nb = rb;
            if (e < hi) { j_next = (unsigned)from[e]; na = rec[2 * (long)e]; nb = rec[2 * (long)e + 1]; }
            const float* tp = tab_l + __float_as_int(ra.x);
            const float w0 = ra.y, w1 = ra.z, w2 = ra.w, w3 = rb.x, ux = rb.y, uy = rb.z, uz = rb.w;
            float f[4][4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 t0 = ld4(tp + k * kSliceChan), t1 = ld4(tp + kSliceRowF + k * kSliceChan),
                             t2 = ld4(tp + 2 * kSliceRowF + k * kSliceChan), t3 = ld4(tp + 3 * kSliceRowF + k * kSliceChan);
                f[k][0] = w0 * t0.x + w1 * t1.x + w2 * t2.x + w3 * t3.x;
                f[k][1] = w0 * t0.y + w1 * t1.y + w2 * t2.y + w3 * t3.y;
                f[k][2] = w0 * t0.z + w1 * t1.z + w2 * t2.z + w3 * t3.z;
                f[k][3] = w0 * t0.w + w1 * t1.w + w2 * t2.w + w3 * t3.w;
            }
            const float gg[12] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w, g2.x, g2.y, g2.z, g2.w};
            const float gs[4] = {ga.x, ga.y, ga.z, ga.w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float x = gg[3 * c], y = gg[3 * c + 1], z = gg[3 * c + 2];
                A[4 * c + 0] = fmaf(f[0][c], x, A[4 * c + 0]);
                A[4 * c + 1] = fmaf(f[0][c], y, A[4 * c + 1]);
                A[4 * c + 2] = fmaf(f[0][c], z, A[4 * c + 2]);
                A[4 * c + 3] = fmaf(f[2][c], ux * x + uy * y + uz * z, A[4 * c + 3]);
                B[4 * c + 0] = fmaf(f[1][c], uy * z - uz * y, B[4 * c + 0]);                 // u x g
                B[4 * c + 1] = fmaf(f[1][c], uz * x - ux * z, B[4 * c + 1]);
                B[4 * c + 2] = fmaf(f[1][c], ux * y - uy * x, B[4 * c + 2]);
                B[4 * c + 3] = fmaf(f[3][c], gs[c], B[4 * c + 3]);
            }
            j = j_next; ra = na; rb = nb;
        }
        const float sA = sum_over_slots(A, lane), sB = sum_over_slots(B, lane);
        const int c = sub >> 2, q = sub & 3;
        const long ch = slice * kSliceChan + 4 * l4 + c, row4 = node * 4L * n + ch;
        const bool edges = lo < hi;                           // (a node without edges has gradient zero whatever it holds)
        const float vq = edges && q < 3 ? v[(node * n + ch) * 3 + q] : 0.f;
        const float a0 = edges ? actv[row4] : 0.f, a1 = edges ? actv[row4 + n] : 0.f;
        float s0 = vq * sA, s1 = vq * sB;                     // v . M0, v . M1: over the lanes q = 0..2 of the channel
        s0 += __shfl_xor(s0, 4); s1 += __shfl_xor(s1, 4);
        s0 += __shfl_xor(s0, 8); s1 += __shfl_xor(s1, 8);
        if (d_v && q < 3) {
            const long at = (node * n + ch) * 3 + q;
            const float own = a0 * sA + a1 * sB;
            d_v[at] = add_v ? own + add_v[at] : own;
        }
        if (d_actv) {
            if (q == 3) { d_actv[row4 + 2 * n] = sA; d_actv[row4 + 3 * n] = sB; }
            else if (q < 2) d_actv[row4 + q * n] = q ? s1 : s0;
        }
    }
}

// ------------------------------------------------------------------------------------------------ gradient of the grid
// part[((row splits + s) 4 + j) 4n + k n + c]: piece s of the edges of a grid row, in order; a wave takes 16 edges per step as
// above, its 64 sums per lane are added over the slots at the end and over the 4 waves in wave order.  Slices are the fastest
// block index (one slice per XCD at n = 128), pieces the slowest: the blocks that run together read the rows of the same part
// of the nodes.  Bound by those reads (11 x 16 bytes per lane and edge against 64 multiply-adds): 9.0 GB in 480 us at 1.6 M edges, n = 128,
// of the 20 TB/s that gathers of this size and alignment reach from the L2 (16 384 x 256 bytes: 21).  With the edges of a bucket in
// the order of their atoms' numbers, whose neighbours are anywhere, 621 us.  32-bit offsets and a peeled last step (four waves per
// SIMD for three) made it slower, 600 us.
__global__ void __launch_bounds__(256) grid_row_grad_kernel(const int* __restrict__ bucket_ptr, const float4* __restrict__ rec,
                                                            long E, int rows, int splits, long n_nodes,
                                                            const float* __restrict__ actv_s, const float* __restrict__ v,
                                                            const float* __restrict__ g_v, const float* __restrict__ g_a, int n,
                                                            float* __restrict__ part) {
    __shared__ float fold[4][4][kWave];
    const int n_slices = n / kSliceChan;
    const int slice = blockIdx.x % n_slices, rest = blockIdx.x / n_slices;
    const int row = rest % rows, s = rest / rows;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int l4 = lane & 3, sub = lane >> 2;
    const long b_lo = max((long)bucket_ptr[row], 0L), b_hi = min((long)bucket_ptr[row + 1], E), len = b_hi - b_lo;
    const long lo = b_lo + len * s / splits, hi = b_lo + len * (s + 1) / splits;
    const float* a_base = actv_s + slice * kSliceCols + 4 * l4;
    const float* v_base = v + (slice * kSliceChan + 4 * l4) * 3;
    const float* gv_base = g_v + (slice * kSliceChan + 4 * l4) * 3;
    const float* ga_base = g_a + slice * kSliceChan + 4 * l4;
    // value 4 k + c of the four taps.  Each is a sum of outer products of an edge's 4 weights with its 4 lanes' values: the
    // 16-block 4 x 4 x 1 matrix instruction in fp32 (block = edge slot, row = tap, column = lane of the slot)
    floatx4 acc[16];
#pragma unroll
    for (int k = 0; k < 16; k++) acc[k] = floatx4{0.f, 0.f, 0.f, 0.f};
    long e = lo + 16 * wave + sub;
    float4 ra = make_float4(0.f, 0.f, 0.f, 0.f), rb = ra;
    if (e < hi) { ra = rec[2 * e]; rb = rec[2 * e + 1]; }
    // (a slot past the end takes part in the matrix instructions with zeros for both operands: what it read are the rows of some
    // other edge or of node 0, and zero times an infinity there would be NaN)
    for (long e0 = lo + 16 * wave; e0 < hi; e0 += 64) {
        const bool live = e < hi;
        const long from = min(max((long)__float_as_int(ra.x), 0L), n_nodes - 1), to = min(max((long)__float_as_int(ra.y), 0L), n_nodes - 1);
        const float* ap = a_base + to * 4 * n;
        const float* vp = v_base + to * 3 * n;
        const float* gp = gv_base + from * 3 * n;
        float4 a[4];
#pragma unroll
        for (int k = 0; k < 4; k++) a[k] = ld4(ap + k * kSliceChan);
        const float4 v0 = ld4(vp), v1 = ld4(vp + 4), v2 = ld4(vp + 8);
        const float4 g0 = ld4(gp), g1 = ld4(gp + 4), g2 = ld4(gp + 8), ga = ld4(ga_base + from * n);
        e += 64;
        float4 na = ra, nb = rb;
        if (e < hi) { na = rec[2 * e]; nb = rec[2 * e + 1]; }
        const float ux = ra.w, uy = rb.x, uz = rb.y;
        float w[4];
        lagrange(ra.z, w);
        const float my_w = live ? (l4 == 0 ? w[0] : l4 == 1 ? w[1] : l4 == 2 ? w[2] : w[3]) : 0.f;
        const float vv[12] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w, v2.x, v2.y, v2.z, v2.w};
        const float gg[12] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w, g2.x, g2.y, g2.z, g2.w};
        const float gs[4] = {ga.x, ga.y, ga.z, ga.w};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float x = gg[3 * c], y = gg[3 * c + 1], z = gg[3 * c + 2];
            const float vx = vv[3 * c], vy = vv[3 * c + 1], vz = vv[3 * c + 2];
            const float av[4] = {c == 0 ? a[0].x : c == 1 ? a[0].y : c == 2 ? a[0].z : a[0].w,
                                 c == 0 ? a[1].x : c == 1 ? a[1].y : c == 2 ? a[1].z : a[1].w,
                                 c == 0 ? a[2].x : c == 1 ? a[2].y : c == 2 ? a[2].z : a[2].w,
                                 c == 0 ? a[3].x : c == 1 ? a[3].y : c == 2 ? a[3].z : a[3].w};
            const float d[4] = {(x * vx + y * vy + z * vz) * av[0],
                                ((uy * z - uz * y) * vx + (uz * x - ux * z) * vy + (ux * y - uy * x) * vz) * av[1],
                                (ux * x + uy * y + uz * z) * av[2], gs[c] * av[3]};
#pragma unroll
            for (int k = 0; k < 4; k++) acc[4 * k + c] = __builtin_amdgcn_mfma_f32_4x4x1f32(my_w, live ? d[k] : 0.f, acc[4 * k + c], 0, 0, 0);
        }
        ra = na; rb = nb;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float tap[16];
#pragma unroll
        for (int k = 0; k < 16; k++) tap[k] = acc[k][j];
        fold[wave][j][lane] = sum_over_slots(tap, lane);
    }
    __syncthreads();
    // wave j adds tap j over the four waves; value `sub` = 4 k + c of the channel quad l4
    const float sum = (fold[0][wave][lane] + fold[1][wave][lane]) + (fold[2][wave][lane] + fold[3][wave][lane]);
    part[(((long)row * splits + s) * 4 + wave) * 4 * n + (sub >> 2) * n + slice * kSliceChan + 4 * l4 + (sub & 3)] = sum;
}

// d_table[m, :] = the sum over pieces and taps of the parts that touch row m, in this order
__global__ void __launch_bounds__(256) grid_grad_finish_kernel(const float* __restrict__ part, int rows, int cols, int splits,
                                                               float* __restrict__ d_table) {
    const int quads = cols >> 2;
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long m = t / quads;
    if (m >= rows) return;
    const int c = (int)(t - m * quads) * 4;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j = 0; j < 4; j++) {
        const long row = (m + 1 - j) & (rows - 1);
        for (int s = 0; s < splits; s++) {
            const float4 p = ld4(part + ((row * splits + s) * 4 + j) * (long)cols + c);
            acc.x += p.x; acc.y += p.y; acc.z += p.z; acc.w += p.w;
        }
    }
    st4(d_table + m * cols + c, acc);
}

// ------------------------------------------------------------------------------------------------ stable sort by small keys
// One pass of a stable radix sort on 9 bits: counts per (digit, chunk), their prefix sums per digit, and the scatter, in which a
// wave ranks 64 elements at a time by comparing digits across lanes.  (torch.sort on these keys takes 10 launches: 150 us for
// 1.6 M edges, 90 for 90 000; this takes 3.)
// What bounds it is the chain within a workgroup, not the bytes: a thread therefore loads all PER of its keys at once and keeps them
// for both loops, and a chunk (256 PER elements) is as short as leaves each compute unit a workgroup, down to two elements a thread.  One pass over
// 78 000 keys: count 3.5, sums 4, scatter 5 us (chunks of 4096 read in the loops: 6-9, 4, 17); 8000 keys 5, 5, 5 (6-8, 5, 20);
// 1.4 M keys 6, 5, 22 (8, 5, 29).
constexpr int kDigits = 512, kDigitBits = 9;
int sort_per_thread(long n) {
    int per = 2;
    while (per < 16 && n > 256L * 256 * per) per *= 2;
    return per;
}
// the PER keys of a thread: element k of wave w is 64 (PER w + k) + lane of the chunk, so that a wave's elements are consecutive
template <int PER>
__device__ __forceinline__ long sort_element(int k) {
    return ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 * PER) + 64 * k + (threadIdx.x & 63);
}

template <int PER>
__global__ void __launch_bounds__(256) sort_count_kernel(const int* __restrict__ keys, long n, int shift, int chunks,
                                                         int* __restrict__ counts) {
    __shared__ int hist[kDigits];
    int key[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const long i = sort_element<PER>(k);
        key[k] = keys[min(i, n - 1)];
    }
    for (int d = threadIdx.x; d < kDigits; d += 256) hist[d] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++)
        if (sort_element<PER>(k) < n) atomicAdd(&hist[(key[k] >> shift) & (kDigits - 1)], 1);
    __syncthreads();
    for (int d = threadIdx.x; d < kDigits; d += 256) counts[(long)d * chunks + blockIdx.x] = hist[d];
}
// counts[d] -> exclusive prefix sums over the chunks; totals[d]
__global__ void __launch_bounds__(64) sort_prefix_kernel(int* __restrict__ counts, int chunks, int* __restrict__ totals) {
    int* row = counts + (long)blockIdx.x * chunks;
    int base = 0;
    for (int c0 = 0; c0 < chunks; c0 += 64) {
        const int c = c0 + threadIdx.x;
        const int own = c < chunks ? row[c] : 0;
        int sum = own;
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(sum, d);
            if ((int)threadIdx.x >= d) sum += up;
        }
        if (c < chunks) row[c] = base + sum - own;
        base += __shfl(sum, 63);
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = base;
}
template <int PER>
__global__ void __launch_bounds__(256) sort_scatter_kernel(const int* __restrict__ keys, const int* __restrict__ values, long n,
                                                           int shift, int chunks, const int* __restrict__ counts,
                                                           const int* __restrict__ totals, int* __restrict__ keys_out,
                                                           int* __restrict__ values_out) {
    __shared__ int at[4][kDigits];                            // next output position per wave and digit
    __shared__ int wave_sum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int key[PER], value[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const long i = min(sort_element<PER>(k), n - 1);
        key[k] = keys[i];
        value[k] = values ? values[i] : (int)i;
    }
    // exclusive prefix sums of the totals: two digits per thread
    {
        const int a = totals[2 * tid], b = totals[2 * tid + 1];
        int sum = a + b;
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(sum, d);
            if (lane >= d) sum += up;
        }
        if (lane == 63) wave_sum[wave] = sum;
        __syncthreads();
        int before = sum - a - b;
        for (int w = 0; w < wave; w++) before += wave_sum[w];
        at[0][2 * tid] = before + counts[(long)(2 * tid) * chunks + blockIdx.x];
        at[0][2 * tid + 1] = before + a + counts[(long)(2 * tid + 1) * chunks + blockIdx.x];
        for (int w = 1; w < 4; w++) { at[w][2 * tid] = 0; at[w][2 * tid + 1] = 0; }
    }
    __syncthreads();
    // how many of each digit the waves before this one hold
    if (wave < 3)
#pragma unroll
        for (int k = 0; k < PER; k++)
            if (sort_element<PER>(k) < n)
                for (int w = wave + 1; w < 4; w++) atomicAdd(&at[w][(key[k] >> shift) & (kDigits - 1)], 1);
    __syncthreads();
    for (int d = tid; d < kDigits; d += 256)
        for (int w = 1; w < 4; w++) at[w][d] += at[0][d];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const bool live = sort_element<PER>(k) < n;
        const int d = (key[k] >> shift) & (kDigits - 1);
        unsigned long long same = __ballot(live);
#pragma unroll
        for (int b = 0; b < kDigitBits; b++) {
            const unsigned long long m = __ballot((d >> b) & 1);
            same &= ((d >> b) & 1) ? m : ~m;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1ull));
        int pos = 0;
        if (live) pos = at[wave][d] + rank;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (live && rank == 0) at[wave][d] = pos + __popcll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (live) {
            values_out[pos] = value[k];
            if (keys_out) keys_out[pos] = key[k];
        }
    }
}

int splits_of(int rows, long E) {
    // pieces of about 400 edges: 6 steps of the 4 waves, against which adding 64 sums over the slots is a third; the fewer edges, the
    // smaller the part of space whose node rows the pieces that run together read (1.6 M edges, pieces of 200 / 400 / 768 / 1600: 526,
    // 479, 504, 716 us, their sums 22, 11, 7, 5)
    long s = ceil_div(E, 400L * rows);
    return (int)(s < 1 ? 1 : (s > 16 ? 16 : s));
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_painn_grid_grad_supported(int table_rows, int n) {
    return n >= kSliceChan && n % kSliceChan == 0 && n <= 256 && table_rows >= 4 && table_rows <= kSliceMaxRows &&
                   (table_rows & (table_rows - 1)) == 0
               ? 1
               : 0;
}

int mg_painn_grid_grad_workspace_bytes(int table_rows, int n, long n_edges, size_t* bytes) {
    MG_REQUIRE(bytes && n_edges >= 0 && mg_painn_grid_grad_supported(table_rows, n), "mg_painn_grid_grad_workspace_bytes: bad argument");
    const size_t by_node = (size_t)n_edges * 36, by_row = (size_t)n_edges * 32 + (size_t)table_rows * splits_of(table_rows, n_edges) * 16 * n * sizeof(float);
    *bytes = (by_node > by_row ? by_node : by_row) + 32;
    return MG_OK;
}

int mg_painn_grid_node_grad(const int* row_ptr, const int* order, const int* src, const int* node_order, int n_nodes, long n_edges,
                            const float* r_ij, const float* table, int table_rows, float period, float epsilon, const float* g_v,
                            const float* g_a, const float* actv, const float* v, int n, void* workspace, float* d_actv, float* d_v,
                            mg_stream_t stream) {
    return mg_painn_grid_node_add_grad(row_ptr, order, src, node_order, n_nodes, n_edges, r_ij, table, table_rows, period, epsilon, g_v,
                                       g_a, actv, v, n, workspace, nullptr, d_actv, d_v, stream);
}

int mg_painn_grid_node_add_grad(const int* row_ptr, const int* order, const int* src, const int* node_order, int n_nodes, long n_edges,
                                const float* r_ij, const float* table, int table_rows, float period, float epsilon, const float* g_v,
                                const float* g_a, const float* actv, const float* v, int n, void* workspace, const float* add_v,
                                float* d_actv, float* d_v, mg_stream_t stream) {
    MG_REQUIRE(n_nodes >= 0 && n_edges >= 0 && n_edges < (1L << 31) && period > 0.f && mg_painn_grid_grad_supported(table_rows, n),
               "mg_painn_grid_node_grad: bad argument");
    if (n_nodes == 0) return MG_OK;
    MG_REQUIRE(row_ptr && table && g_v && g_a && actv && v && workspace && (n_edges == 0 || (src && r_ij)) && aligned16(table) &&
                   aligned16(g_v) && aligned16(g_a),
               "mg_painn_grid_node_grad: null or unaligned pointer");
    hipStream_t st = (hipStream_t)stream;
    float4* rec = reinterpret_cast<float4*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t(15));
    int* from = reinterpret_cast<int*>(rec + 2 * n_edges);
    if (n_edges > 0)
        hipLaunchKernelGGL(node_records_kernel, dim3((unsigned)ceil_div(n_edges, 256)), dim3(256), 0, st, r_ij, order, src, n_edges,
                           table_rows - 1, (float)table_rows / period, epsilon, rec, from);
    const int n_slices = n / kSliceChan;
    MG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(grid_node_grad_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (kSliceMaxRows + kSliceExtraRows) * kSliceRowF * (int)sizeof(float)));
    long groups = ceil_div(256, n_slices);                    // one workgroup per CU
    const long max_groups = ceil_div(n_nodes, 16);
    if (groups > max_groups) groups = max_groups;
    hipLaunchKernelGGL(grid_node_grad_kernel, dim3((unsigned)(groups * n_slices)), dim3(1024),
                       (size_t)(table_rows + kSliceExtraRows) * kSliceRowF * sizeof(float), st, row_ptr, from, node_order,
                       (long)n_nodes, n_edges, rec, table, table_rows, g_v, g_a, actv, v, n, add_v, d_actv, d_v);
    return check_launch("mg_painn_grid_node_grad");
}

int mg_painn_grid_rows(const float* r_ij, long n_edges, int table_rows, float period, int* row, mg_stream_t stream) {
    MG_REQUIRE(n_edges >= 0 && period > 0.f && table_rows >= 4 && (table_rows & (table_rows - 1)) == 0, "mg_painn_grid_rows: bad argument");
    if (n_edges == 0) return MG_OK;
    MG_REQUIRE(r_ij && row, "mg_painn_grid_rows: null pointer");
    hipLaunchKernelGGL(grid_row_kernel, dim3((unsigned)ceil_div(n_edges, 256)), dim3(256), 0, (hipStream_t)stream, r_ij, n_edges,
                       table_rows - 1, (float)table_rows / period, 1.0f, row);
    return check_launch("mg_painn_grid_rows");
}

int mg_painn_grid_rows_by_node_workspace_bytes(int n_nodes, size_t* bytes) {
    MG_REQUIRE(bytes && n_nodes >= 0, "mg_painn_grid_rows_by_node_workspace_bytes: bad argument");
    *bytes = ((size_t)n_nodes + ceil_div(n_nodes, kSlotBlock)) * sizeof(int);
    return MG_OK;
}

int mg_painn_grid_rows_by_node(const float* r_ij, long n_edges, const int* row_ptr, const int* node_order, int n_nodes, int table_rows,
                               float period, void* workspace, int* row, int* edge, mg_stream_t stream) {
    MG_REQUIRE(n_edges >= 0 && n_edges < (1L << 31) && n_nodes >= 0 && (n_nodes > 0 || n_edges == 0) && period > 0.f && table_rows >= 4 &&
                   (table_rows & (table_rows - 1)) == 0,
               "mg_painn_grid_rows_by_node: bad argument");
    if (n_edges == 0) return MG_OK;
    MG_REQUIRE(r_ij && row_ptr && node_order && workspace && row && edge, "mg_painn_grid_rows_by_node: null pointer");
    int* first = static_cast<int*>(workspace);
    int* block_edges = first + n_nodes;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(slot_starts_kernel, dim3((unsigned)ceil_div(n_nodes, kSlotBlock)), dim3(kSlotBlock), 0, st, row_ptr, node_order,
                       (long)n_nodes, first, block_edges);
    hipLaunchKernelGGL(grid_row_by_node_kernel, dim3((unsigned)(ceil_div(n_nodes, 4) + kTailBlocks)), dim3(256), 0, st, r_ij, row_ptr,
                       node_order, (long)n_nodes, n_edges, (const int*)first, (const int*)block_edges, table_rows - 1,
                       (float)table_rows / period, 1.0f, row, edge);
    return check_launch("mg_painn_grid_rows_by_node");
}

int mg_painn_grid_table_grad(const int* order, const int* bucket_ptr, const int* src, const int* dst, int n_nodes, long n_edges,
                             const float* r_ij, int table_rows, float period, float epsilon, const float* g_v, const float* g_a,
                             const float* actv_sliced, const float* v, int n, void* workspace, float* d_table, mg_stream_t stream) {
    MG_REQUIRE(n_nodes >= 0 && n_edges >= 0 && period > 0.f && mg_painn_grid_grad_supported(table_rows, n) && (n_nodes > 0 || n_edges == 0),
               "mg_painn_grid_table_grad: bad argument");
    MG_REQUIRE(bucket_ptr && workspace && d_table && aligned16(d_table), "mg_painn_grid_table_grad: null or unaligned pointer");
    MG_REQUIRE(n_edges == 0 || (order && src && dst && r_ij && g_v && g_a && actv_sliced && v && aligned16(g_v) && aligned16(g_a) &&
                                aligned16(actv_sliced) && aligned16(v)),
               "mg_painn_grid_table_grad: null or unaligned pointer");
    hipStream_t st = (hipStream_t)stream;
    float4* rec = reinterpret_cast<float4*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t(15));
    float* part = reinterpret_cast<float*>(rec + 2 * n_edges);
    const int splits = splits_of(table_rows, n_edges), n_slices = n / kSliceChan;
    if (n_edges > 0)
        hipLaunchKernelGGL(row_records_kernel, dim3((unsigned)ceil_div(n_edges, 256)), dim3(256), 0, st, r_ij, order, src, dst, n_edges,
                           (float)table_rows / period, epsilon, rec);
    hipLaunchKernelGGL(grid_row_grad_kernel, dim3((unsigned)(n_slices * table_rows * splits)), dim3(256), 0, st, bucket_ptr, rec,
                       n_edges, table_rows, splits, (long)n_nodes, actv_sliced, v, g_v, g_a, n, part);
    hipLaunchKernelGGL(grid_grad_finish_kernel, dim3((unsigned)ceil_div((long)table_rows * n, 256)), dim3(256), 0, st,
                       (const float*)part, table_rows, 4 * n, splits, d_table);
    return check_launch("mg_painn_grid_table_grad");
}

int mg_sort_by_key_workspace_bytes(long count, size_t* bytes) {
    MG_REQUIRE(bytes && count >= 0, "mg_sort_by_key_workspace_bytes: bad argument");
    // (up to 256 chunks of every length but the longest: a smaller count may have more chunks than this one)
    const long own = ceil_div(count, 256L * sort_per_thread(count)), shortest = ceil_div(count, 256L * 2);
    const long chunks = std::max(own, std::min(256L, shortest));
    *bytes = ((size_t)(chunks + 1) * kDigits + 3 * (size_t)count) * sizeof(int);
    return MG_OK;
}

int mg_sort_by_key(const int* keys, long count, int key_limit, void* workspace, int* order, int* sorted_keys, mg_stream_t stream) {
    return mg_sort_values_by_key(keys, nullptr, count, key_limit, workspace, order, sorted_keys, stream);
}

int mg_sort_values_by_key(const int* keys, const int* values, long count, int key_limit, void* workspace, int* order, int* sorted_keys,
                          mg_stream_t stream) {
    MG_REQUIRE(count >= 0 && count < (1L << 31) && key_limit >= 1, "mg_sort_by_key: bad argument");
    if (count == 0) return MG_OK;
    MG_REQUIRE(keys && workspace && order && sorted_keys, "mg_sort_by_key: null pointer");
    hipStream_t st = (hipStream_t)stream;
    const int per = sort_per_thread(count), chunks = (int)ceil_div(count, 256L * per);
    int* counts = static_cast<int*>(workspace);
    int* totals = counts + (long)chunks * kDigits;
    int *spare_keys = totals + kDigits, *spare_values = spare_keys + count;
    int passes = 1;
    while (passes < 4 && ((long)key_limit - 1) >> (kDigitBits * passes)) passes++;
    const int *k_in = keys, *v_in = values;
    for (int p = 0; p < passes; p++) {
        // the last pass ends in the caller's arrays
        const bool to_out = (passes - 1 - p) % 2 == 0;
        int *k_out = to_out ? sorted_keys : spare_keys, *v_out = to_out ? order : spare_values;
        const auto pass = [&](auto count_kernel, auto scatter_kernel) {
            hipLaunchKernelGGL(count_kernel, dim3(chunks), dim3(256), 0, st, k_in, count, kDigitBits * p, chunks, counts);
            hipLaunchKernelGGL(sort_prefix_kernel, dim3(kDigits), dim3(64), 0, st, counts, chunks, totals);
            hipLaunchKernelGGL(scatter_kernel, dim3(chunks), dim3(256), 0, st, k_in, v_in, count, kDigitBits * p, chunks,
                               (const int*)counts, (const int*)totals, k_out, v_out);
        };
        switch (per) {
            case 2: pass(sort_count_kernel<2>, sort_scatter_kernel<2>); break;
            case 4: pass(sort_count_kernel<4>, sort_scatter_kernel<4>); break;
            case 8: pass(sort_count_kernel<8>, sort_scatter_kernel<8>); break;
            default: pass(sort_count_kernel<16>, sort_scatter_kernel<16>); break;
        }
        k_in = k_out;
        v_in = v_out;
    }
    return check_launch("mg_sort_by_key");
}

}  // extern "C"
