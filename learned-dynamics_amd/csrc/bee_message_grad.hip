// Gradients of the rank-0/1/2 message products (archs/diffuser_atoms15.py:238-253, the training path of Messages): the 13
// products of the destination's features (a, v, d) with the edge filters enc, enc u and enc u (x) u, u = rh, where the
// products of rank 1 and 2 are summed over the edges of their source node.
//
// The right operands being enc times powers of u, every gradient of an edge is a function of 60 gradient floats of its
// SOURCE (per channel), 3 of the edge and 13 operand floats of its destination:
//   dl0      = enc (s000 + g011.u + u.g022 u)
//   dl1[x]   = enc (s110 u_x + g101_x + (u x g111)_x + u_x (g121.u) + (g112 u)_x)
//   dl2[x,y] = enc (h_x u_y + g202[x,y] + (u x g212[x])_y),   h = g211 + g222 u + s220 u
//   d_enc    = (dl0 l0 + dl1.l1 + dl2:l2) / enc               (the products are linear in l)
//   d_u      = enc times the derivative of that sum in u, summed over channels.
// One wave walks the edges of a source node with 64 channels of the 60 gradients in registers, so they are read once per
// node and not twice per edge; no filters are formed in memory.  dl leaves component-major (E, 13, chan), whole 256-byte
// rows, and a second kernel sums it over the edges of each destination in a fixed order.
// What bounds it: traffic, 17 floats read and 14 written per edge and channel, then 13 read.  131 000 edges, 8192 nodes, 256
// channels, edge vectors not differentiated: 0.70 ms (6.0 TB/s) and 0.44 ms (4.1 TB/s).  Before, the filters were stored
// (0.44 ms), two kernels gathered the 60 gradients at every edge's source (1.8 ms each), a third took the right operands'
// gradients to enc and rh (0.35 ms) and three segment sums followed (0.37 ms).
// Two layouts of operands and gradients: ROWS is component-major, (row, comp, product, chan), the results of the forward kernel
// and of the output linears as they are, a wave's accesses 256 bytes each; the other has every product by itself, (row, chan, comp),
// for callers that hold them so (a module whose linears are called one by one): 0.72 and 0.42 ms, nothing to transpose around it.
// Any multiple of 64 channels; differentiable.message_products comes here for multiples of 256, the widths of its forward
// kernels, and keeps the plain formulation for others.
// The per-edge gradients are stored rather than formed again by destination, which would gather the 60 floats of the source
// for every edge instead of writing and reading 13.
#include "common.hpp"

namespace mg {
namespace {

constexpr int kXcds = 8;
constexpr int kLeft = 13;           // floats of a left operand per channel: 1 + 3 + 9

struct EdgeIn { float l[kLeft], enc, s[3], u[3]; };

__device__ __forceinline__ float dot3(const float* a, const float* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
__device__ __forceinline__ void cross3(const float* a, const float* b, float* o) {
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}
// the T components of channel c of a row: (row, T, product, chan) of PRODUCTS products side by side, p at the first row's channel 0
// of the product, or (row, chan, T)
template <bool ROWS, int T, int PRODUCTS = 1>
__device__ __forceinline__ void load(const float* p, long row, long C, int c, float* o) {
    const float* q = ROWS ? p + row * (T * PRODUCTS) * C + c : p + (row * C + c) * T;
    const long step = ROWS ? PRODUCTS * C : 1;
#pragma unroll
    for (int k = 0; k < T; k++) o[k] = q[k * step];
}

template <bool ROWS>
__device__ __forceinline__ EdgeIn load_edge(const mg_bee_message_grad& a, long e, int node, int c) {
    EdgeIn in;
    const long C = a.chan;
    load<ROWS, 1>(a.l_0, node, C, c, in.l);
    load<ROWS, 3>(a.l_1, node, C, c, in.l + 1);
    load<ROWS, 9>(a.l_2, node, C, c, in.l + 4);
    in.enc = a.enc[e * C + c];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        load<ROWS, 1, 3>(a.dy[k], e, C, c, in.s + k);
        in.u[k] = a.rh[3 * e + k];
    }
    return in;
}

// LEFT: the operands' gradients per edge; RIGHT: d_enc; VEC: d_rh, a sum over this wave's 64 channels
template <bool ROWS, bool LEFT, bool RIGHT, bool VEC>
__global__ void __launch_bounds__(256, 3) bee_message_grad_kernel(mg_bee_message_grad a, long items, long blocks_per_xcd,
                                                                  float* __restrict__ dl, float* __restrict__ part) {
    const int lane = threadIdx.x & 63;
    // consecutive nodes on one XCD: their edges lead to the same rows, which its L2 then holds
    const long block = (blockIdx.x % kXcds) * blocks_per_xcd + blockIdx.x / kXcds;
    const long item = __builtin_amdgcn_readfirstlane((int)(block * 4 + (threadIdx.x >> 6)));
    if (item >= items) return;
    const int C = a.chan, slices = C / 64;
    const int node = (int)(item / slices), slice = (int)(item - (long)node * slices), c = slice * 64 + lane;
    const long begin = a.row_ptr[node], end = a.row_ptr[node + 1];
    if (begin >= end) return;
    float g011[3], g101[3], g121[3], g211[3], g111[3], g022[9], g202[9], g112[9], g222[9], g212[9];
    load<ROWS, 3, 5>(a.dy[3], node, C, c, g011);
    load<ROWS, 3, 5>(a.dy[4], node, C, c, g101);
    load<ROWS, 3, 5>(a.dy[5], node, C, c, g121);
    load<ROWS, 3, 5>(a.dy[6], node, C, c, g211);
    load<ROWS, 9, 5>(a.dy[7], node, C, c, g022);
    load<ROWS, 9, 5>(a.dy[8], node, C, c, g202);
    load<ROWS, 9, 5>(a.dy[9], node, C, c, g112);
    load<ROWS, 9, 5>(a.dy[10], node, C, c, g222);
    load<ROWS, 3, 5>(a.dy[11], node, C, c, g111);
    load<ROWS, 9, 5>(a.dy[12], node, C, c, g212);
    auto destination = [&](long e) {
        const int d = a.dst[e];
        return d < 0 ? 0 : (d >= a.n_rows ? a.n_rows - 1 : d);
    };
    EdgeIn next = load_edge<ROWS>(a, begin, destination(begin), c);
    for (long e = begin; e < end; e++) {
        const EdgeIn in = next;
        const long f = e + 1 < end ? e + 1 : e;              // (the next edge's operands are under way during this one's sums)
        next = load_edge<ROWS>(a, f, destination(f), c);
        const float *u = in.u, *l1 = in.l + 1, *l2 = in.l + 4;
        const float s110 = in.s[1], s220 = in.s[2], gu = dot3(g121, u);
        float w[3], h[3], o[kLeft], t[3];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            w[x] = dot3(g022 + 3 * x, u);
            h[x] = g211[x] + dot3(g222 + 3 * x, u) + s220 * u[x];
        }
        o[0] = in.s[0] + dot3(g011, u) + dot3(w, u);
        cross3(u, g111, t);
#pragma unroll
        for (int x = 0; x < 3; x++) o[1 + x] = s110 * u[x] + g101[x] + t[x] + u[x] * gu + dot3(g112 + 3 * x, u);
#pragma unroll
        for (int x = 0; x < 3; x++) {
            cross3(u, g212 + 3 * x, t);
#pragma unroll
            for (int y = 0; y < 3; y++) o[4 + 3 * x + y] = h[x] * u[y] + g202[3 * x + y] + t[y];
        }
        if constexpr (LEFT) {
#pragma unroll
            for (int k = 0; k < kLeft; k++) dl[(e * kLeft + k) * C + c] = in.enc * o[k];
        }
        if constexpr (RIGHT) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < kLeft; k++) s += o[k] * in.l[k];
            a.d_enc[e * C + c] = s;
        }
        if constexpr (VEC) {
            const float lu = dot3(l1, u);
            float p[3], du[3], b[3];
#pragma unroll
            for (int x = 0; x < 3; x++) p[x] = dot3(l2 + 3 * x, u);
            cross3(g111, l1, b);
#pragma unroll
            for (int y = 0; y < 3; y++) {
                du[y] = in.l[0] * (g011[y] + w[y] + g022[y] * u[0] + g022[3 + y] * u[1] + g022[6 + y] * u[2]) + s110 * l1[y] + b[y] +
                        l1[y] * gu + g121[y] * lu + s220 * p[y];
#pragma unroll
                for (int x = 0; x < 3; x++) du[y] += g112[3 * x + y] * l1[x] + l2[3 * x + y] * h[x] + g222[3 * x + y] * p[x];
            }
#pragma unroll
            for (int x = 0; x < 3; x++) {
                cross3(g212 + 3 * x, l2 + 3 * x, b);
#pragma unroll
                for (int y = 0; y < 3; y++) du[y] += b[y];
            }
#pragma unroll
            for (int y = 0; y < 3; y++) {
                du[y] *= in.enc;
                for (int k = 1; k < 64; k <<= 1) du[y] += __shfl_xor(du[y], k);
            }
            if (lane < 3) part[(e * slices + slice) * 3 + lane] = lane == 0 ? du[0] : (lane == 1 ? du[1] : du[2]);
        }
    }
}

// d_rh[e] = the slices' sums, in their order
__global__ void __launch_bounds__(256) bee_message_grad_rh_kernel(const float* __restrict__ part, long n, int slices,
                                                                  float* __restrict__ d_rh) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const long e = t / 3;
    const int k = (int)(t - 3 * e);
    float s = 0.f;
    for (int j = 0; j < slices; j++) s += part[(e * slices + j) * 3 + k];
    d_rh[t] = s;
}

// (E, 13, chan) rows summed over the edges of each destination, in the order of its sorted edges; one wave per node and 64
// channels, two edges in flight
template <bool ROWS>
__global__ void __launch_bounds__(256) bee_message_grad_sum_kernel(const float* __restrict__ dl, const int* __restrict__ row_ptr,
                                                                   const int* __restrict__ perm, long items, long blocks_per_xcd,
                                                                   int C, float* __restrict__ d_0, float* __restrict__ d_1,
                                                                   float* __restrict__ d_2) {
    const int lane = threadIdx.x & 63;
    const long block = (blockIdx.x % kXcds) * blocks_per_xcd + blockIdx.x / kXcds;
    const long item = __builtin_amdgcn_readfirstlane((int)(block * 4 + (threadIdx.x >> 6)));
    if (item >= items) return;
    const int slices = C / 64, node = (int)(item / slices), c = (int)(item - (long)node * slices) * 64 + lane;
    const int begin = row_ptr[node], end = row_ptr[node + 1];
    float s[kLeft] = {};
    int k = begin;
    for (; k + 1 < end; k += 2) {
        const float *p = dl + (long)(perm ? perm[k] : k) * kLeft * C + c, *q = dl + (long)(perm ? perm[k + 1] : k + 1) * kLeft * C + c;
        float x[kLeft], y[kLeft];
#pragma unroll
        for (int j = 0; j < kLeft; j++) { x[j] = p[(long)j * C]; y[j] = q[(long)j * C]; }
#pragma unroll
        for (int j = 0; j < kLeft; j++) s[j] = (s[j] + x[j]) + y[j];
    }
    if (k < end) {
        const float* p = dl + (long)(perm ? perm[k] : k) * kLeft * C + c;
#pragma unroll
        for (int j = 0; j < kLeft; j++) s[j] += p[(long)j * C];
    }
    const long at = (long)node * C + c;
    d_0[at] = s[0];
#pragma unroll
    for (int j = 0; j < 3; j++) d_1[ROWS ? ((long)node * 3 + j) * C + c : 3 * at + j] = s[1 + j];
#pragma unroll
    for (int j = 0; j < 9; j++) d_2[ROWS ? ((long)node * 9 + j) * C + c : 9 * at + j] = s[4 + j];
}

// floats of the two pieces of the workspace: the operands' gradients per edge, and d_rh's sums per 64 channels
size_t left_floats(long E, int chan) { return (size_t)E * kLeft * chan; }
size_t part_floats(long E, int chan) { return ((size_t)E * (chan / 64) * 3 + 3) / 4 * 4; }

template <bool ROWS, bool LEFT, bool RIGHT>
void launch(const mg_bee_message_grad& a, bool vec, long items, long per_xcd, float* dl, float* part, hipStream_t st) {
    const dim3 grid((unsigned)(per_xcd * kXcds));
    if (vec)
        hipLaunchKernelGGL((bee_message_grad_kernel<ROWS, LEFT, RIGHT, true>), grid, dim3(256), 0, st, a, items, per_xcd, dl, part);
    else
        hipLaunchKernelGGL((bee_message_grad_kernel<ROWS, LEFT, RIGHT, false>), grid, dim3(256), 0, st, a, items, per_xcd, dl, part);
}

template <bool ROWS>
int run(const char* what, const mg_bee_message_grad& a, mg_stream_t stream) {
    MG_REQUIRE(mg_bee_message_grad_supported(a.chan), "%s: chan = %d is no multiple of 64", what, a.chan);
    MG_REQUIRE(a.E >= 0 && a.E < (1L << 31) && a.n_src >= 0 && a.n_rows >= 0, "%s: bad size", what);
    const bool left = a.d_0 || a.d_1 || a.d_2, right = a.d_enc != nullptr, vec = a.d_rh != nullptr;
    MG_REQUIRE(!left || (a.d_0 && a.d_1 && a.d_2 && a.dst_row_ptr), "%s: the three operands' gradients come together", what);
    hipStream_t st = (hipStream_t)stream;
    const long slices = a.chan / 64, items = (long)a.n_src * slices, sums = (long)a.n_rows * slices;
    MG_REQUIRE(items < (1L << 31) - 64 && sums < (1L << 31) - 64, "%s: too many nodes", what);
    float *dl = static_cast<float*>(a.workspace), *part = dl + (left ? left_floats(a.E, a.chan) : 0);
    if (a.E > 0 && (left || right || vec)) {
        MG_REQUIRE(a.row_ptr && a.dst && a.rh && a.enc && a.l_0 && a.l_1 && a.l_2 && a.n_rows > 0 && (a.workspace || !(left || vec)),
                   "%s: null pointer", what);
        for (int k = 0; k < 13; k++) MG_REQUIRE(a.dy[k], "%s: gradient %d is null", what, k);
        const long per_xcd = ceil_div(ceil_div(items, 4), kXcds);
        if (left && right) launch<ROWS, true, true>(a, vec, items, per_xcd, dl, part, st);
        else if (left) launch<ROWS, true, false>(a, vec, items, per_xcd, dl, part, st);
        else if (right) launch<ROWS, false, true>(a, vec, items, per_xcd, dl, part, st);
        else launch<ROWS, false, false>(a, vec, items, per_xcd, dl, part, st);
        if (vec)
            hipLaunchKernelGGL(bee_message_grad_rh_kernel, dim3((unsigned)ceil_div(3 * a.E, 256)), dim3(256), 0, st, part, 3 * a.E,
                               (int)slices, a.d_rh);
    }
    if (left && sums > 0) {
        const long per_xcd = ceil_div(ceil_div(sums, 4), kXcds);
        hipLaunchKernelGGL(bee_message_grad_sum_kernel<ROWS>, dim3((unsigned)(per_xcd * kXcds)), dim3(256), 0, st, dl, a.dst_row_ptr, a.perm,
                           sums, per_xcd, a.chan, a.d_0, a.d_1, a.d_2);
    }
    return check_launch(what);
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_bee_message_grad_supported(int chan) { return chan >= 64 && chan % 64 == 0; }

int mg_bee_message_grad_workspace_bytes(long E, int chan, int want_left, int want_rh, size_t* bytes) {
    MG_REQUIRE(bytes && E >= 0 && mg_bee_message_grad_supported(chan), "mg_bee_message_grad_workspace_bytes: bad argument");
    *bytes = ((want_left ? left_floats(E, chan) : 0) + (want_rh ? part_floats(E, chan) : 0)) * sizeof(float);
    return MG_OK;
}

int mg_bee_message_grad_run(const mg_bee_message_grad* args, mg_stream_t stream) {
    MG_REQUIRE(args, "mg_bee_message_grad_run: null pointer");
    return run<false>("mg_bee_message_grad_run", *args, stream);
}

int mg_bee_message_grad_rows_run(const mg_bee_message_grad_rows* args, mg_stream_t stream) {
    MG_REQUIRE(args, "mg_bee_message_grad_rows_run: null pointer");
    const mg_bee_message_grad_rows& r = *args;
    mg_bee_message_grad a{};
    a.l_0 = r.l_0; a.l_1 = r.l_1; a.l_2 = r.l_2; a.enc = r.enc; a.rh = r.rh;
    // the products of a rank lie side by side, in the order 011 101 121 211 111 and 022 202 112 222 212
    static const int s1[5] = {3, 4, 5, 6, 11}, s2[5] = {7, 8, 9, 10, 12};
    for (int k = 0; k < 3; k++) a.dy[k] = r.d_P0 ? r.d_P0 + (long)k * r.chan : nullptr;
    for (int k = 0; k < 5; k++) {
        a.dy[s1[k]] = r.d_S1 ? r.d_S1 + (long)k * r.chan : nullptr;
        a.dy[s2[k]] = r.d_S2 ? r.d_S2 + (long)k * r.chan : nullptr;
    }
    a.row_ptr = r.row_ptr; a.dst = r.dst; a.dst_row_ptr = r.dst_row_ptr; a.perm = r.perm;
    a.E = r.E; a.n_src = r.n_src; a.n_rows = r.n_rows; a.chan = r.chan;
    a.workspace = r.workspace;
    a.d_0 = r.d_0; a.d_1 = r.d_1; a.d_2 = r.d_2; a.d_enc = r.d_enc; a.d_rh = r.d_rh;
    return run<true>("mg_bee_message_grad_rows_run", a, stream);
}

}  // extern "C"
