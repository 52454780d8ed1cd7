// Rank-0/1/2 ("a/v/d") message passing with the 13 Cartesian products, fused
// over CSR rows.
//
// For edge e = (i <- j): phi_a = lin_enc(radial_encode_8(r_ij)) (chan),
// rh = s / sqrt(1 + |s|^2) with s = r_ij * 7 / r0, phi_v = phi_a (x) rh,
// phi_d = phi_a (x) rh (x) rh; left operands are the node features
// l_k = (L_k x_k)[j]; the 13 products p_lab = prod_lab(l, phi) follow.
// Because every right operand is phi_a[c] times a per-edge geometric factor, each
// product is phi_a[c] * g_lab(l[c], rh): nothing of size E x chan x 3 x 3 exists.
//
// What leaves the kernel:
//   P0 (E, 3, chan)      the three scalar products per edge (they feed a per-edge
//                        MLP, which does not commute with the sum over edges)
//   S1 (N, 3, 5, chan)   sum over the edges of node i of the five vector products
//   S2 (N, 9, 5, chan)   ... of the five rank-2 products
// The bias-free output linears Y_lab commute with the sum over edges, so they are
// applied to S1/S2 on N rows afterwards; the (comp, label, chan) order makes
// each of those one plain GEMM with K = 5*chan.
//
// With Y2F the rank-2 sums do not leave the kernel either: the four waves of a workgroup hold the sums of
// 4 / chunks whole nodes, the bias-free output linear of the rank-2 channel (K = 5 chan, dim_d <= 16 outputs) is
// applied to them (rank2_linear.hpp),
// the waves' partial results are summed through LDS, and (node, dim_d, 9) is stored instead of (node, 9, 5, chan):
// 45 chan floats per node less to write, the same again less to read, and one GEMM launch less.
//
// Node features are read in component-major layout (node, comp, chan): the 13
// gathers of a wave are unit-stride reads of 64 channels.  A lane owns one channel
// and keeps its running sums in registers; rows are summed in edge order.
#include "common.hpp"
#include "rank2_linear.hpp"
#include <type_traits>

namespace mg {
namespace {

struct Jacobi8 {
    double a[8][9];   // coefficient of z^j in the i-th shifted Jacobi(1,0) polynomial
};

// binomial coefficients as doubles (exact for the sizes used here)
double binom(int n, int k) {
    if (k < 0 || k > n) return 0.0;
    double r = 1.0;
    for (int i = 1; i <= k; i++) r = r * (n - k + i) / i;
    return r;
}

// P_n^{(1,0)}(2x-1) = sum_s C(n+1, n-s) C(n, s) (x-1)^s x^(n-s)
Jacobi8 jacobi_table() {
    Jacobi8 t{};
    for (int n = 0; n < 8; n++)
        for (int s = 0; s <= n; s++) {
            const double w = binom(n + 1, n - s) * binom(n, s);
            for (int k = 0; k <= s; k++)
                t.a[n][k + n - s] += w * binom(s, k) * (((s - k) & 1) ? -1.0 : 1.0);
        }
    return t;
}

// enc (E,8): radial_encode_8; rhat (E,3): tens_sigmoid(1, r * 7 / r0).
// The polynomial is evaluated in fp64: its monomial form has alternating
// coefficients up to ~1e5, so an fp32 evaluation carries ~1e-3 of rounding noise.
__global__ void __launch_bounds__(256) bee_geometry_kernel(const float* __restrict__ r_ij, long E, float r0,
                                                           float scale, Jacobi8 jac, float* __restrict__ enc,
                                                           float* __restrict__ rhat) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const float x = r_ij[3 * e], y = r_ij[3 * e + 1], z = r_ij[3 * e + 2];
    const float d = sqrtf(x * x + y * y + z * z);
    const float zz = d / r0;
    const double zd = (double)zz;
    const double cut = zd < 1.0 ? 1.0 - zd : 0.0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        double acc = jac.a[i][8];
#pragma unroll
        for (int j = 7; j >= 0; j--) acc = acc * zd + jac.a[i][j];
        enc[8 * e + i] = (float)(acc * cut);
    }
    const float sx = x * scale, sy = y * scale, sz = z * scale;
    const float len = sqrtf(1.0f + (sx * sx + sy * sy + sz * sz));
    rhat[3 * e] = sx / len;
    rhat[3 * e + 1] = sy / len;
    rhat[3 * e + 2] = sz / len;
}

__device__ __forceinline__ long uniform(long v) {
    // the value is the same in every lane: keep it in scalar registers
    const int lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffffL));
    const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    return ((long)hi << 32) | (unsigned)lo;
}

// Gathers of node rows go through buffer loads: the row's byte offset is uniform (scalar offset operand), the lane's
// channel offset a constant vector register, so a gather needs no vector address arithmetic at all (with global
// loads every one of the 13 gathers of an edge built its own 64-bit per-lane address: a tenth of the loop).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t node_rows(const void* base, long bytes) {
    const unsigned n = bytes > 0xffffffffL ? 0xffffffffu : (unsigned)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)n, 0x00020000);
}
__device__ __forceinline__ float gather_row(__amdgpu_buffer_rsrc_t r, unsigned lane_bytes, unsigned row_bytes, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)lane_bytes, (int)row_bytes, 0));
}
__device__ __forceinline__ __bf16 gather_row(__amdgpu_buffer_rsrc_t r, unsigned lane_bytes, unsigned row_bytes, __bf16) {
    return __builtin_bit_cast(__bf16, __builtin_amdgcn_raw_buffer_load_b16(r, (int)lane_bytes, (int)row_bytes, 0));
}

// the arguments of a message; T: storage type of the node features and of the outputs (float, or __bf16 with fp32 arithmetic)
template <typename T>
struct MessageArgs {
    const int *row_ptr, *dst, *order;
    long n_nodes;
    const float *rhat, *enc;
    const T *La, *Lv, *Ld;
    int chan;
    const float *enc_W, *enc_b;
    T *P0, *S1, *S2;
    float *node_max, *edge_max;
    const float* y2_packed;
    int dim_d;
    float* out_d;
    int out_d_accumulate;
    int split;                                                // the rank-2 linear may take fp16 pieces
};

// largest |sum| of a (node, channel): with the other channels of a chunk a row bound for the GEMMs that read S1 / S2
__device__ __forceinline__ float largest(const float (&s1)[15], const float (&s2)[45]) {
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < 15; k++) mx = fmaxf(mx, fabsf(s1[k]));
#pragma unroll
    for (int k = 0; k < 45; k++) mx = fmaxf(mx, fabsf(s2[k]));
    return mx;
}

// (streaming)
__device__ __forceinline__ void put_row(__amdgpu_buffer_rsrc_t r, unsigned lane_bytes, unsigned row_bytes, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)lane_bytes, (int)row_bytes, 2);
}
__device__ __forceinline__ void put_row(__amdgpu_buffer_rsrc_t r, unsigned lane_bytes, unsigned row_bytes, __bf16 v) {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, (int)lane_bytes, (int)row_bytes, 2);
}

// The running sums of one (node, channel).  phi rh is formed once per edge and multiplies l directly, and the sums 022 are symmetric:
// 57 values and 112 multiply-adds an edge make the 60 sums and the three products (122 with every product formed by itself).
// Where features lie along the edges or across them, cross and scalar products cancel: these are formed of l and rh, whose
// products cancel to a rounding of their own, before phi multiplies them.  (Taken apart further they lose what is left: 111 as the
// antisymmetric part of the sum 112 was 2.8 times as far from float64 at 16 neighbours along the edges and 4.2 times at 90, 212 out
// of l and phi rh, its two products added one after the other, 1.3 to 1.8 times on any features, 110 and 121 out of l . phi rh 1.5
// times across the edges; 93 multiply-adds with all three.)
struct NodeSums {
    float v011[3], v101[3], v121[3], v211[3], v111[3], d022[6], d202[9], d112[9], d222[9], d212[9];
    static __device__ __forceinline__ constexpr int sym(int x, int y) { return x <= y ? x * (5 - x) / 2 + y : y * (5 - y) / 2 + x; }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int x = 0; x < 3; x++) v011[x] = v101[x] = v121[x] = v211[x] = v111[x] = 0.f;
#pragma unroll
        for (int k = 0; k < 6; k++) d022[k] = 0.f;
#pragma unroll
        for (int k = 0; k < 9; k++) d202[k] = d112[k] = d222[k] = d212[k] = 0.f;
    }
    // l: the 13 operands; p0: the three scalar products 000, 110, 220 of the edge
    __device__ __forceinline__ void add(float phi, const float (&rh)[3], const float (&l)[13], float (&p0)[3]) {
        const float *l1 = l + 1, *l2 = l + 4;
        float pr[3], t[3];                                                              // phi rh, L rh
#pragma unroll
        for (int x = 0; x < 3; x++) {
            pr[x] = phi * rh[x];
            t[x] = l2[3 * x] * rh[0] + l2[3 * x + 1] * rh[1] + l2[3 * x + 2] * rh[2];
        }
        auto cross = [&](const float* v, int x) { return v[(x + 1) % 3] * rh[(x + 2) % 3] - v[(x + 2) % 3] * rh[(x + 1) % 3]; };
        p0[0] = phi * l[0];
        p0[1] = phi * (l1[0] * rh[0] + l1[1] * rh[1] + l1[2] * rh[2]);
        p0[2] = t[0] * pr[0] + t[1] * pr[1] + t[2] * pr[2];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            const float plx = p0[0] * rh[x];
            v011[x] += plx;
            v101[x] += phi * l1[x];
            v121[x] += p0[1] * rh[x];
            v211[x] += phi * t[x];
            v111[x] += phi * cross(l1, x);
#pragma unroll
            for (int y = 0; y < 3; y++) {
                const int k = 3 * x + y;
                if (y >= x) d022[sym(x, y)] += plx * rh[y];
                d202[k] += phi * l2[k];
                d112[k] += l1[x] * pr[y];
                d222[k] += t[x] * pr[y];
                d212[k] += phi * cross(l2 + 3 * x, y);
            }
        }
    }
    // s1: label order 011, 101, 121, 211, 111; s2: 022, 202, 112, 222, 212, component xy -> 3x + y
    __device__ __forceinline__ void rows(float (&s1)[15], float (&s2)[45]) const {
#pragma unroll
        for (int x = 0; x < 3; x++) {
            s1[x * 5] = v011[x];
            s1[x * 5 + 1] = v101[x];
            s1[x * 5 + 2] = v121[x];
            s1[x * 5 + 3] = v211[x];
            s1[x * 5 + 4] = v111[x];
#pragma unroll
            for (int y = 0; y < 3; y++) {
                const int k = 3 * x + y;
                s2[k * 5] = d022[sym(x, y)];
                s2[k * 5 + 1] = d202[k];
                s2[k * 5 + 2] = d112[k];
                s2[k * 5 + 3] = d222[k];
                s2[k * 5 + 4] = d212[k];
            }
        }
    }
};

// Which items a wave takes.  Workgroup ids go round-robin over the 8 XCDs and an XCD starts its workgroups in id order as slots free
// up: XCD x takes the x-th eighth of the items and workgroup (id >> 3) of it the four items 4 (id >> 3) .. + 3, one
// per wave.  The waves in flight on an XCD are then a window of consecutive nodes of the processing order (cell
// order) that slides forward, and the gathers of neighbouring atoms, which ask for the same rows, come close
// enough in time to meet in the L2.  A persistent grid whose waves stride over the items put a different
// system's nodes into flight at every trip: 2.66 ms against 2.37 ms at 32 x 2048 atoms, 256 channels, and 5.26
// against 4.44 ms at 65536 atoms with 90 neighbours, 128 channels.  (Giving each XCD one 64-channel chunk, so
// that its L2 sees a quarter of each row, was measured with both grids and is slower by 5 %.)
// WHOLE: a workgroup's four items are whole nodes, and its four waves make the same trips (barriers)
template <bool WHOLE>
struct ItemsOfWave {
    long per_xcd, first, step, local;
    __device__ __forceinline__ explicit ItemsOfWave(long items) {
        per_xcd = WHOLE ? (((items + 7) / 8 + 3) & ~3L) : (items + 7) / 8;
        first = (blockIdx.x & 7) * per_xcd;
        step = (long)(gridDim.x >> 3) * (blockDim.x / kWave);
        local = (long)(blockIdx.x >> 3) * (blockDim.x / kWave) + threadIdx.x / kWave;
    }
};

// Operands in registers, one edge ahead where PIPE (pays on long rows): any channel count and alignment.
// Y2F: the rank-2 output linear is applied here (float storage, chan % 64 == 0, 1, 2 or 4 chunks, dim_d <= 16):
// y2_packed as written by pack_rank2_weight_kernel, out_d (nodes, dim_d, 9); S2 is not touched
template <typename T, bool PIPE, bool Y2F>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 4)))
bee_message_kernel(const MessageArgs<T> g) {
    const int lane = threadIdx.x & (kWave - 1);
    const int chan = g.chan, chunks = (chan + kWave - 1) / kWave;
    const long a_bytes = g.n_nodes * chan * (long)sizeof(T);
    const __amdgpu_buffer_rsrc_t rs_a = node_rows(g.La, a_bytes), rs_v = node_rows(g.Lv, 3 * a_bytes), rs_d = node_rows(g.Ld, 9 * a_bytes);
    const long items = g.n_nodes * chunks;
    const ItemsOfWave<Y2F> mine(items);
    for (long local = mine.local; local < mine.per_xcd; local += mine.step) {
        long item = uniform(mine.first + local);
        const bool valid = item < items;                       // uniform over the wave
        if constexpr (Y2F) {
            item = valid ? item : items - 1;                   // a wave without an item still meets the barriers
        } else {
            if (!valid) break;
        }
        const long k_node = item / chunks;
        const int chunk = (int)(item - k_node * chunks);
        const int c = chunk * kWave + lane;
        const bool active = c < chan;
        const int cc = active ? c : chan - 1;   // inactive lanes shadow a valid channel, stores are masked
        const long node = g.order ? (long)g.order[k_node] : k_node;
        const long lo = valid ? g.row_ptr[node] : 0, hi = valid ? g.row_ptr[node + 1] : 0, last = hi - 1;

        float w[8];
#pragma unroll
        for (int m = 0; m < 8; m++) w[m] = g.enc_W[cc * 8 + m];
        const float bias = g.enc_b[cc];
        NodeSums sums;
        sums.clear();

        // Software pipeline: the 13 gathered rows, the encoding and the direction of edge e + 1 are
        // requested before edge e is consumed (the gathers are L2 / fabric latency, and a wave has
        // nothing else to do while it waits), and dst of edge e + 2 one step earlier still.  The
        // look-ahead indices are clamped to the row, so no load is predicated.
        struct EdgeOps {
            T l[13];
            float en[8], rh[3];
        };
        const unsigned lane_off = (unsigned)cc;   // rows are addressed as (uniform base) + 32-bit lane offset
        const unsigned lane_bytes = lane_off * (unsigned)sizeof(T);
        const unsigned row_bytes = (unsigned)chan * (unsigned)sizeof(T);
        auto fetch = [&](EdgeOps& o, long e, long j) {
            const unsigned jr = (unsigned)__builtin_amdgcn_readfirstlane((int)j) * row_bytes;   // byte offset of La[j]
            o.l[0] = gather_row(rs_a, lane_bytes, jr, T{});
#pragma unroll
            for (int t = 0; t < 3; t++) o.l[1 + t] = gather_row(rs_v, lane_bytes, 3u * jr + (unsigned)t * row_bytes, T{});
#pragma unroll
            for (int k = 0; k < 9; k++) o.l[4 + k] = gather_row(rs_d, lane_bytes, 9u * jr + (unsigned)k * row_bytes, T{});
#pragma unroll
            for (int m = 0; m < 8; m++) o.en[m] = g.enc[8 * e + m];
#pragma unroll
            for (int t = 0; t < 3; t++) o.rh[t] = g.rhat[3 * e + t];
        };
        auto consume = [&](const EdgeOps& o, long e) {
            float l[13], p0[3], phi = bias;
#pragma unroll
            for (int k = 0; k < 13; k++) l[k] = (float)o.l[k];
#pragma unroll
            for (int m = 0; m < 8; m++) phi += w[m] * o.en[m];
            sums.add(phi, o.rh, l, p0);
            if (active) {
                // outputs are written once and not read back here: streaming stores leave the L2 to the gathered rows
                const __amdgpu_buffer_rsrc_t p = node_rows(g.P0 + (e * 3) * chan, 3L * row_bytes);
#pragma unroll
                for (int k = 0; k < 3; k++) put_row(p, lane_bytes, k * row_bytes, (T)p0[k]);
            }
            if (g.edge_max) {
                // largest |P0| entry of this (edge, 64-channel chunk): a row bound for the per-edge GEMM
                const float mx = wave_max_nonneg_last_lane(active ? fmaxf(fmaxf(fabsf(p0[0]), fabsf(p0[1])), fabsf(p0[2])) : 0.f);
                if (lane == kWave - 1) g.edge_max[e * chunks + chunk] = mx;
            }
        };
        EdgeOps cur;
        if constexpr (PIPE) {
            // two sets of operands in turn: no copies
            EdgeOps nxt;
            long j_next = 0;
            if (lo < hi) {
                fetch(cur, lo, g.dst[lo]);
                j_next = g.dst[lo + 1 < hi ? lo + 1 : last];
            }
            for (long e = lo; e < hi; e += 2) {
                fetch(nxt, e + 1 < hi ? e + 1 : last, j_next);
                j_next = g.dst[e + 2 < hi ? e + 2 : last];
                consume(cur, e);
                if (e + 1 >= hi) break;
                fetch(cur, e + 2 < hi ? e + 2 : last, j_next);
                j_next = g.dst[e + 3 < hi ? e + 3 : last];
                consume(nxt, e + 1);
            }
        } else {
            for (long e = lo; e < hi; e++) {
                fetch(cur, e, g.dst[e]);
                consume(cur, e);
            }
        }
        float s1[15], s2[45];
        sums.rows(s1, s2);
        if (active && valid) {
            const __amdgpu_buffer_rsrc_t o1 = node_rows(g.S1 + node * 15 * chan, 15L * row_bytes);
#pragma unroll
            for (int k = 0; k < 15; k++) put_row(o1, lane_bytes, k * row_bytes, (T)s1[k]);
            if constexpr (!Y2F) {
                const __amdgpu_buffer_rsrc_t o2 = node_rows(g.S2 + node * 45 * chan, 45L * row_bytes);
#pragma unroll
                for (int k = 0; k < 45; k++) put_row(o2, lane_bytes, k * row_bytes, (T)s2[k]);
            }
        }
        if (g.node_max) {
            const float mx = wave_max_nonneg_last_lane(active ? largest(s1, s2) : 0.f);
            if (lane == kWave - 1 && valid) g.node_max[node * chunks + chunk] = mx;
        }
        if constexpr (Y2F) {
            __shared__ __attribute__((aligned(16))) float lds[4 * kRank2Share];
            rank2_linear_of_node_sums<>(s2, g.split != 0, lds, chunk, chunks, valid, g.y2_packed, g.dim_d,
                                        g.out_d + node * (long)g.dim_d * 9, g.out_d_accumulate != 0);
        }
    }
}

// Rows of whole chunks of 64 channels through LDS, kDepth edges ahead of the one being consumed: 16 bytes a lane go straight there,
// no registers wait for them.  The compiler waits for every such load before any read of LDS, so they are written out and
// counted here: a load reads its address registers when it issues and has no destination registers, nothing depends on it
// but the wave's own slice of LDS.
// Against operands one edge ahead in registers and 122 multiply-adds an edge (bee_message_kernel before NodeSums), both in turn on
// one machine: 65 536 nodes with 90 neighbours, 128 channels of bf16, 3.22 -> 2.77 ms; 32 x 2048 with 16, 256 channels of float with
// the rank-2 linear, 2.11 -> 2.02 ms; 2048 nodes of it 87 -> 80 us.  With 93 multiply-adds an edge it was 2.66 ms, 1.99 ms and 76 us,
// three edges ahead 2.94 ms, 2.07 ms and 78 us, two chunks a wave (two waves a SIMD) 3.34 ms, 2.18 ms and 85 us.  What bounds it:
// bf16 vector issue (128 vector instructions an edge; with 109 of them 0.9 of the cycles at the 2.0 GHz that the power leaves);
// float what it stores and gathers (without the stores of P0 1.61 of 2.04 ms, with every gather a hit 1.76).
constexpr int kDepth = 2;
typedef int intx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ intx4 row_words(const void* base, long bytes) {
    const unsigned long at = reinterpret_cast<unsigned long>(base);
    return intx4{(int)(unsigned)at, (int)((at >> 32) & 0xffff), (int)(bytes > 0xffffffffL ? 0xffffffffu : (unsigned)bytes), 0x00020000};
}
template <int AT>
__device__ __forceinline__ void rows_to_lds(intx4 rsrc, unsigned lane_bytes, unsigned row_bytes, unsigned lds_at) {
    // (five wait states: an operand in scalar registers may just have been written by a vector instruction)
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_at), "v"(lane_bytes), "s"(rsrc), "s"(row_bytes), "n"(AT) : "memory", "scc");
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N < 64, "six bits");
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
// Waits for the loads of the k-th edge of a row, `after` edges before its end.  The queue completes in order; behind those loads
// are the loads of the edge after it and the stores of the two edges before it, fewer at the ends of the row.  Operations that are
// not counted here only make it wait longer.
template <int LOADS, int STORES>
__device__ __forceinline__ void wait_for_edge(int k, int after) {
    static_assert(kDepth == 2, "the cases below");
    if (after >= 1) {
        if (k >= 2) wait_vmcnt<LOADS + 2 * STORES>();
        else if (k == 1) wait_vmcnt<LOADS + STORES>();
        else wait_vmcnt<LOADS>();
    } else if (k >= 2) {
        wait_vmcnt<2 * STORES>();
    } else {
        wait_vmcnt<0>();
    }
}
// EMAX: the edges' maxima are asked for.  Y2F: as above.
template <typename T, bool EMAX, bool Y2F>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 5, sizeof(T) == 4 ? 4 : 5)))
bee_message_ring_kernel(const MessageArgs<T> g) {
    static_assert(!Y2F || std::is_same<T, float>::value, "the fused output linear is for float storage");
    constexpr int kPart = kWave * (int)sizeof(T);                                  // bytes of a row that a wave takes
    constexpr int kRowLanes = kPart / 16, kRowsPerLoad = kWave / kRowLanes;
    static_assert(kRowsPerLoad == 4 || kRowsPerLoad == 8, "two loads and one row, or one and one, make nine rows");
    constexpr int kLoads = sizeof(T) == 4 ? 5 : 4, kStores = EMAX ? 4 : 3, kSlot = 13 * kPart;
    // each wave has a share of LDS of its own: the ring, and once it has run dry what the rank-2 linear needs
    constexpr int kShare = Y2F && 4 * kRank2Share > kDepth * kSlot ? 4 * kRank2Share : kDepth * kSlot;
    __shared__ __attribute__((aligned(16))) unsigned char lds[4 * kShare];
    unsigned char* const ring = lds + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * kShare;
    const unsigned ring_at = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned long)(__attribute__((address_space(3))) unsigned char*)ring);

    const int lane = threadIdx.x & (kWave - 1);
    const int chan = g.chan, chunks = chan / kWave;
    const long items = g.n_nodes * chunks, a_bytes = g.n_nodes * chan * (long)sizeof(T);
    const intx4 words_a = row_words(g.La, a_bytes), words_v = row_words(g.Lv, 3 * a_bytes), words_d = row_words(g.Ld, 9 * a_bytes);
    const unsigned row_bytes = (unsigned)chan * (unsigned)sizeof(T);
    const ItemsOfWave<Y2F> mine(items);
    for (long local = mine.local; local < mine.per_xcd; local += mine.step) {
        long item = uniform(mine.first + local);
        const bool valid = item < items;                       // uniform over the wave
        if constexpr (Y2F) {
            item = valid ? item : items - 1;                   // a wave without an item still meets the barriers
        } else {
            if (!valid) break;
        }
        const long k_node = item / chunks;
        const int chunk = (int)(item - k_node * chunks), c = chunk * kWave + lane;
        const long node = g.order ? (long)scalar_at(g.order + k_node) : k_node;
        const int lo = valid ? scalar_at(g.row_ptr + node) : 0, n = valid ? scalar_at(g.row_ptr + node + 1) - lo : 0;

        // the lane's place in a load: row lane / kRowLanes of its array, 16 bytes of the chunk's part of it
        const unsigned at = (unsigned)(lane / kRowLanes) * row_bytes + (unsigned)(chunk * kPart) + 16u * (unsigned)(lane % kRowLanes);
        auto request = [&](int j, unsigned slot) {                                 // kLoads of them
            const unsigned jr = (unsigned)j * row_bytes;
            rows_to_lds<4 * kPart>(words_d, at, 9u * jr, slot);
            if constexpr (kRowsPerLoad == 4) rows_to_lds<8 * kPart>(words_d, at, 9u * jr + 4u * row_bytes, slot);
            if (lane < 3 * kRowLanes) {
                rows_to_lds<kPart>(words_v, at, 3u * jr, slot);
                if (lane < kRowLanes) {
                    rows_to_lds<12 * kPart>(words_d, at, 9u * jr + 8u * row_bytes, slot);
                    rows_to_lds<0>(words_a, at, jr, slot);
                }
            }
        };
        struct Uniform {
            float en[8], rh[3];
        };
        const int* dst = g.dst + lo;
        const float *enc = g.enc + 8L * lo, *rhat = g.rhat + 3L * lo;
        auto scalars = [&](Uniform& u, int k) {
#pragma unroll
            for (int m = 0; m < 8; m++) u.en[m] = scalar_at(enc + 8L * k + m);
#pragma unroll
            for (int t = 0; t < 3; t++) u.rh[t] = scalar_at(rhat + 3L * k + t);
        };

        float w[8];
#pragma unroll
        for (int m = 0; m < 8; m++) w[m] = g.enc_W[c * 8 + m];
        const float bias = g.enc_b[c];
        NodeSums sums;
        sums.clear();
        const unsigned lane_bytes = (unsigned)c * (unsigned)sizeof(T);
        T* p0_row = g.P0 + 3L * lo * chan;
        float* emax = EMAX ? g.edge_max + (long)lo * chunks + chunk : nullptr;
        const unsigned emax_bytes = lane == kWave - 1 ? 0u : 0x10000u;                  // (the other lanes' are out of range and dropped)
        int slot = 0, j_next = 0;
        auto step = [&](const Uniform& u, Uniform& u_next, int k) {
            wait_for_edge<kLoads, kStores>(k, n - 1 - k);
            const T* rows = reinterpret_cast<const T*>(ring + slot) + lane;
            float l[13], p0[3], phi = bias;
#pragma unroll
            for (int r = 0; r < 13; r++) l[r] = (float)rows[r * kWave];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                          // the slot has been read: it may be filled again
            if (k + kDepth < n) request(j_next, ring_at + (unsigned)slot);
            j_next = scalar_at(dst + (k + kDepth + 1 < n ? k + kDepth + 1 : n - 1));
            scalars(u_next, k + 1 < n ? k + 1 : k);
#pragma unroll
            for (int m = 0; m < 8; m++) phi += w[m] * u.en[m];
            sums.add(phi, u.rh, l, p0);
            // outputs are written once and not read back here: streaming stores leave the L2 to the gathered rows
            const __amdgpu_buffer_rsrc_t out = node_rows(p0_row, 3L * row_bytes);
#pragma unroll
            for (int t = 0; t < 3; t++) put_row(out, lane_bytes, t * row_bytes, (T)p0[t]);
            if constexpr (EMAX) {
                // largest |P0| entry of this (edge, 64-channel chunk): a row bound for the per-edge GEMM
                const float mx = wave_max_nonneg_last_lane(fmaxf(fmaxf(fabsf(p0[0]), fabsf(p0[1])), fabsf(p0[2])));
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(mx), node_rows(emax, 4), (int)emax_bytes, 0, 0);
                emax += chunks;
            }
            p0_row += 3L * chan;
            slot = kSlot - slot;
        };
        if (n > 0) {
            Uniform even, odd;
            request(scalar_at(dst), ring_at);
            if (n > 1) request(scalar_at(dst + 1), ring_at + kSlot);
            j_next = scalar_at(dst + (kDepth < n ? kDepth : n - 1));
            scalars(even, 0);
            for (int k = 0;;) {                                                         // two sets of scalars in turn: no copies
                step(even, odd, k);
                if (++k == n) break;
                step(odd, even, k);
                if (++k == n) break;
            }
        }

        float s1[15], s2[45];
        sums.rows(s1, s2);
        if (valid) {
            const __amdgpu_buffer_rsrc_t o1 = node_rows(g.S1 + node * 15 * chan, 15L * row_bytes);
#pragma unroll
            for (int k = 0; k < 15; k++) put_row(o1, lane_bytes, k * row_bytes, (T)s1[k]);
            if constexpr (!Y2F) {
                const __amdgpu_buffer_rsrc_t o2 = node_rows(g.S2 + node * 45 * chan, 45L * row_bytes);
#pragma unroll
                for (int k = 0; k < 45; k++) put_row(o2, lane_bytes, k * row_bytes, (T)s2[k]);
            }
        }
        if (g.node_max) {
            const float mx = wave_max_nonneg_last_lane(largest(s1, s2));
            if (lane == kWave - 1 && valid) g.node_max[node * chunks + chunk] = mx;
        }
        if constexpr (Y2F)
            rank2_linear_of_node_sums<kShare / 4>(s2, g.split != 0, reinterpret_cast<float*>(lds), chunk, chunks, valid, g.y2_packed, g.dim_d,
                                                  g.out_d + node * (long)g.dim_d * 9, g.out_d_accumulate != 0);
    }
}

// The inverse scales of the 16 outputs of a rank-2 weight, one workgroup each
__global__ void __launch_bounds__(256) rank2_weight_scales_kernel(const float* __restrict__ Y2, long ld, int chan, int dim_d,
                                                                  float* __restrict__ inv) {
    __shared__ float part[4];
    __shared__ int odd;
    const int j = blockIdx.x;
    if (threadIdx.x == 0) odd = 0;
    __syncthreads();
    float mx = 0.f;
    for (int k = threadIdx.x; j < dim_d && k < 5 * chan; k += 256) {
        const float v = fabsf(Y2[j * ld + k]);
        if (v < __builtin_inff()) mx = fmaxf(mx, v);
        else odd = 1;
    }
    mx = wave_max_nonneg_last_lane(mx);
    if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        float one;
        pow2_scale(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])), &one);
        inv[j] = odd ? mark_weight(one) : one;
    }
}
// Y2 (dim_d, 5 chan), row stride ld, into the order of rank2_linear.hpp: threads below 5120 chunks one fp32 value each, those behind
// them eight pieces
__global__ void __launch_bounds__(256) pack_rank2_weight_kernel(const float* __restrict__ Y2, long ld, int chan,
                                                                int dim_d, float* __restrict__ packed) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int chunks = chan / 64;
    const long plain = (long)chunks * kRank2Fp32;
    const int lane = (int)(idx < plain ? idx >> 2 : idx) & 63, j = lane & 15, kk = lane >> 4;
    auto weight = [&](int chunk, int label, int c) { return j < dim_d ? Y2[j * ld + (long)label * chan + 64 * chunk + 16 * kk + c] : 0.f; };
    if (idx < plain) {
        const int tr = (int)(idx & 3), tq = (int)((idx >> 8) & 3);
        const long rest = idx >> 10;                          // chunk * 5 + label
        packed[idx] = weight((int)(rest / 5), (int)(rest % 5), 4 * tq + tr);
        return;
    }
    const long of = (idx - plain) >> 6;                       // chunk * 24 + fragment (plain is a multiple of 64)
    if (of >= chunks * 24L) return;
    const int chunk = (int)(of / 24), f = (int)(of % 24), t = (f >> 1) & 3;
    _Float16* const pieces = reinterpret_cast<_Float16*>(packed + plain);
    const float scale = 1.0f / unmark_weight(reinterpret_cast<const float*>(pieces + (long)chunks * kRank2Pieces)[j]);   // (a power of two)
    halfx8 out;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float v = weight(chunk, f < 16 ? 2 * (f >> 3) + (e & 1) : 4, 4 * t + (e >> 1)) * scale;
        const _Float16 hi = (_Float16)v, lo = (_Float16)(v - (float)hi);
        out[e] = (f & 1) ? lo : hi;
    }
    *reinterpret_cast<halfx8*>(pieces + (of * 64 + lane) * 8) = out;
}

}  // namespace
}  // namespace mg

using namespace mg;

template <typename T>
static int launch_bee_message(const char* what, const int* row_ptr, const int* dst, const int* node_order, int n_nodes,
                              long n_edges, const float* rhat, const float* enc, const T* La, const T* Lv, const T* Ld,
                              int chan, const float* enc_W, const float* enc_b, T* P0, T* S1, T* S2,
                              float* node_max, float* edge_max, mg_stream_t stream, const float* y2_packed = nullptr,
                              int dim_d = 0, float* out_d = nullptr, int out_d_accumulate = 0) {
    MG_REQUIRE(n_nodes >= 0 && n_edges >= 0 && chan >= 0, "%s: negative size", what);
    if (n_nodes == 0 || chan == 0) return MG_OK;
    const bool fused = y2_packed != nullptr;
    MG_REQUIRE(row_ptr && La && Lv && Ld && enc_W && enc_b && S1 && (fused ? out_d != nullptr : S2 != nullptr),
               "%s: null pointer", what);
    MG_REQUIRE(n_edges == 0 || (dst && rhat && enc && P0), "%s: null edge operand", what);
    MG_REQUIRE((long)n_nodes * 9 * chan * (long)sizeof(T) < (1L << 32),
               "%s: the rank-2 node rows must stay below 4 GiB (32-bit row offsets)", what);
    const MessageArgs<T> args{row_ptr, dst, node_order, (long)n_nodes, rhat, enc, La, Lv, Ld, chan, enc_W, enc_b, P0, S1, S2,
                              node_max, edge_max, y2_packed, dim_d, out_d, out_d_accumulate, mg_get_linear_mode() == kLinearF16x2};
    // one item per wave, four per workgroup, an eighth of the items per XCD (the kernel's loop then makes one trip)
    auto launch = [&](auto kernel, long items) -> int {
        const long blocks = 8 * ceil_div(ceil_div(items, 8), 4);
        MG_REQUIRE(blocks < (1L << 31), "%s: too many (node, channel chunk) items for one launch", what);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, args);
        return check_launch(what);
    };
    const long items = (long)n_nodes * ceil_div(chan, kWave);
    // whole chunks, in 16-byte pieces
    const bool ring = chan % kWave == 0 && aligned16(La) && aligned16(Lv) && aligned16(Ld);
    if constexpr (std::is_same<T, float>::value) {
        if (fused) {
            MG_REQUIRE(rank2_fusable(chan, dim_d), "%s: the fused rank-2 linear needs chan = 64, 128 or 256 and dim_d <= 16", what);
            MG_REQUIRE(aligned16(y2_packed), "%s: packed weight must be 16-byte aligned", what);
            if (!ring) return launch(bee_message_kernel<T, true, true>, items);
            return edge_max ? launch(bee_message_ring_kernel<T, true, true>, items) : launch(bee_message_ring_kernel<T, false, true>, items);
        }
    }
    if (ring) {
        if constexpr (std::is_same<T, float>::value)
            if (edge_max) return launch(bee_message_ring_kernel<T, true, false>, items);
        if (!edge_max) return launch(bee_message_ring_kernel<T, false, false>, items);
    }
    // rows of a few edges do not repay the pipeline's start-up (one extra set of loads per row), unless the system
    // is so small that the chip is not filled and a row's chain of load latencies is all there is to the time
    return n_edges >= 8L * n_nodes || items <= 16384 ? launch(bee_message_kernel<T, true, false>, items) : launch(bee_message_kernel<T, false, false>, items);
}

extern "C" {

int mg_bee_edge_geometry(const float* r_ij, long n_edges, float r0, float* enc, float* rhat, mg_stream_t stream) {
    MG_REQUIRE(n_edges >= 0, "mg_bee_edge_geometry: negative size");
    MG_REQUIRE(r0 > 0.f, "mg_bee_edge_geometry: r0 must be positive");
    if (n_edges == 0) return MG_OK;
    MG_REQUIRE(r_ij && enc && rhat, "mg_bee_edge_geometry: null pointer");
    static const Jacobi8 table = jacobi_table();
    const float scale = (float)(7.0 / (double)r0);
    hipLaunchKernelGGL(bee_geometry_kernel, dim3((unsigned)ceil_div(n_edges, 256)), dim3(256), 0, (hipStream_t)stream,
                       r_ij, n_edges, r0, scale, table, enc, rhat);
    return check_launch("mg_bee_edge_geometry");
}

int mg_bee_message(const int* row_ptr, const int* dst, const int* node_order, int n_nodes, long n_edges,
                   const float* rhat, const float* enc, const float* La, const float* Lv, const float* Ld, int chan,
                   const float* enc_W, const float* enc_b, float* P0, float* S1, float* S2, float* node_max,
                   float* edge_max, mg_stream_t stream) {
    return launch_bee_message<float>("mg_bee_message", row_ptr, dst, node_order, n_nodes, n_edges, rhat, enc, La, Lv,
                                     Ld, chan, enc_W, enc_b, P0, S1, S2, node_max, edge_max, stream);
}

int mg_bee_message_rank2_supported(int chan, int dim_d) { return rank2_fusable(chan, dim_d) ? 1 : 0; }

int mg_bee_rank2_weight_bytes(int chan, size_t* bytes) {
    MG_REQUIRE(bytes != nullptr && chan >= 0, "mg_bee_rank2_weight_bytes: bad argument");
    *bytes = rank2_weight_bytes(chan);
    return MG_OK;
}

int mg_bee_pack_rank2_weight(const float* Y2, long ld, int chan, int dim_d, float* packed, mg_stream_t stream) {
    MG_REQUIRE(rank2_fusable(chan, dim_d), "mg_bee_pack_rank2_weight: needs chan = 64, 128 or 256 and dim_d <= 16");
    MG_REQUIRE(Y2 && packed && ld >= 5L * chan, "mg_bee_pack_rank2_weight: null pointer or short rows");
    const long chunks = chan / 64, total = chunks * (kRank2Fp32 + kRank2Pieces / 8);
    hipLaunchKernelGGL(rank2_weight_scales_kernel, dim3(16), dim3(256), 0, (hipStream_t)stream, Y2, ld, chan, dim_d,
                       packed + chunks * (kRank2Fp32 + kRank2Pieces / 2));
    if (int code = check_launch("rank2_weight_scales_kernel")) return code;
    hipLaunchKernelGGL(pack_rank2_weight_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, (hipStream_t)stream,
                       Y2, ld, chan, dim_d, packed);
    return check_launch("mg_bee_pack_rank2_weight");
}

int mg_bee_message_rank2(const int* row_ptr, const int* dst, const int* node_order, int n_nodes, long n_edges,
                         const float* rhat, const float* enc, const float* La, const float* Lv, const float* Ld, int chan,
                         const float* enc_W, const float* enc_b, const float* packed_Y2, int dim_d, float* P0, float* S1,
                         float* out_d, int accumulate, float* node_max, float* edge_max, mg_stream_t stream) {
    MG_REQUIRE(packed_Y2 != nullptr, "mg_bee_message_rank2: null weight");
    return launch_bee_message<float>("mg_bee_message_rank2", row_ptr, dst, node_order, n_nodes, n_edges, rhat, enc, La,
                                     Lv, Ld, chan, enc_W, enc_b, P0, S1, nullptr, node_max, edge_max, stream, packed_Y2,
                                     dim_d, out_d, accumulate);
}

int mg_bee_message_bf16(const int* row_ptr, const int* dst, const int* node_order, int n_nodes, long n_edges,
                        const float* rhat, const float* enc, const void* La, const void* Lv, const void* Ld, int chan,
                        const float* enc_W, const float* enc_b, void* P0, void* S1, void* S2, mg_stream_t stream) {
    return launch_bee_message<__bf16>("mg_bee_message_bf16", row_ptr, dst, node_order, n_nodes, n_edges, rhat, enc,
                                      static_cast<const __bf16*>(La), static_cast<const __bf16*>(Lv),
                                      static_cast<const __bf16*>(Ld), chan, enc_W, enc_b, static_cast<__bf16*>(P0),
                                      static_cast<__bf16*>(S1), static_cast<__bf16*>(S2), nullptr, nullptr, stream);
}

}  // extern "C"
