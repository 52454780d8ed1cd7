// The PaiNN layers under differentiation (archs/meanflow_painn8.py:25-100): the passes between the linear maps, forward and
// adjoint, for values alone and for (value, forward-mode tangent) pairs, as the meanflow loss differentiates them
// (archs/meanflow_painn8.py:274-296).  A pair travels as ONE array of 2 R rows, the values in the first R and the tangents in
// the last R, so that every linear map and every weight gradient of a pair is one launch over 2 R rows; the kernels here
// read and write both halves in one pass.
// What bounds them: nothing but memory traffic and launches.  In tensor arithmetic the same layers were two dozen launches a
// piece, each streaming its whole array (a training step of 3 blocks on 4096 nodes: 2400 launches, of which 1400 were
// elementwise or reductions); here every operand is read once and every result written once, and the row maxima that the
// split-fp16 linears scale by come out of the pass that writes the rows.
// DUAL = false: no tangents (R rows); the tangent operands are ignored.
#include "common.hpp"
#include "silu.hpp"
#include <algorithm>

namespace mg {
namespace {

struct Vec3 { float x, y, z; };
__device__ __forceinline__ Vec3 operator+(Vec3 a, Vec3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ Vec3 operator*(float s, Vec3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ Vec3 cross(Vec3 a, Vec3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float dot(Vec3 a, Vec3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// V channels of one row, and V channels x 3 components as they lie in memory: (c, k) at 3 c + k
template <int V>
struct Chans { float f[V]; };
using F4 = Chans<4>;
__device__ __forceinline__ F4 ld4(const float* p) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    return {{v.x, v.y, v.z, v.w}};
}
__device__ __forceinline__ void st4(float* p, const F4& v) {
    *reinterpret_cast<float4*>(p) = make_float4(v.f[0], v.f[1], v.f[2], v.f[3]);
}
__device__ __forceinline__ F4 zero4() { return {{0.f, 0.f, 0.f, 0.f}}; }

template <int V>
struct Vec3s {
    float f[3 * V];
    __device__ __forceinline__ Vec3 get(int j) const { return {f[3 * j], f[3 * j + 1], f[3 * j + 2]}; }
    __device__ __forceinline__ void set(int j, Vec3 v) { f[3 * j] = v.x; f[3 * j + 1] = v.y; f[3 * j + 2] = v.z; }
    __device__ __forceinline__ void add(int j, Vec3 v) { f[3 * j] += v.x; f[3 * j + 1] += v.y; f[3 * j + 2] += v.z; }
};
using Vec3x4 = Vec3s<4>;
__device__ __forceinline__ Vec3x4 ld12(const float* p) {
    Vec3x4 r;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const F4 v = ld4(p + 4 * q);
#pragma unroll
        for (int j = 0; j < 4; j++) r.f[4 * q + j] = v.f[j];
    }
    return r;
}
__device__ __forceinline__ void st12(float* p, const Vec3x4& r) {
#pragma unroll
    for (int q = 0; q < 3; q++) st4(p + 4 * q, {{r.f[4 * q], r.f[4 * q + 1], r.f[4 * q + 2], r.f[4 * q + 3]}});
}
__device__ __forceinline__ Vec3x4 zero12() {
    Vec3x4 r;
#pragma unroll
    for (int q = 0; q < 12; q++) r.f[q] = 0.f;
    return r;
}

// lanes that share a row of n values (n % 4 == 0): a power of two <= 64, so that a row never straddles waves
inline int row_lanes(int n) {
    int g = 1;
    while (g < 64 && 4 * g < n) g *= 2;
    return g;
}
__device__ __forceinline__ float group_max(float v, int lanes) {
    for (int s = 1; s < lanes; s <<= 1) v = fmaxf(v, __shfl_xor(v, s));
    return v;
}
__device__ __forceinline__ float group_sum(float v, int lanes) {
    for (int s = 1; s < lanes; s <<= 1) v += __shfl_xor(v, s);
    return v;
}
__device__ __forceinline__ float max4(float m, const F4& v) {
    return fmaxf(fmaxf(m, fmaxf(fabsf(v.f[0]), fabsf(v.f[1]))), fmaxf(fabsf(v.f[2]), fabsf(v.f[3])));
}

// ------------------------------------------------------------------------------------------------ activation of a layer
// h = SiLU(z), h_t = SiLU'(z) z_t, and the row maxima of both
template <bool DUAL>
__global__ void __launch_bounds__(256) silu_rows_fwd_kernel(const float* __restrict__ z, long R, int n, int lanes,
                                                            float* __restrict__ h, float* __restrict__ h_max) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long r_raw = t / lanes;
    const bool live = r_raw < R;
    const long r = live ? r_raw : R - 1;
    const int lane = (int)(t - r_raw * lanes);
    const long half = R * n;
    float mx = 0.f, mxt = 0.f;
    for (int c = 4 * lane; c < n; c += 4 * lanes) {
        const long k = r * n + c;
        const F4 v = ld4(z + k);
        F4 vt, o, ot;
        if constexpr (DUAL) vt = ld4(z + half + k);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const Silu s = silu(v.f[j]);
            o.f[j] = s.f;
            if constexpr (DUAL) ot.f[j] = s.d1 * vt.f[j];
        }
        mx = max4(mx, o);
        if (live) st4(h + k, o);
        if constexpr (DUAL) {
            mxt = max4(mxt, ot);
            if (live) st4(h + half + k, ot);
        }
    }
    mx = group_max(mx, lanes);
    if constexpr (DUAL) mxt = group_max(mxt, lanes);
    if (live && lane == 0) {
        h_max[r] = mx;
        if constexpr (DUAL) h_max[R + r] = mxt;
    }
}

// dz = dh SiLU'(z) + dh_t z_t SiLU''(z), dz_t = dh_t SiLU'(z), and the row maxima of both
template <bool DUAL>
__global__ void __launch_bounds__(256) silu_rows_bwd_kernel(const float* __restrict__ z, const float* __restrict__ dh, long R,
                                                            int n, int lanes, float* __restrict__ dz,
                                                            float* __restrict__ dz_max) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long r_raw = t / lanes;
    const bool live = r_raw < R;
    const long r = live ? r_raw : R - 1;
    const int lane = (int)(t - r_raw * lanes);
    const long half = R * n;
    float mx = 0.f, mxt = 0.f;
    for (int c = 4 * lane; c < n; c += 4 * lanes) {
        const long k = r * n + c;
        const F4 v = ld4(z + k), g = ld4(dh + k);
        F4 vt, gt, o, ot;
        if constexpr (DUAL) { vt = ld4(z + half + k); gt = ld4(dh + half + k); }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const Silu s = silu(v.f[j]);
            o.f[j] = g.f[j] * s.d1;
            if constexpr (DUAL) {
                o.f[j] += gt.f[j] * vt.f[j] * s.d2;
                ot.f[j] = gt.f[j] * s.d1;
            }
        }
        mx = max4(mx, o);
        if (live) st4(dz + k, o);
        if constexpr (DUAL) {
            mxt = max4(mxt, ot);
            if (live) st4(dz + half + k, ot);
        }
    }
    mx = group_max(mx, lanes);
    if constexpr (DUAL) mxt = group_max(mxt, lanes);
    if (live && lane == 0) {
        dz_max[r] = mx;
        if constexpr (DUAL) dz_max[R + r] = mxt;
    }
}

// ------------------------------------------------------------------------------------------------ edge vectors
// radial_encode: columns k < hn are cos(phase_k), the others sin(phase_{k - hn}), phase_k = (pi / rmax) (1 + k / 2) d
__device__ __forceinline__ float coefficient(int k, float pi_over_rmax) { return (float)(1 + k / 2) * pi_over_rmax; }

// enc (E or 2E, n), its row bounds, and u = r / sqrt(|r|^2 + eps) with its tangent
template <bool DUAL>
__global__ void __launch_bounds__(256) edge_encode_fwd_kernel(const float* __restrict__ r, const float* __restrict__ r_t, long E,
                                                              int n, int lanes, float pi_over_rmax, float eps,
                                                              float* __restrict__ enc, float* __restrict__ enc_bound,
                                                              float* __restrict__ dir, float* __restrict__ dir_t) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long e = t / lanes;
    if (e >= E) return;
    const int lane = (int)(t - e * lanes);
    const Vec3 x = {r[3 * e], r[3 * e + 1], r[3 * e + 2]};
    Vec3 xt = {0.f, 0.f, 0.f};
    if constexpr (DUAL) xt = {r_t[3 * e], r_t[3 * e + 1], r_t[3 * e + 2]};
    const float q = dot(x, x), d = sqrtf(q), inv_d = d > 0.f ? 1.0f / d : 0.f;
    const float p = dot(x, xt), d_t = p * inv_d;
    const int hn = (n + 1) / 2;
    for (int k = lane; k < n; k += lanes) {
        const bool is_sin = k >= hn;
        const float c = coefficient(is_sin ? k - hn : k, pi_over_rmax);
        float sn, cs;
        sincosf(d * c, &sn, &cs);
        enc[e * n + k] = is_sin ? sn : cs;
        if constexpr (DUAL) enc[(E + e) * n + k] = (is_sin ? cs : -sn) * (c * d_t);
    }
    if (lane == 0) {
        enc_bound[e] = 1.0f;
        if constexpr (DUAL) enc_bound[E + e] = fabsf(d_t) * coefficient(hn - 1, pi_over_rmax);
        const float s = 1.0f / sqrtf(q + eps);
        dir[3 * e] = s * x.x; dir[3 * e + 1] = s * x.y; dir[3 * e + 2] = s * x.z;
        if constexpr (DUAL) {
            const float b = s * s * s * p;
            dir_t[3 * e] = s * xt.x - b * x.x; dir_t[3 * e + 1] = s * xt.y - b * x.y; dir_t[3 * e + 2] = s * xt.z - b * x.z;
        }
    }
}

// its adjoint: g_enc (E or 2E, n), g_dir, g_dir_t -> g_r, g_r_t
template <bool DUAL>
__global__ void __launch_bounds__(256) edge_encode_bwd_kernel(const float* __restrict__ r, const float* __restrict__ r_t, long E,
                                                              int n, int lanes, float pi_over_rmax, float eps,
                                                              const float* __restrict__ g_enc, const float* __restrict__ g_dir,
                                                              const float* __restrict__ g_dir_t, float* __restrict__ g_r,
                                                              float* __restrict__ g_r_t) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long e_raw = t / lanes;
    const bool live = e_raw < E;
    const long e = live ? e_raw : E - 1;
    const int lane = (int)(t - e_raw * lanes);
    const Vec3 x = {r[3 * e], r[3 * e + 1], r[3 * e + 2]};
    Vec3 xt = {0.f, 0.f, 0.f};
    if constexpr (DUAL) xt = {r_t[3 * e], r_t[3 * e + 1], r_t[3 * e + 2]};
    const float q = dot(x, x), d = sqrtf(q), inv_d = d > 0.f ? 1.0f / d : 0.f;
    const float p = dot(x, xt), d_t = p * inv_d;
    const int hn = (n + 1) / 2;
    float g_d = 0.f, g_dt = 0.f;
    for (int k = lane; k < n; k += lanes) {
        const bool is_sin = k >= hn;
        const float c = coefficient(is_sin ? k - hn : k, pi_over_rmax);
        float sn, cs;
        sincosf(d * c, &sn, &cs);
        const float first = (is_sin ? cs : -sn) * c;
        g_d += g_enc[e * n + k] * first;
        if constexpr (DUAL) {
            const float gt = g_enc[(E + e) * n + k];
            g_d -= gt * (is_sin ? sn : cs) * c * c * d_t;
            g_dt += gt * first;
        }
    }
    g_d = group_sum(g_d, lanes);
    if constexpr (DUAL) g_dt = group_sum(g_dt, lanes);
    if (!live || lane != 0) return;
    const float s = 1.0f / sqrtf(q + eps), s3 = s * s * s;
    const Vec3 gu = {g_dir[3 * e], g_dir[3 * e + 1], g_dir[3 * e + 2]};
    Vec3 out = (g_d * inv_d - s3 * dot(x, gu)) * x + s * gu;
    if constexpr (DUAL) {
        const Vec3 gut = {g_dir_t[3 * e], g_dir_t[3 * e + 1], g_dir_t[3 * e + 2]};
        const float w = dot(x, gut);
        out = out + (g_dt * inv_d - s3 * w) * xt + (-s3 * p) * gut +
              (3.0f * s3 * s * s * p * w - s3 * dot(xt, gut) - g_dt * p * inv_d * inv_d * inv_d) * x;
        const Vec3 out_t = (g_dt * inv_d - s3 * w) * x + s * gut;
        g_r_t[3 * e] = out_t.x; g_r_t[3 * e + 1] = out_t.y; g_r_t[3 * e + 2] = out_t.z;
    }
    g_r[3 * e] = out.x; g_r[3 * e + 1] = out.y; g_r[3 * e + 2] = out.z;
}

// ------------------------------------------------------------------------------------------------ the message
// m = v p0 + (v x d) p1 + d p2, a = p3 with p = dist actv (archs/meanflow_painn8.py:94-100), summed over the edges of a
// source node, and the tangents of both sums: the tangent of a product has one term per factor, and all of them use the
// operands that the value loads.  One group of n / 4 lanes per source node walks its edges, as painn_combine_fwd_rows_kernel.
// Any of the four tangents may be a null pointer (that operand has none).
struct CombineIn {
    const float *dist, *dist_t, *actv, *actv_t, *v, *v_t, *dir, *dir_t;
};
// V floats (V even) at p, or zeros for a null pointer (uniform)
template <int V, class T>
__device__ __forceinline__ T ld_or_zero(const float* p, long off) {
    T r;
#pragma unroll
    for (int j = 0; j < V; j++) r.f[j] = 0.f;
    if (!p) return r;
    if constexpr (V % 4 == 0) {
#pragma unroll
        for (int q = 0; q < V; q += 4) {
            const float4 x = *reinterpret_cast<const float4*>(p + off + q);
            r.f[q] = x.x; r.f[q + 1] = x.y; r.f[q + 2] = x.z; r.f[q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int q = 0; q < V; q += 2) {
            const float2 x = *reinterpret_cast<const float2*>(p + off + q);
            r.f[q] = x.x; r.f[q + 1] = x.y;
        }
    }
    return r;
}
template <int V, class T>
__device__ __forceinline__ void st_unless_null(float* p, long off, const T& r) {
    if (!p) return;
    if constexpr (V % 4 == 0) {
#pragma unroll
        for (int q = 0; q < V; q += 4) *reinterpret_cast<float4*>(p + off + q) = make_float4(r.f[q], r.f[q + 1], r.f[q + 2], r.f[q + 3]);
    } else {
#pragma unroll
        for (int q = 0; q < V; q += 2) *reinterpret_cast<float2*>(p + off + q) = make_float2(r.f[q], r.f[q + 1]);
    }
}
// a + b with a rounded as it would be where it is stored: contracted into the product that a may be, x + q w moved a layer's results
// by a spacing of the sum, and with them the positions that a step subtracts from the old ones (an instruction more: the kernels wait
// for memory)
template <int V>
__device__ __forceinline__ Chans<V> plus(Chans<V> a, const Chans<V>& b) {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < V; j++) a.f[j] += b.f[j];
    return a;
}
template <int V>
__device__ __forceinline__ Vec3s<V> plus(Vec3s<V> a, const Vec3s<V>& b) {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < 3 * V; j++) a.f[j] += b.f[j];
    return a;
}
template <int V> __device__ __forceinline__ Chans<V> ld_chans(const float* p, long off) { return ld_or_zero<V, Chans<V>>(p, off); }
template <int V> __device__ __forceinline__ Vec3s<V> ld_vecs(const float* p, long off) { return ld_or_zero<3 * V, Vec3s<V>>(p, off); }
__device__ __forceinline__ Vec3 ld3_or_zero(const float* p, long off) {
    return p ? Vec3{p[off], p[off + 1], p[off + 2]} : Vec3{0.f, 0.f, 0.f};
}

// Workgroups go round-robin over the 8 XCDs: each XCD takes a contiguous eighth of the rows, whose neighbours' rows its L2 then holds
// (the grid is a multiple of 8 workgroups).  4 systems of 1024 atoms, 78 000 edges, 128 channels: 119 -> 113 us forward (mean of
// three blocks), 170 -> 155 adjoint; rows in no order (a random graph): no difference.
__device__ __forceinline__ long xcd_block() { return (long)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

template <int V>
__global__ void __launch_bounds__(256) combine_dual_fwd_kernel(CombineIn in, const int* __restrict__ node, long n_rows,
                                                               const int* __restrict__ row_ptr, long n_out, long E, int n,
                                                               mg_painn_rows res, float* __restrict__ out_v, float* __restrict__ out_vt,
                                                               float* __restrict__ out_a, float* __restrict__ out_at) {
    const int tpe = n / V;
    const long t = xcd_block() * 256 + threadIdx.x;
    const long r = t / tpe;
    if (r >= n_out) return;
    const int c = (int)(t - r * tpe) * V;
    Vec3s<V> am = ld_vecs<V>(nullptr, 0), amt = ld_vecs<V>(nullptr, 0);
    Chans<V> aa = ld_chans<V>(nullptr, 0), aat = ld_chans<V>(nullptr, 0);
    const long lo = max((long)row_ptr[r], 0L), hi = min((long)row_ptr[r + 1], E);
    long next = lo < hi ? (long)node[lo] : 0;                     // an edge ahead: its row's address is known when the edge begins
    for (long e = lo; e < hi; e++) {
        const long en = min(max(next, 0L), n_rows - 1);
        next = node[min(e + 1, hi - 1)];
        Chans<V> p[4], pt[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const Chans<V> d = ld_chans<V>(in.dist, e * 4 * n + k * n + c), a = ld_chans<V>(in.actv, en * 4 * n + k * n + c);
            const Chans<V> dt = ld_chans<V>(in.dist_t, e * 4 * n + k * n + c), at = ld_chans<V>(in.actv_t, en * 4 * n + k * n + c);
#pragma unroll
            for (int j = 0; j < V; j++) {
                p[k].f[j] = d.f[j] * a.f[j];
                pt[k].f[j] = dt.f[j] * a.f[j] + d.f[j] * at.f[j];
            }
        }
        const Vec3s<V> v = ld_vecs<V>(in.v, (en * n + c) * 3), vt = ld_vecs<V>(in.v_t, (en * n + c) * 3);
        const Vec3 d = ld3_or_zero(in.dir, 3 * e), dt = ld3_or_zero(in.dir_t, 3 * e);
#pragma unroll
        for (int j = 0; j < V; j++) {
            const Vec3 x = v.get(j), xt = vt.get(j), xd = cross(x, d);
            am.add(j, p[0].f[j] * x + p[1].f[j] * xd + p[2].f[j] * d);
            amt.add(j, p[0].f[j] * xt + pt[0].f[j] * x + p[1].f[j] * (cross(xt, d) + cross(x, dt)) + pt[1].f[j] * xd +
                           p[2].f[j] * dt + pt[2].f[j] * d);
            aa.f[j] += p[3].f[j];
            aat.f[j] += pt[3].f[j];
        }
    }
    st_unless_null<3 * V>(out_v, (r * n + c) * 3, plus(am, ld_vecs<V>(res.v, (r * n + c) * 3)));
    st_unless_null<3 * V>(out_vt, (r * n + c) * 3, plus(amt, ld_vecs<V>(res.v_t, (r * n + c) * 3)));
    st_unless_null<V>(out_a, r * n + c, plus(aa, ld_chans<V>(res.a, r * n + c)));
    st_unless_null<V>(out_at, r * n + c, plus(aat, ld_chans<V>(res.a_t, r * n + c)));
}

// Its adjoint, by destination row as painn_combine_bwd_rows_kernel: the gradients of actv and v (and of their tangents) are
// summed over the edges that read a row, those of dist and the direction stay per edge.  Outputs may be null.
struct CombineGrad {
    float *dist, *dist_t, *actv, *actv_t, *v, *v_t, *dir, *dir_t;
};
template <int V>
__global__ void __launch_bounds__(256, 2) combine_dual_bwd_kernel(CombineIn in, const int* __restrict__ row_ptr,
                                                                  const int* __restrict__ order, long n_rows,
                                                                  const float* __restrict__ gm, const float* __restrict__ gmt,
                                                                  const float* __restrict__ ga, const float* __restrict__ gat,
                                                                  const int* __restrict__ grad_row, long n_grad_rows, long E, int n,
                                                                  CombineGrad out, mg_painn_rows add) {
    const int tpe = n / V;                                        // a power of two <= 64: a group never straddles waves
    const long t = xcd_block() * 256 + threadIdx.x;
    const long r_raw = t / tpe;
    const bool live = r_raw < n_rows;
    const long r = live ? r_raw : n_rows - 1;
    const int c = (int)(t - r_raw * tpe) * V;
    Chans<V> a[4], at[4], acc_a[4], acc_at[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        a[k] = ld_chans<V>(in.actv, r * 4 * n + k * n + c);
        at[k] = ld_chans<V>(in.actv_t, r * 4 * n + k * n + c);
        acc_a[k] = ld_chans<V>(nullptr, 0);
        acc_at[k] = ld_chans<V>(nullptr, 0);
    }
    const Vec3s<V> v = ld_vecs<V>(in.v, (r * n + c) * 3), vt = ld_vecs<V>(in.v_t, (r * n + c) * 3);
    Vec3s<V> acc_v = ld_vecs<V>(nullptr, 0), acc_vt = ld_vecs<V>(nullptr, 0);
    const int lo = max(row_ptr[r], 0), hi = live ? min(row_ptr[r + 1], (int)min(E, 0x7fffffffL)) : lo;
    auto edge_at = [&](int pos) { return min(max(order ? (long)order[pos] : (long)pos, 0L), E - 1); };
    // the edge two positions ahead and the gradient row one ahead, so that neither index is waited for
    long e = 0, e_next = 0, eg = 0;
    if (lo < hi) {
        e = edge_at(lo);
        e_next = edge_at(min(lo + 1, hi - 1));
        eg = grad_row[e];
    }
    for (int pos = lo; pos < hi; pos++) {
        const long row = min(max(eg, 0L), n_grad_rows - 1);
        const Vec3s<V> g = ld_vecs<V>(gm, (row * n + c) * 3), gt = ld_vecs<V>(gmt, (row * n + c) * 3);
        const Chans<V> g3 = ld_chans<V>(ga, row * n + c), g3t = ld_chans<V>(gat, row * n + c);
        const Vec3 d = ld3_or_zero(in.dir, 3 * e), dt = ld3_or_zero(in.dir_t, 3 * e);
        Chans<V> f[4], ft[4], dp[4], dpt[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            f[k] = ld_chans<V>(in.dist, e * 4 * n + k * n + c);
            ft[k] = ld_chans<V>(in.dist_t, e * 4 * n + k * n + c);
        }
        const long e_now = e;
        e = e_next;
        eg = grad_row[e];
        e_next = edge_at(pos < hi - 2 ? pos + 2 : hi - 1);
        Vec3 gd = {0.f, 0.f, 0.f}, gdt = {0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < V; j++) {
            const Vec3 x = v.get(j), xt = vt.get(j), w = g.get(j), wt = gt.get(j), xd = cross(x, d);
            float p[3], pt[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                p[k] = f[k].f[j] * a[k].f[j];
                pt[k] = ft[k].f[j] * a[k].f[j] + f[k].f[j] * at[k].f[j];
            }
            dp[0].f[j] = dot(w, x) + dot(wt, xt);
            dpt[0].f[j] = dot(wt, x);
            dp[1].f[j] = dot(w, xd) + dot(wt, cross(xt, d) + cross(x, dt));
            dpt[1].f[j] = dot(wt, xd);
            dp[2].f[j] = dot(w, d) + dot(wt, dt);
            dpt[2].f[j] = dot(wt, d);
            dp[3].f[j] = g3.f[j];
            dpt[3].f[j] = g3t.f[j];
            const Vec3 d_wt = cross(d, wt);
            acc_v.add(j, p[0] * w + p[1] * (cross(d, w) + cross(dt, wt)) + pt[0] * wt + pt[1] * d_wt);
            acc_vt.add(j, p[0] * wt + p[1] * d_wt);
            const Vec3 wt_x = cross(wt, x);
            gd = gd + p[1] * (cross(w, x) + cross(wt, xt)) + p[2] * w + pt[1] * wt_x + pt[2] * wt;
            gdt = gdt + p[1] * wt_x + p[2] * wt;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            Chans<V> o, ot;
#pragma unroll
            for (int j = 0; j < V; j++) {
                o.f[j] = dp[k].f[j] * a[k].f[j] + dpt[k].f[j] * at[k].f[j];
                ot.f[j] = dpt[k].f[j] * a[k].f[j];
                acc_a[k].f[j] += dp[k].f[j] * f[k].f[j] + dpt[k].f[j] * ft[k].f[j];
                acc_at[k].f[j] += dpt[k].f[j] * f[k].f[j];
            }
            st_unless_null<V>(out.dist, e_now * 4 * n + k * n + c, o);
            st_unless_null<V>(out.dist_t, e_now * 4 * n + k * n + c, ot);
        }
        if (out.dir) {                                            // (uniform)
            for (int sh = 1; sh < tpe; sh <<= 1) {
                gd.x += __shfl_xor(gd.x, sh); gd.y += __shfl_xor(gd.y, sh); gd.z += __shfl_xor(gd.z, sh);
                gdt.x += __shfl_xor(gdt.x, sh); gdt.y += __shfl_xor(gdt.y, sh); gdt.z += __shfl_xor(gdt.z, sh);
            }
            if (c == 0) {
                float* o = out.dir + 3 * e_now;
                o[0] = gd.x; o[1] = gd.y; o[2] = gd.z;
                if (out.dir_t) {
                    float* ot = out.dir_t + 3 * e_now;
                    ot[0] = gdt.x; ot[1] = gdt.y; ot[2] = gdt.z;
                }
            }
        }
    }
    if (!live) return;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        st_unless_null<V>(out.actv, r * 4 * n + k * n + c, acc_a[k]);
        st_unless_null<V>(out.actv_t, r * 4 * n + k * n + c, acc_at[k]);
    }
    st_unless_null<3 * V>(out.v, (r * n + c) * 3, plus(acc_v, ld_vecs<V>(add.v, (r * n + c) * 3)));
    st_unless_null<3 * V>(out.v_t, (r * n + c) * 3, plus(acc_vt, ld_vecs<V>(add.v_t, (r * n + c) * 3)));
}

// ------------------------------------------------------------------------------------------------ the update
// (archs/meanflow_painn8.py:63-75)  lrv (R or 2R, 3, 3n): the three linear maps l, r, v of x_v, component-major.
//   ip = l . r,  cat = [x_a, |r|],  y = mlp(cat) = [y1, y2, y3],
//   out_a = groupnorm(ip y2) + y3,  out_v = w / sqrt(|w|^2 + 1) with w = v y1
__device__ __forceinline__ void ld_components(const float* lrv, long row, int n, int part, int c, F4 (&x)[3]) {
#pragma unroll
    for (int k = 0; k < 3; k++) x[k] = ld4(lrv + (row * 3 + k) * 3 * n + part * n + c);
}
__device__ __forceinline__ Vec3 comp(const F4 (&x)[3], int j) { return {x[0].f[j], x[1].f[j], x[2].f[j]}; }

template <bool DUAL>
__global__ void __launch_bounds__(256) update_pre_fwd_kernel(const float* __restrict__ lrv, const float* __restrict__ x_a,
                                                             const float* __restrict__ x_at, long R, int n, int lanes,
                                                             float* __restrict__ ip, float* __restrict__ cat,
                                                             float* __restrict__ cat_max) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long r_raw = t / lanes;
    const bool live = r_raw < R;
    const long r = live ? r_raw : R - 1;
    const int lane = (int)(t - r_raw * lanes);
    float mx = 0.f, mxt = 0.f;
    for (int c = 4 * lane; c < n; c += 4 * lanes) {
        F4 xl[3], xr[3], xlt[3], xrt[3];
        ld_components(lrv, r, n, 0, c, xl);
        ld_components(lrv, r, n, 1, c, xr);
        if constexpr (DUAL) {
            ld_components(lrv, R + r, n, 0, c, xlt);
            ld_components(lrv, R + r, n, 1, c, xrt);
        }
        F4 o, ot, nu, nut;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const Vec3 a = comp(xl, j), b = comp(xr, j);
            o.f[j] = dot(a, b);
            nu.f[j] = sqrtf(dot(b, b));
            if constexpr (DUAL) {
                const Vec3 at = comp(xlt, j), bt = comp(xrt, j);
                ot.f[j] = dot(at, b) + dot(a, bt);
                nut.f[j] = nu.f[j] > 0.f ? dot(b, bt) / nu.f[j] : 0.f;
            }
        }
        const F4 xa = ld4(x_a + r * n + c);
        mx = max4(max4(mx, nu), xa);
        if (live) {
            st4(ip + r * n + c, o);
            st4(cat + r * 2 * n + c, xa);
            st4(cat + r * 2 * n + n + c, nu);
        }
        if constexpr (DUAL) {
            const F4 xat = x_at ? ld4(x_at + r * n + c) : zero4();
            mxt = max4(max4(mxt, nut), xat);
            if (live) {
                st4(ip + (R + r) * n + c, ot);
                st4(cat + (R + r) * 2 * n + c, xat);
                st4(cat + (R + r) * 2 * n + n + c, nut);
            }
        }
    }
    mx = group_max(mx, lanes);
    if constexpr (DUAL) mxt = group_max(mxt, lanes);
    if (live && lane == 0) {
        cat_max[r] = mx;
        if constexpr (DUAL) cat_max[R + r] = mxt;
    }
}

// Group statistics of x = ip y2 over the nodes of a box and the channels of a group: pieces of kPiece values, each with its
// mean, sum of squared deviations, mean of the tangent and co-moment, which the readers merge in piece order.
constexpr int kPiece = 4096, kPieceStats = 5;      // count, mean, m2, mean of the tangent, co-moment
template <bool DUAL>
__global__ void __launch_bounds__(256) gn_pieces_kernel(const float* __restrict__ ip, const float* __restrict__ y, long R, int N,
                                                        int n, int groups, int pieces, float* __restrict__ part) {
    const int bg = blockIdx.x / pieces, piece = blockIdx.x - bg * pieces, b = bg / groups, g = bg - b * groups;
    const int cpg = n / groups;
    const long total = (long)N * cpg, lo = (long)piece * kPiece, hi = min(lo + kPiece, total);
    __shared__ float red[2][4];
    float x[kPiece / 256], xt[kPiece / 256];
    float sum = 0.f, sumt = 0.f;
#pragma unroll
    for (int i = 0; i < kPiece / 256; i++) {
        const long k = lo + i * 256 + threadIdx.x;
        x[i] = 0.f; xt[i] = 0.f;
        if (k < hi) {
            const long node = k / cpg, row = (long)b * N + node;
            const int c = g * cpg + (int)(k - node * cpg);
            const float i0 = ip[row * n + c], y2 = y[row * 3 * n + n + c];
            x[i] = i0 * y2;
            if constexpr (DUAL) xt[i] = ip[(R + row) * n + c] * y2 + i0 * y[(R + row) * 3 * n + n + c];
        }
        sum += x[i];
        sumt += xt[i];
    }
    auto block_sums = [&](float u, float w, float& su, float& sw) {
        u = group_sum(u, 64);
        w = group_sum(w, 64);
        __syncthreads();
        if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = u; red[1][threadIdx.x >> 6] = w; }
        __syncthreads();
        su = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        sw = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    };
    const float inv = 1.0f / (float)(hi - lo);
    float m, mt;
    block_sums(sum, sumt, m, mt);
    m *= inv;
    mt *= inv;
    sum = 0.f; sumt = 0.f;
#pragma unroll
    for (int i = 0; i < kPiece / 256; i++) {
        if (lo + i * 256 + threadIdx.x < hi) {
            const float dx = x[i] - m;
            sum += dx * dx;
            sumt += dx * (xt[i] - mt);
        }
    }
    float m2, cm;
    block_sums(sum, sumt, m2, cm);
    if (threadIdx.x == 0) {
        float* o = part + (((long)b * groups + g) * pieces + piece) * kPieceStats;
        o[0] = (float)(hi - lo); o[1] = m; o[2] = m2; o[3] = mt; o[4] = cm;
    }
}

// Per (box, group): mean, s = 1 / sqrt(var + eps), mean of the tangent, mean of c c_t.  One wave merges the pieces: each lane
// its share in order, the lanes pairwise.
struct GroupStats { float mean, s, mean_t, cov; };
__device__ __forceinline__ void merge(float (&a)[kPieceStats], const float (&b)[kPieceStats]) {
    const float cnt = a[0] + b[0];
    if (b[0] == 0.f) return;
    const float w = b[0] / cnt, d = b[1] - a[1], dt = b[3] - a[3];
    a[2] += b[2] + d * d * a[0] * w;
    a[4] += b[4] + d * dt * a[0] * w;
    a[1] += d * w;
    a[3] += dt * w;
    a[0] = cnt;
}
__global__ void __launch_bounds__(64) gn_finish_kernel(const float* __restrict__ part, int pieces, float eps,
                                                       GroupStats* __restrict__ stats) {
    const float* src = part + (long)blockIdx.x * pieces * kPieceStats;
    float a[kPieceStats] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = threadIdx.x; k < pieces; k += 64) {
        float b[kPieceStats];
#pragma unroll
        for (int q = 0; q < kPieceStats; q++) b[q] = src[k * kPieceStats + q];
        merge(a, b);
    }
    for (int d = 1; d < 64; d <<= 1) {
        float b[kPieceStats];
#pragma unroll
        for (int q = 0; q < kPieceStats; q++) b[q] = __shfl_down(a[q], d);
        if ((threadIdx.x & (2 * d - 1)) == 0) merge(a, b);
    }
    if (threadIdx.x == 0) stats[blockIdx.x] = {a[1], 1.0f / sqrtf(a[2] / a[0] + eps), a[3], a[4] / a[0]};
}

template <bool DUAL>
__global__ void __launch_bounds__(256) update_post_fwd_kernel(const float* __restrict__ lrv, const float* __restrict__ ip,
                                                              const float* __restrict__ y, const GroupStats* __restrict__ stats,
                                                              const float* __restrict__ gamma, const float* __restrict__ beta,
                                                              long R, int N, int n, int groups, mg_painn_rows res,
                                                              float* __restrict__ out_a, float* __restrict__ out_at,
                                                              float* __restrict__ out_v, float* __restrict__ out_vt) {
    const int quads = n >> 2, cpg = n / groups;
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long r = t / quads;
    if (r >= R) return;
    const int c = (int)(t - r * quads) * 4;
    const F4 i0 = ld4(ip + r * n + c), y1 = ld4(y + r * 3 * n + c), y2 = ld4(y + r * 3 * n + n + c), y3 = ld4(y + r * 3 * n + 2 * n + c);
    F4 i0t, y1t, y2t, y3t;
    F4 v[3], vt[3];
    ld_components(lrv, r, n, 2, c, v);
    if constexpr (DUAL) {
        const long rt = R + r;
        i0t = ld4(ip + rt * n + c); y1t = ld4(y + rt * 3 * n + c); y2t = ld4(y + rt * 3 * n + n + c); y3t = ld4(y + rt * 3 * n + 2 * n + c);
        ld_components(lrv, rt, n, 2, c, vt);
    }
    const GroupStats* st = stats + (r / N) * groups;
    F4 oa, oat;
    Vec3x4 ov, ovt;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const GroupStats s = st[(c + j) / cpg];
        const float gm = gamma[c + j];
        const float x = i0.f[j] * y2.f[j] - s.mean;
        oa.f[j] = gm * (x * s.s) + beta[c + j] + y3.f[j];
        const Vec3 w = y1.f[j] * comp(v, j);
        const float q = 1.0f / sqrtf(dot(w, w) + 1.0f);
        ov.set(j, q * w);
        if constexpr (DUAL) {
            const float xt = i0t.f[j] * y2.f[j] + i0.f[j] * y2t.f[j] - s.mean_t;
            oat.f[j] = gm * (xt * s.s - x * (s.s * s.s * s.s) * s.cov) + y3t.f[j];
            const Vec3 wt = y1.f[j] * comp(vt, j) + y1t.f[j] * comp(v, j);
            ovt.set(j, q * wt + (-q * q * q * dot(w, wt)) * w);
        }
    }
    st4(out_a + r * n + c, plus(oa, ld_chans<4>(res.a, r * n + c)));
    st12(out_v + (r * n + c) * 3, plus(ov, ld_vecs<4>(res.v, (r * n + c) * 3)));
    if constexpr (DUAL) {
        st4(out_at + r * n + c, plus(oat, ld_chans<4>(res.a_t, r * n + c)));
        st12(out_vt + (r * n + c) * 3, plus(ovt, ld_vecs<4>(res.v_t, (r * n + c) * 3)));
    }
}

// Sums over the nodes of a piece, per channel: of g, g c, g_t c, g_t c_t and g_t, where g, g_t are the gradients of out_a and
// c, c_t the centred x and its tangent.  Everything the adjoint of the norm sums is made of these.
constexpr int kGradNodes = 64, kGradSums = 5;
template <bool DUAL>
__global__ void __launch_bounds__(256) gn_grad_pieces_kernel(const float* __restrict__ ip, const float* __restrict__ y,
                                                             const GroupStats* __restrict__ stats, const float* __restrict__ g_a,
                                                             const float* __restrict__ g_at, long R, int N, int n, int groups,
                                                             int pieces, float* __restrict__ part) {
    const int b = blockIdx.x / pieces, piece = blockIdx.x - b * pieces;
    const int cpg = n / groups;
    const int lo = piece * kGradNodes, hi = min(lo + kGradNodes, N);
    __shared__ float red[256 * kGradSums];
    // threads of a block: `cols` channels x `lines` nodes side by side
    for (int c0 = 0; c0 < n; c0 += 256) {
        const int cols = min(n - c0, 256), lines = 256 / cols;
        const int line = threadIdx.x / cols, c = c0 + threadIdx.x - line * cols;
        float acc[kGradSums] = {0.f, 0.f, 0.f, 0.f, 0.f};
        if (line < lines) {
            const GroupStats s = stats[b * groups + c / cpg];
            for (int node = lo + line; node < hi; node += lines) {
                const long row = (long)b * N + node;
                const float i0 = ip[row * n + c], y2 = y[row * 3 * n + n + c];
                const float x = i0 * y2 - s.mean, g = g_a[row * n + c];
                acc[0] += g;
                acc[1] += g * x;
                if constexpr (DUAL) {
                    const float xt = ip[(R + row) * n + c] * y2 + i0 * y[(R + row) * 3 * n + n + c] - s.mean_t;
                    const float gt = g_at[row * n + c];
                    acc[2] += gt * x;
                    acc[3] += gt * xt;
                    acc[4] += gt;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kGradSums; q++) red[q * 256 + threadIdx.x] = acc[q];
        __syncthreads();
        if (line == 0) {
            float* o = part + ((long)(b * pieces + piece) * kGradSums) * n + c;
#pragma unroll
            for (int q = 0; q < kGradSums; q++) {
                float sum = 0.f;
                for (int l = 0; l < lines; l++) sum += red[q * 256 + l * cols + threadIdx.x];
                o[(long)q * n] = sum;
            }
        }
    }
}

// per (box, channel) sums over the pieces in order, and the gradients of gamma and beta over the boxes: a workgroup per channel
// (a wave per sum would be five lanes wide: the lanes of a wave take the pieces instead)
__global__ void __launch_bounds__(64) gn_grad_finish_kernel(const float* __restrict__ part, const GroupStats* __restrict__ stats,
                                                            int B, int n, int groups, int pieces, float* __restrict__ sums,
                                                            float* __restrict__ d_gamma, float* __restrict__ d_beta) {
    const int c = blockIdx.x, cpg = n / groups;
    float dg = 0.f, db = 0.f;
    for (int b = 0; b < B; b++) {
        float acc[kGradSums] = {0.f, 0.f, 0.f, 0.f, 0.f};
        for (int p = threadIdx.x; p < pieces; p += 64)
#pragma unroll
            for (int q = 0; q < kGradSums; q++) acc[q] += part[((long)(b * pieces + p) * kGradSums + q) * n + c];
#pragma unroll
        for (int q = 0; q < kGradSums; q++) acc[q] = group_sum(acc[q], 64);
        const GroupStats s = stats[b * groups + c / cpg];
        const float s_t = -s.s * s.s * s.s * s.cov;
        dg += s.s * (acc[1] + acc[3]) + s_t * acc[2];
        db += acc[0];
        if (threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < kGradSums; q++) sums[((long)b * kGradSums + q) * n + c] = acc[q];
    }
    if (threadIdx.x == 0) { d_gamma[c] = dg; d_beta[c] = db; }
}

// Gradients of y (R or 2R, 3n) with their row maxima, of ip (R or 2R, n), and of the v third of lrv.
template <bool DUAL>
__global__ void __launch_bounds__(256) update_post_bwd_kernel(const float* __restrict__ lrv, const float* __restrict__ ip,
                                                              const float* __restrict__ y, const GroupStats* __restrict__ stats,
                                                              const float* __restrict__ sums, const float* __restrict__ gamma,
                                                              const float* __restrict__ g_a, const float* __restrict__ g_at,
                                                              const float* __restrict__ g_v, const float* __restrict__ g_vt,
                                                              long R, int N, int n, int groups, int lanes,
                                                              float* __restrict__ g_y, float* __restrict__ g_y_max,
                                                              float* __restrict__ g_ip, float* __restrict__ g_lrv) {
    const int cpg = n / groups;
    const int rows_per_block = 256 / lanes;
    const long r_raw = (long)blockIdx.x * rows_per_block + threadIdx.x / lanes;
    const bool live = r_raw < R;
    const long r = live ? r_raw : R - 1;
    const int lane = threadIdx.x & (lanes - 1);
    const long b = r / N;
    // the group sums of this row's box, weighted by gamma: a handful of cached loads per lane
    const float M = (float)((long)N * cpg);
    float mx = 0.f, mxt = 0.f;
    for (int c = 4 * lane; c < n; c += 4 * lanes) {
        const F4 i0 = ld4(ip + r * n + c), y1 = ld4(y + r * 3 * n + c), y2 = ld4(y + r * 3 * n + n + c);
        const F4 ga = ld4(g_a + r * n + c);
        const Vec3x4 gv = ld12(g_v + (r * n + c) * 3);
        F4 i0t, y1t, y2t, gat;
        Vec3x4 gvt;
        F4 v[3], vt[3];
        ld_components(lrv, r, n, 2, c, v);
        if constexpr (DUAL) {
            const long rt = R + r;
            i0t = ld4(ip + rt * n + c); y1t = ld4(y + rt * 3 * n + c); y2t = ld4(y + rt * 3 * n + n + c);
            gat = ld4(g_at + r * n + c);
            gvt = ld12(g_vt + (r * n + c) * 3);
            ld_components(lrv, rt, n, 2, c, vt);
        }
        F4 o1, o2, o3, oi, o1t, o2t, o3t, oit, ov[3], ovt[3];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int grp = (c + j) / cpg;
            const GroupStats s = stats[b * groups + grp];
            const float* G = sums + ((long)b * groups + grp) * kGradSums;      // sums of a, a c, b c, b c_t, b over the group
            const float gm = gamma[c + j];
            const float x = i0.f[j] * y2.f[j] - s.mean, s3 = s.s * s.s * s.s, s_t = -s3 * s.cov;
            const float a = gm * ga.f[j];
            float dx = a * s.s, dxt = 0.f;
            if constexpr (DUAL) {
                const float xt = i0t.f[j] * y2.f[j] + i0.f[j] * y2t.f[j] - s.mean_t;
                const float bb = gm * gat.f[j];
                const float S = G[1] + G[3] - 3.0f * s.s * s.s * s.cov * G[2];
                dx += bb * s_t - (s3 * G[2] * xt + S * s3 * x + s.s * G[0] + s_t * G[4]) / M;
                dxt = bb * s.s - (s3 * G[2] * x + s.s * G[4]) / M;
                oi.f[j] = dx * y2.f[j] + dxt * y2t.f[j];
                oit.f[j] = dxt * y2.f[j];
                o2.f[j] = dx * i0.f[j] + dxt * i0t.f[j];
                o2t.f[j] = dxt * i0.f[j];
                o3t.f[j] = gat.f[j];
            } else {
                dx -= (G[1] * s3 * x + s.s * G[0]) / M;
                oi.f[j] = dx * y2.f[j];
                o2.f[j] = dx * i0.f[j];
            }
            o3.f[j] = ga.f[j];
            const Vec3 v0 = comp(v, j), w = y1.f[j] * v0, gw0 = gv.get(j);
            const float q = 1.0f / sqrtf(dot(w, w) + 1.0f), q3 = q * q * q;
            Vec3 gw = q * gw0 + (-q3 * dot(w, gw0)) * w;
            if constexpr (DUAL) {
                const Vec3 v0t = comp(vt, j), wt = y1.f[j] * v0t + y1t.f[j] * v0, gt = gvt.get(j);
                const float wwt = dot(w, wt), wg = dot(w, gt);
                gw = gw + (3.0f * q3 * q * q * wwt * wg - q3 * dot(wt, gt)) * w + (-q3 * wg) * wt + (-q3 * wwt) * gt;
                const Vec3 gwt = q * gt + (-q3 * wg) * w;
                const Vec3 dv = y1.f[j] * gw + y1t.f[j] * gwt, dvt = y1.f[j] * gwt;
                ov[0].f[j] = dv.x; ov[1].f[j] = dv.y; ov[2].f[j] = dv.z;
                ovt[0].f[j] = dvt.x; ovt[1].f[j] = dvt.y; ovt[2].f[j] = dvt.z;
                o1.f[j] = dot(gw, v0) + dot(gwt, v0t);
                o1t.f[j] = dot(gwt, v0);
            } else {
                const Vec3 dv = y1.f[j] * gw;
                ov[0].f[j] = dv.x; ov[1].f[j] = dv.y; ov[2].f[j] = dv.z;
                o1.f[j] = dot(gw, v0);
            }
        }
        mx = max4(max4(max4(mx, o1), o2), o3);
        if constexpr (DUAL) mxt = max4(max4(max4(mxt, o1t), o2t), o3t);
        if (live) {
            st4(g_y + r * 3 * n + c, o1); st4(g_y + r * 3 * n + n + c, o2); st4(g_y + r * 3 * n + 2 * n + c, o3);
            st4(g_ip + r * n + c, oi);
#pragma unroll
            for (int k = 0; k < 3; k++) st4(g_lrv + (r * 3 + k) * 3 * n + 2 * n + c, ov[k]);
            if constexpr (DUAL) {
                const long rt = R + r;
                st4(g_y + rt * 3 * n + c, o1t); st4(g_y + rt * 3 * n + n + c, o2t); st4(g_y + rt * 3 * n + 2 * n + c, o3t);
                st4(g_ip + rt * n + c, oit);
#pragma unroll
                for (int k = 0; k < 3; k++) st4(g_lrv + (rt * 3 + k) * 3 * n + 2 * n + c, ovt[k]);
            }
        }
    }
    mx = group_max(mx, lanes);
    if constexpr (DUAL) mxt = group_max(mxt, lanes);
    if (live && lane == 0) {
        g_y_max[r] = mx;
        if constexpr (DUAL) g_y_max[R + r] = mxt;
    }
}

// sums of gamma-weighted channel sums per group: (box, group, 5)
__global__ void __launch_bounds__(64) gn_grad_groups_kernel(const float* __restrict__ sums, const float* __restrict__ gamma,
                                                            int n, int groups, float* __restrict__ out) {
    const int b = blockIdx.x / groups, g = blockIdx.x - b * groups, cpg = n / groups;
#pragma unroll
    for (int q = 0; q < kGradSums; q++) {
        float acc = 0.f;
        for (int i = threadIdx.x; i < cpg; i += 64) acc += gamma[g * cpg + i] * sums[((long)b * kGradSums + q) * n + g * cpg + i];
        acc = group_sum(acc, 64);
        if (threadIdx.x == 0) out[((long)b * groups + g) * kGradSums + q] = acc;
    }
}

// Gradients of the l and r thirds of lrv and of x_a; row maxima of all of g_lrv's rows (the v third is there already).
template <bool DUAL>
__global__ void __launch_bounds__(256) update_pre_bwd_kernel(const float* __restrict__ lrv, const float* __restrict__ g_ip,
                                                             const float* __restrict__ g_cat, long R, int n, int lanes,
                                                             float* __restrict__ g_lrv, float* __restrict__ g_lrv_max,
                                                             mg_painn_rows add, float* __restrict__ g_xa) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long r_raw = t / lanes;
    const bool live = r_raw < R;
    const long r = live ? r_raw : R - 1, rt = R + r;
    const int lane = (int)(t - r_raw * lanes);
    float mx[3] = {0.f, 0.f, 0.f}, mxt[3] = {0.f, 0.f, 0.f};
    for (int c = 4 * lane; c < n; c += 4 * lanes) {
        F4 xl[3], xr[3], xlt[3], xrt[3], gl[3], gr[3], glt[3], grt[3], gv[3], gvt[3];
        ld_components(lrv, r, n, 0, c, xl);
        ld_components(lrv, r, n, 1, c, xr);
        ld_components(g_lrv, r, n, 2, c, gv);
        const F4 gi = ld4(g_ip + r * n + c), gn = ld4(g_cat + r * 2 * n + n + c);
        F4 git, gnt;
        if constexpr (DUAL) {
            ld_components(lrv, rt, n, 0, c, xlt);
            ld_components(lrv, rt, n, 1, c, xrt);
            ld_components(g_lrv, rt, n, 2, c, gvt);
            git = ld4(g_ip + rt * n + c);
            gnt = ld4(g_cat + rt * 2 * n + n + c);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const Vec3 a = comp(xl, j), b = comp(xr, j);
            const float nu = sqrtf(dot(b, b)), inv = nu > 0.f ? 1.0f / nu : 0.f;
            Vec3 da = gi.f[j] * b, db = gi.f[j] * a + (gn.f[j] * inv) * b;
            if constexpr (DUAL) {
                const Vec3 at = comp(xlt, j), bt = comp(xrt, j);
                da = da + git.f[j] * bt;
                db = db + git.f[j] * at + (gnt.f[j] * inv) * bt + (-gnt.f[j] * dot(b, bt) * inv * inv * inv) * b;
                const Vec3 dat = git.f[j] * b, dbt = git.f[j] * a + (gnt.f[j] * inv) * b;
                glt[0].f[j] = dat.x; glt[1].f[j] = dat.y; glt[2].f[j] = dat.z;
                grt[0].f[j] = dbt.x; grt[1].f[j] = dbt.y; grt[2].f[j] = dbt.z;
            }
            gl[0].f[j] = da.x; gl[1].f[j] = da.y; gl[2].f[j] = da.z;
            gr[0].f[j] = db.x; gr[1].f[j] = db.y; gr[2].f[j] = db.z;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            mx[k] = max4(max4(max4(mx[k], gl[k]), gr[k]), gv[k]);
            if constexpr (DUAL) mxt[k] = max4(max4(max4(mxt[k], glt[k]), grt[k]), gvt[k]);
        }
        if (live) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                st4(g_lrv + (r * 3 + k) * 3 * n + c, gl[k]);
                st4(g_lrv + (r * 3 + k) * 3 * n + n + c, gr[k]);
                if constexpr (DUAL) {
                    st4(g_lrv + (rt * 3 + k) * 3 * n + c, glt[k]);
                    st4(g_lrv + (rt * 3 + k) * 3 * n + n + c, grt[k]);
                }
            }
            st4(g_xa + r * n + c, plus(ld4(g_cat + r * 2 * n + c), ld_chans<4>(add.a, r * n + c)));
            if constexpr (DUAL) st4(g_xa + rt * n + c, plus(ld4(g_cat + rt * 2 * n + c), ld_chans<4>(add.a_t, r * n + c)));
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        mx[k] = group_max(mx[k], lanes);
        if constexpr (DUAL) mxt[k] = group_max(mxt[k], lanes);
        if (live && lane == 0) {
            g_lrv_max[r * 3 + k] = mx[k];
            if constexpr (DUAL) g_lrv_max[rt * 3 + k] = mxt[k];
        }
    }
}

bool rows_ok(long R, int n) { return R >= 0 && n >= 4 && n % 4 == 0; }
unsigned row_blocks(long R, int lanes) { return (unsigned)ceil_div(R * lanes, 256); }

}  // namespace
}  // namespace mg

using namespace mg;

// launches KERNEL<true> or KERNEL<false>
#define MG_DUAL_LAUNCH(KERNEL, GRID, BLOCK, ...)                                                          \
    do {                                                                                                  \
        if (dual) hipLaunchKernelGGL((KERNEL<true>), GRID, BLOCK, 0, (hipStream_t)stream, __VA_ARGS__);   \
        else hipLaunchKernelGGL((KERNEL<false>), GRID, BLOCK, 0, (hipStream_t)stream, __VA_ARGS__);       \
    } while (0)

extern "C" {

int mg_silu_rows_fwd(const float* z, long rows, int n, int dual, float* h, float* h_rowmax, mg_stream_t stream) {
    MG_REQUIRE(rows_ok(rows, n) && z && h && h_rowmax && aligned16(z) && aligned16(h),
               "mg_silu_rows_fwd: n % 4 == 0 and aligned arrays expected");
    if (rows == 0) return MG_OK;
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(silu_rows_fwd_kernel, dim3(row_blocks(rows, lanes)), dim3(256), z, rows, n, lanes, h, h_rowmax);
    return check_launch("mg_silu_rows_fwd");
}

int mg_silu_rows_bwd(const float* z, const float* dh, long rows, int n, int dual, float* dz, float* dz_rowmax, mg_stream_t stream) {
    MG_REQUIRE(rows_ok(rows, n) && z && dh && dz && dz_rowmax && aligned16(z) && aligned16(dh) && aligned16(dz),
               "mg_silu_rows_bwd: n % 4 == 0 and aligned arrays expected");
    if (rows == 0) return MG_OK;
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(silu_rows_bwd_kernel, dim3(row_blocks(rows, lanes)), dim3(256), z, dh, rows, n, lanes, dz, dz_rowmax);
    return check_launch("mg_silu_rows_bwd");
}

int mg_painn_edge_encode_fwd(const float* r, const float* r_t, long E, int n, float rmax, float eps, float* enc, float* enc_bound,
                             float* dir, float* dir_t, mg_stream_t stream) {
    const bool dual = r_t != nullptr;
    MG_REQUIRE(E >= 0 && n >= 1 && rmax > 0.f, "mg_painn_edge_encode_fwd: bad argument");
    if (E == 0) return MG_OK;
    MG_REQUIRE(r && enc && enc_bound && dir && (!dual || dir_t), "mg_painn_edge_encode_fwd: null pointer");
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(edge_encode_fwd_kernel, dim3(row_blocks(E, lanes)), dim3(256), r, r_t, E, n, lanes, (float)(M_PI / (double)rmax),
                   eps, enc, enc_bound, dir, dir_t);
    return check_launch("mg_painn_edge_encode_fwd");
}

int mg_painn_edge_encode_bwd(const float* r, const float* r_t, long E, int n, float rmax, float eps, const float* g_enc,
                             const float* g_dir, const float* g_dir_t, float* g_r, float* g_r_t, mg_stream_t stream) {
    const bool dual = r_t != nullptr;
    MG_REQUIRE(E >= 0 && n >= 1 && rmax > 0.f, "mg_painn_edge_encode_bwd: bad argument");
    if (E == 0) return MG_OK;
    MG_REQUIRE(r && g_enc && g_dir && g_r && (!dual || (g_dir_t && g_r_t)), "mg_painn_edge_encode_bwd: null pointer");
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(edge_encode_bwd_kernel, dim3(row_blocks(E, lanes)), dim3(256), r, r_t, E, n, lanes, (float)(M_PI / (double)rmax),
                   eps, g_enc, g_dir, g_dir_t, g_r, g_r_t);
    return check_launch("mg_painn_edge_encode_bwd");
}

static bool combine_aligned(const mg_painn_combine_dual* a) {
    for (const float* p : {a->dist, a->dist_t, a->actv, a->actv_t, a->v, a->v_t})
        if (!aligned16(p)) return false;
    return true;
}

static mg_painn_rows rows_or_none(const mg_painn_rows* p) { return p ? *p : mg_painn_rows{nullptr, nullptr, nullptr, nullptr}; }
static bool rows_aligned(const mg_painn_rows& p) { return aligned16(p.a) && aligned16(p.a_t) && aligned16(p.v) && aligned16(p.v_t); }

// Channels of a lane of the message kernels: two, so that a row of 128 channels is a whole wave and a lane's operands leave room for
// several waves on a SIMD (the adjoint: 153 registers, three waves; with four channels 266, one); four where two would spread a row
// over two waves (n = 256).  78 000 edges of 4096 nodes in no order, before (four channels a lane) -> now: n = 128 forward
// 140 -> 133 us (320 MB of filters and 550 MB of gathered rows out of the caches: 6.5 TB/s), adjoint 265 -> 212; n = 64 78 -> 72 and
// 144 -> 118; n = 256 275 -> 269 and, bounded to two waves, 478 -> 354.
static int combine_channels(int n) { return n <= 128 ? 2 : 4; }

int mg_painn_combine_dual_fwd(const mg_painn_combine_dual* a, const int* node, const int* row_ptr, long n_out, float* out_v,
                              float* out_v_t, float* out_a, float* out_a_t, mg_stream_t stream) {
    return mg_painn_combine_dual_add_fwd(a, node, row_ptr, n_out, nullptr, out_v, out_v_t, out_a, out_a_t, stream);
}

int mg_painn_combine_dual_add_fwd(const mg_painn_combine_dual* a, const int* node, const int* row_ptr, long n_out,
                                  const mg_painn_rows* residual, float* out_v, float* out_v_t, float* out_a, float* out_a_t,
                                  mg_stream_t stream) {
    const mg_painn_rows res = rows_or_none(residual);
    MG_REQUIRE(a != nullptr && a->E >= 0 && a->n_rows >= 0 && n_out >= 0 && mg_painn_combine_supported(a->n),
               "mg_painn_combine_dual_fwd: n must be a power of two in 4..256");
    if (n_out == 0) return MG_OK;
    MG_REQUIRE(row_ptr && out_v && out_v_t && out_a && out_a_t && aligned16(out_v) && aligned16(out_v_t) && aligned16(out_a) &&
                   aligned16(out_a_t) && combine_aligned(a) && rows_aligned(res) &&
                   (a->E == 0 || (a->dist && a->actv && a->v && a->dir && node && a->n_rows > 0)),
               "mg_painn_combine_dual_fwd: null or unaligned pointer");
    const CombineIn in{a->dist, a->dist_t, a->actv, a->actv_t, a->v, a->v_t, a->dir, a->dir_t};
    const int per_lane = combine_channels(a->n);
    hipLaunchKernelGGL(per_lane == 2 ? combine_dual_fwd_kernel<2> : combine_dual_fwd_kernel<4>,
                       dim3((unsigned)(8 * ceil_div(n_out * (a->n / per_lane), 8 * 256))), dim3(256), 0, (hipStream_t)stream, in, node,
                       a->n_rows, row_ptr, n_out, a->E, a->n, res, out_v, out_v_t, out_a, out_a_t);
    return check_launch("mg_painn_combine_dual_fwd");
}

int mg_painn_combine_dual_bwd(const mg_painn_combine_dual* a, const int* row_ptr, const int* order, const float* g_v,
                              const float* g_v_t, const float* g_a, const float* g_a_t, const int* grad_row, long n_grad_rows,
                              const mg_painn_combine_dual_grad* d, mg_stream_t stream) {
    return mg_painn_combine_dual_add_bwd(a, row_ptr, order, g_v, g_v_t, g_a, g_a_t, grad_row, n_grad_rows, nullptr, d, stream);
}

int mg_painn_combine_dual_add_bwd(const mg_painn_combine_dual* a, const int* row_ptr, const int* order, const float* g_v,
                                  const float* g_v_t, const float* g_a, const float* g_a_t, const int* grad_row, long n_grad_rows,
                                  const mg_painn_rows* added, const mg_painn_combine_dual_grad* d, mg_stream_t stream) {
    const mg_painn_rows add = rows_or_none(added);
    MG_REQUIRE(a != nullptr && d != nullptr && a->E >= 0 && a->E < (1L << 31) && a->n_rows >= 0 && mg_painn_combine_supported(a->n),
               "mg_painn_combine_dual_bwd: n must be a power of two in 4..256");
    if (a->n_rows == 0) return MG_OK;
    MG_REQUIRE(a->actv && a->v && row_ptr && combine_aligned(a) &&
                   (a->E == 0 || (a->dist && a->dir && g_v && g_v_t && g_a && g_a_t && grad_row && n_grad_rows > 0)) &&
                   aligned16(g_v) && aligned16(g_v_t) && aligned16(g_a) && aligned16(g_a_t) && rows_aligned(add),
               "mg_painn_combine_dual_bwd: null or unaligned pointer");
    for (const float* p : {d->dist, d->dist_t, d->actv, d->actv_t, d->v, d->v_t})
        MG_REQUIRE(aligned16(p), "mg_painn_combine_dual_bwd: gradients must be 16-byte aligned");
    const CombineIn in{a->dist, a->dist_t, a->actv, a->actv_t, a->v, a->v_t, a->dir, a->dir_t};
    const CombineGrad out{d->dist, d->dist_t, d->actv, d->actv_t, d->v, d->v_t, d->dir, d->dir_t};
    const int per_lane = combine_channels(a->n);
    hipLaunchKernelGGL(per_lane == 2 ? combine_dual_bwd_kernel<2> : combine_dual_bwd_kernel<4>,
                       dim3((unsigned)(8 * ceil_div(a->n_rows * (a->n / per_lane), 8 * 256))), dim3(256), 0, (hipStream_t)stream, in, row_ptr, order, a->n_rows, g_v, g_v_t, g_a, g_a_t, grad_row, n_grad_rows, a->E, a->n,
                       out, add);
    return check_launch("mg_painn_combine_dual_bwd");
}

int mg_painn_update_pre_fwd(const float* lrv, const float* x_a, const float* x_a_t, long rows, int n, int dual, float* ip,
                            float* cat, float* cat_rowmax, mg_stream_t stream) {
    MG_REQUIRE(rows_ok(rows, n), "mg_painn_update_pre_fwd: n % 4 == 0 expected");
    if (rows == 0) return MG_OK;
    MG_REQUIRE(lrv && x_a && ip && cat && cat_rowmax && aligned16(lrv) && aligned16(x_a) && aligned16(x_a_t) && aligned16(ip) &&
                   aligned16(cat),
               "mg_painn_update_pre_fwd: null or unaligned pointer");
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(update_pre_fwd_kernel, dim3(row_blocks(rows, lanes)), dim3(256), lrv, x_a, x_a_t, rows, n, lanes, ip, cat,
                   cat_rowmax);
    return check_launch("mg_painn_update_pre_fwd");
}

// floats of scratch: the forward pass's pieces; the backward pass's pieces, channel sums and group sums
int mg_painn_update_scratch_floats(int batch, int nodes, int n, int groups, long* forward, long* backward) {
    MG_REQUIRE(batch >= 0 && nodes >= 0 && groups >= 1 && n % groups == 0 && forward && backward,
               "mg_painn_update_scratch_floats: bad argument");
    *forward = (long)batch * groups * ceil_div((long)nodes * (n / groups), kPiece) * kPieceStats;
    *backward = (long)batch * kGradSums * ((ceil_div(nodes, kGradNodes) + 1) * (long)n + groups);
    return MG_OK;
}

int mg_painn_update_post_fwd(const float* lrv, const float* ip, const float* y, const float* gamma, const float* beta, int batch,
                             int nodes, int n, int groups, float eps, int dual, float* scratch, float* stats, float* out_a,
                             float* out_v, mg_stream_t stream) {
    const long values = (long)batch * nodes * n;
    return mg_painn_update_post_add_fwd(lrv, ip, y, gamma, beta, batch, nodes, n, groups, eps, dual, scratch, stats, nullptr, out_a,
                                        dual && out_a ? out_a + values : nullptr, out_v, dual && out_v ? out_v + 3 * values : nullptr,
                                        stream);
}

int mg_painn_update_post_add_fwd(const float* lrv, const float* ip, const float* y, const float* gamma, const float* beta, int batch,
                                 int nodes, int n, int groups, float eps, int dual, float* scratch, float* stats,
                                 const mg_painn_rows* residual, float* out_a, float* out_a_t, float* out_v, float* out_v_t,
                                 mg_stream_t stream) {
    const mg_painn_rows res = rows_or_none(residual);
    const long R = (long)batch * nodes;
    MG_REQUIRE(batch >= 0 && nodes >= 0 && groups >= 1 && rows_ok(R, n) && n % groups == 0,
               "mg_painn_update_post_fwd: bad shape");
    if (R == 0) return MG_OK;
    MG_REQUIRE(lrv && ip && y && gamma && beta && scratch && stats && out_a && out_v && aligned16(lrv) && aligned16(ip) &&
                   aligned16(y) && aligned16(out_a) && aligned16(out_v) && aligned16(stats) && rows_aligned(res) &&
                   (!dual || (out_a_t && out_v_t && aligned16(out_a_t) && aligned16(out_v_t))),
               "mg_painn_update_post_fwd: null or unaligned pointer");
    const int pieces = (int)ceil_div((long)nodes * (n / groups), kPiece);
    MG_REQUIRE((long)pieces * groups * batch <= 0x7fffffffL, "mg_painn_update_post_fwd: too many boxes");
    GroupStats* st = reinterpret_cast<GroupStats*>(stats);
    MG_DUAL_LAUNCH(gn_pieces_kernel, dim3((unsigned)(pieces * groups * batch)), dim3(256), ip, y, R, nodes, n, groups, pieces, scratch);
    hipLaunchKernelGGL(gn_finish_kernel, dim3((unsigned)(batch * groups)), dim3(64), 0, (hipStream_t)stream, scratch, pieces, eps, st);
    MG_DUAL_LAUNCH(update_post_fwd_kernel, dim3((unsigned)ceil_div(R * (n / 4), 256)), dim3(256), lrv, ip, y, st, gamma, beta, R,
                   nodes, n, groups, res, out_a, out_a_t, out_v, out_v_t);
    return check_launch("mg_painn_update_post_fwd");
}

int mg_painn_update_post_bwd(const float* lrv, const float* ip, const float* y, const float* stats, const float* gamma,
                             const float* g_a, const float* g_a_t, const float* g_v, const float* g_v_t, int batch, int nodes, int n,
                             int groups, int dual, float* scratch, float* g_y, float* g_y_rowmax, float* g_ip, float* g_lrv,
                             float* d_gamma, float* d_beta, mg_stream_t stream) {
    const long R = (long)batch * nodes;
    MG_REQUIRE(batch >= 1 && nodes >= 1 && groups >= 1 && rows_ok(R, n) && n % groups == 0,
               "mg_painn_update_post_bwd: bad shape");
    MG_REQUIRE(lrv && ip && y && stats && gamma && g_a && g_v && (!dual || (g_a_t && g_v_t)) && scratch && g_y && g_y_rowmax && g_ip &&
                   g_lrv && d_gamma && d_beta,
               "mg_painn_update_post_bwd: null pointer");
    MG_REQUIRE(aligned16(lrv) && aligned16(ip) && aligned16(y) && aligned16(stats) && aligned16(g_a) && aligned16(g_a_t) &&
                   aligned16(g_v) && aligned16(g_v_t) && aligned16(g_y) && aligned16(g_ip) && aligned16(g_lrv),
               "mg_painn_update_post_bwd: unaligned pointer");
    const int pieces = (int)ceil_div(nodes, kGradNodes);
    MG_REQUIRE((long)std::max(pieces, groups) * batch <= 0x7fffffffL, "mg_painn_update_post_bwd: too many boxes");
    const GroupStats* st = reinterpret_cast<const GroupStats*>(stats);
    float* channel = scratch + (long)batch * pieces * kGradSums * n;
    float* group = channel + (long)batch * kGradSums * n;
    hipStream_t s = (hipStream_t)stream;
    MG_DUAL_LAUNCH(gn_grad_pieces_kernel, dim3((unsigned)(pieces * batch)), dim3(256), ip, y, st, g_a, g_a_t, R, nodes, n, groups, pieces, scratch);
    hipLaunchKernelGGL(gn_grad_finish_kernel, dim3((unsigned)n), dim3(64), 0, s, scratch, st, batch, n, groups, pieces, channel,
                       d_gamma, d_beta);
    hipLaunchKernelGGL(gn_grad_groups_kernel, dim3((unsigned)(groups * batch)), dim3(64), 0, s, channel, gamma, n, groups, group);
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(update_post_bwd_kernel, dim3(row_blocks(R, lanes)), dim3(256), lrv, ip, y, st, group, gamma, g_a, g_a_t, g_v, g_v_t,
                   R, nodes, n, groups, lanes, g_y, g_y_rowmax, g_ip, g_lrv);
    return check_launch("mg_painn_update_post_bwd");
}

int mg_painn_update_pre_bwd(const float* lrv, const float* g_ip, const float* g_cat, long rows, int n, int dual, float* g_lrv,
                            float* g_lrv_rowmax, float* g_xa, mg_stream_t stream) {
    return mg_painn_update_pre_add_bwd(lrv, g_ip, g_cat, rows, n, dual, g_lrv, g_lrv_rowmax, nullptr, g_xa, stream);
}

int mg_painn_update_pre_add_bwd(const float* lrv, const float* g_ip, const float* g_cat, long rows, int n, int dual, float* g_lrv,
                                float* g_lrv_rowmax, const mg_painn_rows* added, float* g_xa, mg_stream_t stream) {
    const mg_painn_rows add = rows_or_none(added);
    MG_REQUIRE(rows_ok(rows, n), "mg_painn_update_pre_bwd: n % 4 == 0 expected");
    if (rows == 0) return MG_OK;
    MG_REQUIRE(lrv && g_ip && g_cat && g_lrv && g_lrv_rowmax && g_xa && aligned16(lrv) && aligned16(g_ip) && aligned16(g_cat) &&
                   aligned16(g_lrv) && aligned16(g_xa) && rows_aligned(add),
               "mg_painn_update_pre_bwd: null or unaligned pointer");
    const int lanes = row_lanes(n);
    MG_DUAL_LAUNCH(update_pre_bwd_kernel, dim3(row_blocks(rows, lanes)), dim3(256), lrv, g_ip, g_cat, rows, n, lanes, g_lrv,
                   g_lrv_rowmax, add, g_xa);
    return check_launch("mg_painn_update_pre_bwd");
}

}  // extern "C"
