// Node-level pieces of the layers that call the hot path: group norms over the
// atoms of a box, the tensor squash, the elementwise parts of the PaiNN update, and
// the remaining radial encodings.  All HBM-bound streaming over node-sized (or, for
// the encodings, edge-sized) arrays; the norms need one box-wide reduction each.
//
// Reductions are deterministic: workgroup partials in a caller-provided scratch
// array (fp64), folded in a fixed order by the apply kernels.
#include "common.hpp"

namespace mg {
namespace {

constexpr int kChunks = 64;   // partial sums per (box, group)

__device__ __forceinline__ double block_sum(double v, double* lds) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d);
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    double t = 0.0;
    for (int k = 0; k < (int)(blockDim.x / kWave); k++) t += lds[k];
    return t;
}

// x element (box b, node i, channel c, comp t) at x[((b*N + i)*x_stride + c)*T + t]; optional elementwise
// multiplier mul at the same index pattern with mul_stride.  partial[(b*G + g)*kChunks + chunk][0..1] =
// (sum, sum of squares) over that chunk's nodes, the group's channels and all components.
// A group's channels and components of one node are cg*T consecutive floats, so an element is addressed by its
// node and its offset in that run; both advance by constants from one trip to the next (no division per element).
__global__ void __launch_bounds__(256) group_stats_kernel(const float* __restrict__ x, long x_stride,
                                                          const float* __restrict__ mul, long mul_stride, int N,
                                                          int chan, int groups, int T, double* __restrict__ partial) {
    __shared__ double lds[8];
    const int bg = blockIdx.x, chunk = blockIdx.y;
    const int b = bg / groups, g = bg - b * groups;
    const int cg = chan / groups;
    const int per = (N + kChunks - 1) / kChunks;
    const int n_lo = chunk * per, n_hi = n_lo + per < N ? n_lo + per : N;
    const int run = cg * T;
    const int step_i = (int)blockDim.x / run, step_r = (int)blockDim.x % run;
    int i = n_lo + (int)threadIdx.x / run, r = (int)threadIdx.x % run;
    const float* xg = x + (long)g * cg * T;
    const float* mul_g = mul ? mul + (long)g * cg * T : nullptr;
    const long x_row = x_stride * T, m_row = mul_stride * T;
    double s = 0.0, ss = 0.0;
    // four trips' loads are requested before the first is used (a trip alone waits out the memory latency); a trip
    // past the end re-reads the chunk's last node and counts as zero
    constexpr int kAhead = 4;
    while (i < n_hi) {
        float v[kAhead], m[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const bool live = i < n_hi;
            const long row = (long)b * N + (live ? i : n_hi - 1);
            v[u] = xg[row * x_row + r];
            m[u] = mul_g ? mul_g[row * m_row + r] : 1.0f;
            if (!live) m[u] = 0.f;
            i += step_i;
            r += step_r;
            if (r >= run) { r -= run; i++; }
        }
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const float w = v[u] * m[u];
            s += w;
            ss += (double)w * w;
        }
    }
    const double ts = block_sum(s, lds);
    const double tss = block_sum(ss, lds);
    if (threadIdx.x == 0) {
        partial[((long)bg * kChunks + chunk) * 2] = ts;
        partial[((long)bg * kChunks + chunk) * 2 + 1] = tss;
    }
}

// The kChunks partials of a (box, group), folded in a fixed order by a wave: in every lane .x the mean that is subtracted (0 for the
// tensor norm), .y the denominator sqrt(eps + variance or mean square), both as the apply kernels take them
__device__ __forceinline__ float2 fold_group(const double* __restrict__ partial, long bg, double count, int mode, float eps) {
    static_assert(kChunks == kWave, "a lane to a partial sum");
    const double* p = partial + (bg * kChunks + (threadIdx.x & (kWave - 1))) * 2;
    double s = p[0], ss = p[1];
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        s += __shfl_xor(s, d);
        ss += __shfl_xor(ss, d);
    }
    if (mode == 0) return make_float2(0.f, sqrtf(eps + (float)(ss / count)));   // mean over nodes, group channels of sum_comp v^2
    const double mean = s / count;
    double var = ss / count - mean * mean;
    var = var > 0.0 ? var : 0.0;
    return make_float2((float)mean, sqrtf(eps + (float)var));
}

template <bool COMP_MAJOR>
__device__ __forceinline__ float lrv_at(const float* __restrict__ row, int n, int j, int x) {
    return COMP_MAJOR ? row[x * 3 * n + j] : row[j * 3 + x];
}

// PaiNN Update, vector output: v = lin_v(x_v) * y[0:n]; out = res_v + v / sqrt(1 + |v|^2), out (rows, n, 3).  LAYOUT: of lrv, as
// lrv_comp_major of mg_painn_update_vec
struct UpdateVec {
    const float *lrv, *y, *res_v;
    float* out_v;
};
template <int LAYOUT>
__device__ __forceinline__ void update_vec(const UpdateVec& a, long r, int n, int c) {
    const float s = a.y[r * 3 * n + c];
    auto v_at = [&](int x) { return LAYOUT == 2 ? a.lrv[(r * 3 + x) * n + c] : lrv_at<LAYOUT == 1>(a.lrv + r * 9 * n, n, 2 * n + c, x); };
    const float v0 = v_at(0) * s, v1 = v_at(1) * s, v2 = v_at(2) * s;
    const float inv = 1.0f / sqrtf(1.0f + (v0 * v0 + v1 * v1 + v2 * v2));
    float o0 = v0 * inv, o1 = v1 * inv, o2 = v2 * inv;
    const long t = 3 * (r * n + c);
    if (a.res_v) { o0 += a.res_v[t]; o1 += a.res_v[t + 1]; o2 += a.res_v[t + 2]; }
    a.out_v[t] = o0; a.out_v[t + 1] = o1; a.out_v[t + 2] = o2;
}

// (y + first) + second, each rounded: neither is contracted into the product that y is, nor are they added to each other first
__device__ __forceinline__ float added(float y, float first, float second) {
#pragma clang fp contract(off)
    y += first;
    return y + second;
}

// mode 0 (TensGroupNorm): y = gamma[c] * v / sqrt(eps + mean(sum_comp v^2))
// mode 1 (ScalGroupNorm, T = 1): y = beta[c] + gamma[c] * (v - mean) / sqrt(eps + var)
// then y += add (optional, add_stride) and y += res (optional, same layout as out).
// A thread keeps one (channel, component) position k = c*T + comp of the rows of box blockIdx.z and walks over
// nodes: channel, group, gamma, beta and the group's statistics are fixed per thread, consecutive threads touch
// consecutive floats.  A workgroup folds the partial sums of the groups that its positions belong to by itself (a launch for it took
// 3 us on one system and 5 on 32 of them; each node array had one).
// VEC: the vector output of a PaiNN Update, whose rows have as many channels, beside it (layout VEC - 1): 16 336 nodes of
// 128 channels 22.5 us, 26.0 in two launches, 337 nodes 9.7, 9.6 and a launch.
template <int VEC>
__device__ __forceinline__ void group_apply(const float* __restrict__ x, long x_stride, const float* __restrict__ mul, long mul_stride,
                                            const double* __restrict__ partial, int N, int chan, int groups, int T, int mode, float eps,
                                            const float* __restrict__ gamma, const float* __restrict__ beta,
                                            const float* __restrict__ add, long add_stride, const float* __restrict__ res,
                                            float* __restrict__ out, const UpdateVec& vec, int k_block) {
    __shared__ float2 stats[256];                                  // (a position a thread: no more groups than that)
    const int CT = chan * T, b = blockIdx.z, per = chan / groups * T;
    const int k_first = k_block * blockDim.x, k = k_first + (int)threadIdx.x;
    const int k_last = k_first + (int)blockDim.x < CT ? k_first + (int)blockDim.x - 1 : CT - 1, g_first = k_first / per;
    const bool live = k < CT;
    const long x_row = x_stride * T, m_row = mul_stride * T, a_row = add_stride * T;
    constexpr int kAhead = 4;                                      // nodes at a time; the first ones are on their way during the fold
    float v[kAhead], first[kAhead], second[kAhead];                // value, what is added
    auto fetch = [&](int i) {
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const int node = i + u * (int)gridDim.y;
            const long row = (long)b * N + (node < N ? node : N - 1);
            v[u] = live ? x[row * x_row + k] : 0.f;
            if (mul && live) v[u] *= mul[row * m_row + k];
            first[u] = add && live ? add[row * a_row + k] : 0.f;
            second[u] = res && live ? res[row * CT + k] : 0.f;
        }
    };
    fetch(blockIdx.y);
    for (int g = g_first + (int)(threadIdx.x / kWave); g <= k_last / per; g += (int)(blockDim.x / kWave)) {
        const float2 f = fold_group(partial, (long)b * groups + g, (double)N * (chan / groups), mode, eps);
        if ((threadIdx.x & (kWave - 1)) == 0) stats[g - g_first] = f;
    }
    __syncthreads();
    if (!live) return;
    const int c = k / T;
    const float mean = stats[k / per - g_first].x, denom = stats[k / per - g_first].y;
    const float ga = gamma[c], be = mode == 0 ? 0.f : beta[c];
    for (int i = blockIdx.y; i < N; i += kAhead * (int)gridDim.y) {
        if (i != (int)blockIdx.y) fetch(i);
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            const int node = i + u * (int)gridDim.y;
            const float y = mode == 0 ? ga * (v[u] / denom) : be + ga * ((v[u] - mean) / denom);
            if (node < N) out[((long)b * N + node) * CT + k] = added(y, first[u], second[u]);
            if constexpr (VEC != 0)
                if (node < N) update_vec<VEC - 1>(vec, (long)b * N + node, CT, k);
        }
    }
}
template <int VEC = 0>
__global__ void __launch_bounds__(256) group_apply_kernel(const float* __restrict__ x, long x_stride,
                                                          const float* __restrict__ mul, long mul_stride,
                                                          const double* __restrict__ partial, int N, int chan,
                                                          int groups, int T, int mode, float eps,
                                                          const float* __restrict__ gamma, const float* __restrict__ beta,
                                                          const float* __restrict__ add, long add_stride,
                                                          const float* __restrict__ res, float* __restrict__ out,
                                                          const UpdateVec vec) {
    group_apply<VEC>(x, x_stride, mul, mul_stride, partial, N, chan, groups, T, mode, eps, gamma, beta, add, add_stride, res, out, vec, blockIdx.x);
}

// Several tensor norms of the same nodes (those of the three ranks) in the two launches of one.
struct NormJob {
    const float *x, *gamma, *res;
    float* out;
    double* partial;
    int chan, groups, T, first_block;                              // of the apply kernel's grid
    float eps;
};
struct NormJobs {
    NormJob job[MG_TENS_NORMS];
    int count;
};
// Sums of squares over a chunk's nodes (x), a box (y) and a job (z), for all groups at once: a thread keeps one position k = c T + t of
// the rows (and a workgroup takes several rows at a time where they are shorter than it), whole rows are read, and the positions of a
// group are added at the end (group_stats_kernel has a workgroup for every group as well, each with two reductions of its own).  The norms of
// 256, 64 x 3 and 16 x 9 floats a node with a residual, in this pair of launches and one after the other: 32 boxes of 2048 nodes 119 and
// 207 us, of 150 nodes 29 and 95, one box of 2048 15 and 51 with the host calls.  Bound by reading x twice and what is added once.
__global__ void __launch_bounds__(256) tens_stats_kernel(const NormJobs jobs, int N) {
    __shared__ double sums[256];
    const NormJob& j = jobs.job[blockIdx.z];
    const int chunk = blockIdx.x, b = blockIdx.y, CT = j.chan * j.T, per = j.chan / j.groups * j.T;
    const int nodes = (N + kChunks - 1) / kChunks, n_lo = chunk * nodes, n_hi = n_lo + nodes < N ? n_lo + nodes : N;
    const int across = CT < 256 ? CT : 256, down = 256 / across;   // positions of a row, rows at a time
    const int sub = threadIdx.x / across, lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    double* const partial = j.partial + (long)b * j.groups * kChunks * 2;
    for (int k0 = 0; k0 < CT; k0 += 256) {
        const int k = k0 + (int)threadIdx.x - sub * across;
        const bool live = sub < down && k < CT;
        const float* at = j.x + (long)b * N * CT + (live ? k : 0);
        double ss = 0.0;
        constexpr int kAhead = 8;
        for (int i = n_lo + sub; i < n_hi; i += kAhead * down) {
            float v[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const int node = i + u * down;
                v[u] = at[(long)(node < n_hi ? node : n_hi - 1) * CT];
                if (node >= n_hi) v[u] = 0.f;
            }
#pragma unroll
            for (int u = 0; u < kAhead; u++) ss += (double)v[u] * v[u];
        }
        __syncthreads();                                           // (the block of positions before this one has been added)
        sums[threadIdx.x] = live ? ss : 0.0;
        __syncthreads();
        const int k_end = k0 + across < CT ? k0 + across : CT;
        // a wave to a group, the same one in every block: its positions in this block, all rows of a trip
        for (int g = k0 / per + ((wave - k0 / per) & 3); g * per < k_end; g += 4) {
            const int lo = g * per > k0 ? g * per : k0, hi = (g + 1) * per < k_end ? (g + 1) * per : k_end;
            double t = 0.0;
            for (int q = lo + lane; q < hi; q += kWave)
                for (int r = 0; r < down; r++) t += sums[r * across + q - k0];
#pragma unroll
            for (int d = kWave / 2; d > 0; d >>= 1) t += __shfl_xor(t, d);
            if (lane == 0) {
                double* to = partial + ((long)g * kChunks + chunk) * 2;
                to[1] = lo == g * per ? t : to[1] + t;             // (a group that began in the block before: this lane wrote it there)
                to[0] = 0.0;
            }
        }
    }
}
__global__ void __launch_bounds__(256) tens_apply_kernel(const NormJobs jobs, int N) {
    int which = 0;
    while (which + 1 < jobs.count && (int)blockIdx.x >= jobs.job[which + 1].first_block) which++;     // (uniform)
    const NormJob& j = jobs.job[which];
    group_apply<0>(j.x, j.chan, nullptr, 0, j.partial, N, j.chan, j.groups, j.T, 0, j.eps, j.gamma, nullptr, nullptr, 0, j.res, j.out,
                   UpdateVec{}, (int)blockIdx.x - j.first_block);
}

// Gradient of the tensor norm y = gamma x / s, s = sqrt(eps + mean x^2) over a (box, group):
//     dgamma[c] = sum dy x / s,   dx = gamma dy / s - x D / (s^3 count),   D = sum over the group of gamma dy x.
// One pass sums dy x per channel position over chunks of a box's nodes, a second folds them group by group, a third forms dx:
// 8192 nodes of 256 channels 21 us where a dozen of torch's passes took 130.  Both sums in fp64.
// Chunks of a box: of four nodes, the loads that a thread has on its way at once, or as many as make 64 of them.  (64 for boxes of any
// size asked for 545 MB beside 84 MB of x for 4096 boxes of 20 nodes and 256 channels; so 42.)
int grad_chunks(int N) { return N < 4 * kChunks ? (int)ceil_div(N, 4) : kChunks; }
// sums: [b][k][chunk]
__global__ void __launch_bounds__(256) tensor_norm_grad_sums_kernel(const float* __restrict__ dy, const float* __restrict__ x, int N,
                                                                    int CT, double* __restrict__ sums) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.z, chunk = blockIdx.y, chunks = gridDim.y;
    if (k >= CT) return;
    const int per = (N + chunks - 1) / chunks, lo = chunk * per, hi = lo + per < N ? lo + per : N;
    const long at = (long)b * N * CT + k;
    double sum = 0.0;
    int i = lo;
    for (; i + 4 <= hi; i += 4) {                                  // (eight loads on their way)
        float g[4], v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            g[u] = dy[at + (long)(i + u) * CT];
            v[u] = x[at + (long)(i + u) * CT];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) sum += (double)g[u] * v[u];
    }
    for (; i < hi; i++) sum += (double)dy[at + (long)i * CT] * x[at + (long)i * CT];
    sums[((long)b * CT + k) * chunks + chunk] = sum;
}

// A workgroup to a (group, box).  coef[b groups + g] = (1 / s, D / (s^3 count)); of_box[b chan + c] = sum over the box of dy x / s
__global__ void __launch_bounds__(256) tensor_norm_grad_fold_kernel(const double* __restrict__ sums, int chunks, const double* __restrict__ partial,
                                                                    const float* __restrict__ gamma, int N, int chan, int groups, int T,
                                                                    float eps, float2* __restrict__ coef, double* __restrict__ of_box) {
    __shared__ double of_wave[4];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int g = blockIdx.x, b = blockIdx.y, cg = chan / groups;
    const double count = (double)N * cg, s = (double)fold_group(partial, (long)b * groups + g, count, 0, eps).y;
    double d = 0.0;
    for (int c = g * cg + wave; c < (g + 1) * cg; c += 4) {
        double q = 0.0;
        for (int t = 0; t < T; t++) q += lane < chunks ? sums[((long)b * chan * T + (long)c * T + t) * chunks + lane] : 0.0;
#pragma unroll
        for (int e = kWave / 2; e > 0; e >>= 1) q += __shfl_xor(q, e);
        d += (double)gamma[c] * q;
        if (lane == 0) of_box[(long)b * chan + c] = q / s;
    }
    if (lane == 0) of_wave[wave] = d;
    __syncthreads();
    if (threadIdx.x == 0)
        coef[b * groups + g] = make_float2((float)(1.0 / s), (float)((of_wave[0] + of_wave[1] + of_wave[2] + of_wave[3]) / (s * s * s * count)));
}

// (the first workgroups also add up dgamma over the boxes)
__global__ void __launch_bounds__(256) tensor_norm_grad_apply_kernel(const float* __restrict__ dy, const float* __restrict__ x, int batch,
                                                                     int N, int chan, int groups, int T, const float* __restrict__ gamma,
                                                                     const float2* __restrict__ coef, const double* __restrict__ of_box,
                                                                     float* __restrict__ dx, float* __restrict__ dgamma) {
    const int CT = chan * T, k = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.z;
    if (k >= CT) return;
    const float2 f = coef[b * groups + k / T / (chan / groups)];
    const float scale = gamma[k / T] * f.x;
    for (int i = blockIdx.y; i < N; i += gridDim.y) {
        const long at = ((long)b * N + i) * CT + k;
        dx[at] = scale * dy[at] - f.y * x[at];
    }
    if (blockIdx.y == 0 && b == 0 && k % T == 0) {
        double sum = 0.0;
        for (int j = 0; j < batch; j++) sum += of_box[(long)j * chan + k / T];
        dgamma[k / T] = (float)sum;
    }
}

// x / sqrt(1 + sum_comp x^2) per (row, chan)
__global__ void __launch_bounds__(256) tens_sigmoid_kernel(const float* __restrict__ x, long n, int T,
                                                           float* __restrict__ out) {
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        float v[9], q = 0.f;
        for (int t = 0; t < T; t++) { v[t] = x[e * T + t]; q += v[t] * v[t]; }
        const float inv = 1.0f / sqrtf(1.0f + q);
        for (int t = 0; t < T; t++) out[e * T + t] = v[t] * inv;
    }
}

// PaiNN Update, first elementwise stage: lrv = [lin_l | lin_r | lin_v](x_v), stored (rows, 3n, 3) or, COMP_MAJOR,
// (rows, 3, 3n) (what the GEMM stores at full rate, and what a wave reads here with unit stride)
//   ip[r,c] = sum_x l[c,x] r[c,x];  cat[r] = [x_a[r] | |r[c]|]   (rows, 2n)
// One workgroup row per node row: blockIdx.x = r, the channel from blockIdx.y and the thread.
// cat_rowmax (rows; or null): max |cat[r, :]|, the row bound of the MLP that reads cat; written when one workgroup
// covers a row (n <= 256: gridDim.y == 1)
template <bool COMP_MAJOR>
__global__ void __launch_bounds__(256) painn_update_pre_kernel(const float* __restrict__ lrv, const float* __restrict__ x_a,
                                                               int n, float* __restrict__ ip, float* __restrict__ cat,
                                                               float* __restrict__ cat_rowmax) {
    __shared__ float wave_max[4];
    const long r = blockIdx.x;
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    float mx = 0.f;
    if (c < n) {
        const float* row = lrv + r * 9 * n;
        float l[3], rr[3];
#pragma unroll
        for (int x = 0; x < 3; x++) { l[x] = lrv_at<COMP_MAJOR>(row, n, c, x); rr[x] = lrv_at<COMP_MAJOR>(row, n, n + c, x); }
        ip[r * n + c] = l[0] * rr[0] + l[1] * rr[1] + l[2] * rr[2];
        const float a = x_a[r * n + c], nr = sqrtf(rr[0] * rr[0] + rr[1] * rr[1] + rr[2] * rr[2]);
        cat[r * 2 * n + c] = a;
        cat[r * 2 * n + n + c] = nr;
        mx = fmaxf(fabsf(a), nr);
    }
    if (cat_rowmax) {                                         // uniform over the workgroup
        for (int d = 1; d < kWave; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
        if ((threadIdx.x & (kWave - 1)) == 0) wave_max[threadIdx.x / kWave] = mx;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < (int)(blockDim.x / kWave); w++) mx = fmaxf(mx, wave_max[w]);
            cat_rowmax[r] = mx;
        }
    }
}

template <int LAYOUT>
__global__ void __launch_bounds__(256) painn_update_vec_kernel(const UpdateVec a, int n) {
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c < n) update_vec<LAYOUT>(a, blockIdx.x, n, c);
}

// kinds: 1 sq_radial_encode of normed_sq_dist (archs/diffuser_atoms14.py:32-48)
//        2 radial_encode_edge (archs/diffuser_atoms5.py:25-30)
__global__ void __launch_bounds__(256) radial_encode_kernel(int kind, const float* __restrict__ r_ij, long E, int n,
                                                            float rmax, float c0, float c1, float* __restrict__ out) {
    const long total = E * n;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const long e = t / n;
        const int m = (int)(t - e * n);
        const float x = r_ij[3 * e], y = r_ij[3 * e + 1], z = r_ij[3 * e + 2];
        const float sq = x * x + y * y + z * z;
        if (kind == 1) {
            const float q = sq / (rmax * rmax);
            const float h = sqrtf(1.0f + q);
            const float coeff = c0 * expf(c1 * (float)m);        // (pi / sqrt 2) exp(n^-0.7 m)
            out[t] = sinf(coeff * h) * (0.70710678118654752f - h);
        } else {
            const float q = sq / rmax;                             // divided by rmax, not rmax^2, as in the reference
            const float cut = fmaxf(1.0f - q, 0.0f);
            out[t] = cosf((c0 * (float)m) * sqrtf(q)) * cut;      // c0 = pi
        }
    }
}

long grid_for(long total) {
    long b = ceil_div(total, 256);
    return b > 256L * 32 ? 256L * 32 : (b < 1 ? 1 : b);
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_group_norm_scratch_bytes(int batch, int groups, size_t* bytes) {
    MG_REQUIRE(bytes && batch >= 0 && groups >= 0, "mg_group_norm_scratch_bytes: bad argument");
    *bytes = (size_t)batch * groups * kChunks * 2 * sizeof(double);
    return MG_OK;
}

// Positions across, nodes of a box down: four nodes a thread, which it has on their way at once, and more where that is beyond 4096
// workgroups, each of which folds by itself (2048 nodes of 256 channels 6.3 us, 8.4 at one node a thread, 7.4 in two launches; 65 536
// 45 us in 4096 workgroups, 49 in 8192, 63 in 1024, 49 in two launches of 8192; 16 336 12.5, 15.5 in two)
static dim3 apply_grid(int batch, int nodes, int CT, int* threads) {
    *threads = CT >= 256 ? 256 : (int)ceil_div(CT, kWave) * kWave;
    const long kx = ceil_div(CT, *threads), most = ceil_div(4096L, kx * batch);
    long ny = ceil_div(nodes, 4);
    ny = ny > most ? most : ny;
    return dim3((unsigned)kx, (unsigned)ny, (unsigned)batch);
}

// vec: 0, or 1 + the layout of `with`, the vector output written beside it
static int group_norm(int mode, const float* x, long x_stride, const float* mul, long mul_stride, int batch, int nodes, int chan, int groups,
                      int comps, float eps, const float* gamma, const float* beta, const float* add, long add_stride, const float* res,
                      void* scratch, float* out, int vec, const UpdateVec& with, mg_stream_t stream) {
    MG_REQUIRE(mode == 0 || mode == 1, "mg_group_norm: mode must be 0 (tensor) or 1 (scalar)");
    MG_REQUIRE(batch >= 0 && nodes >= 0 && chan >= 0 && groups > 0 && chan % groups == 0, "mg_group_norm: bad sizes");
    MG_REQUIRE(comps == 1 || comps == 3 || comps == 9, "mg_group_norm: comps must be 1, 3 or 9");
    MG_REQUIRE(mode == 0 || comps == 1, "mg_group_norm: the scalar norm takes comps == 1");
    const long total = (long)batch * nodes * chan * comps;
    if (total == 0) return MG_OK;
    MG_REQUIRE(x && gamma && out && scratch && (mode == 0 || beta), "mg_group_norm: null pointer");
    MG_REQUIRE(batch <= 65535 && (long)chan * comps <= 0x7fffffffL, "mg_group_norm: more than 65535 boxes");
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(group_stats_kernel, dim3((unsigned)(batch * groups), kChunks), dim3(256), 0, st, x, x_stride, mul,
                       mul_stride, nodes, chan, groups, comps, static_cast<double*>(scratch));
    int threads;
    const dim3 grid = apply_grid(batch, nodes, chan * comps, &threads);
    const auto kernel = vec == 0 ? group_apply_kernel<0> : vec == 1 ? group_apply_kernel<1> : vec == 2 ? group_apply_kernel<2> : group_apply_kernel<3>;
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, st, x, x_stride, mul, mul_stride, static_cast<const double*>(scratch), nodes, chan,
                       groups, comps, mode, eps, gamma, beta, add, add_stride, res, out, with);
    return check_launch("mg_group_norm");
}

int mg_group_norm(int mode, const float* x, long x_stride, const float* mul, long mul_stride, int batch, int nodes,
                  int chan, int groups, int comps, float eps, const float* gamma, const float* beta, const float* add,
                  long add_stride, const float* res, void* scratch, float* out, mg_stream_t stream) {
    return group_norm(mode, x, x_stride, mul, mul_stride, batch, nodes, chan, groups, comps, eps, gamma, beta, add, add_stride, res, scratch,
                      out, 0, UpdateVec{}, stream);
}

int mg_painn_update_post(const float* lrv, int lrv_comp_major, const float* ip, const float* y, int batch, int nodes, int n, int groups,
                         float eps, const float* gamma, const float* beta, const float* res_a, const float* res_v, void* scratch,
                         float* out_a, float* out_v, mg_stream_t stream) {
    MG_REQUIRE(lrv_comp_major >= 0 && lrv_comp_major <= 2, "mg_painn_update_post: lrv_comp_major must be 0, 1 or 2");
    MG_REQUIRE((long)batch * nodes * n == 0 || (lrv && y && ip && out_v), "mg_painn_update_post: null pointer");
    return group_norm(1, ip, n, y + n, 3L * n, batch, nodes, n, groups, 1, eps, gamma, beta, y + 2 * n, 3L * n, res_a, scratch, out_a,
                      1 + lrv_comp_major, UpdateVec{lrv, y, res_v, out_v}, stream);
}

int mg_tens_group_norms(const mg_tens_norm* norms, int count, int batch, int nodes, void* scratch, mg_stream_t stream) {
    MG_REQUIRE(count >= 0 && count <= MG_TENS_NORMS && (norms || count == 0), "mg_tens_group_norms: at most %d norms", MG_TENS_NORMS);
    MG_REQUIRE(batch >= 0 && nodes >= 0 && batch <= 65535, "mg_tens_group_norms: bad sizes, or more than 65535 boxes");
    NormJobs jobs{};
    double* partial = static_cast<double*>(scratch);
    long blocks = 0;
    for (int k = 0; k < count; k++) {
        const mg_tens_norm& n = norms[k];
        MG_REQUIRE(n.chan >= 0 && n.groups > 0 && n.chan % n.groups == 0, "mg_tens_group_norms: bad sizes");
        MG_REQUIRE(n.comps == 1 || n.comps == 3 || n.comps == 9, "mg_tens_group_norms: comps must be 1, 3 or 9");
        MG_REQUIRE((long)n.chan * n.comps <= 65536, "mg_tens_group_norms: rows of more than 65536 floats");
        if ((long)batch * nodes * n.chan == 0) continue;
        MG_REQUIRE(n.x && n.gamma && n.out && scratch, "mg_tens_group_norms: null pointer");
        jobs.job[jobs.count++] = NormJob{n.x, n.gamma, n.res, n.out, partial, n.chan, n.groups, n.comps, (int)blocks, n.eps};
        partial += (size_t)batch * n.groups * kChunks * 2;
        blocks += ceil_div((long)n.chan * n.comps, 256);
    }
    if (jobs.count == 0) return MG_OK;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(tens_stats_kernel, dim3(kChunks, (unsigned)batch, (unsigned)jobs.count), dim3(256), 0, st, jobs, nodes);
    // (as apply_grid)
    const long most = ceil_div(4096L * jobs.count, blocks * batch), strips = ceil_div(nodes, 4);
    hipLaunchKernelGGL(tens_apply_kernel, dim3((unsigned)blocks, (unsigned)(strips < most ? strips : most), (unsigned)batch), dim3(256), 0, st,
                       jobs, nodes);
    return check_launch("mg_tens_group_norms");
}

int mg_tensor_norm_grad_workspace_bytes_of(int batch, int nodes, int chan, int groups, int comps, size_t* bytes) {
    MG_REQUIRE(bytes && batch >= 0 && nodes >= 0 && chan >= 0 && groups >= 0 && comps >= 0, "mg_tensor_norm_grad_workspace_bytes: bad argument");
    *bytes = (size_t)batch * chan * ((size_t)comps * grad_chunks(nodes) + 1) * sizeof(double) + (size_t)batch * groups * sizeof(float2);
    return MG_OK;
}

int mg_tensor_norm_grad_workspace_bytes(int batch, int chan, int groups, int comps, size_t* bytes) {
    return mg_tensor_norm_grad_workspace_bytes_of(batch, 4 * kChunks, chan, groups, comps, bytes);
}

int mg_tensor_norm_grad(const float* dy, const float* x, int batch, int nodes, int chan, int groups, int comps, float eps,
                        const float* gamma, const void* scratch, void* workspace, float* dx, float* dgamma, mg_stream_t stream) {
    MG_REQUIRE(batch >= 0 && nodes >= 0 && chan >= 0 && groups > 0 && chan % groups == 0, "mg_tensor_norm_grad: bad sizes");
    MG_REQUIRE(comps == 1 || comps == 3 || comps == 9, "mg_tensor_norm_grad: comps must be 1, 3 or 9");
    MG_REQUIRE(batch > 0 && nodes > 0 && chan > 0, "mg_tensor_norm_grad: nothing to differentiate");
    MG_REQUIRE(dy && x && gamma && scratch && workspace && dx && dgamma, "mg_tensor_norm_grad: null pointer");
    MG_REQUIRE(batch <= 65535 && (long)chan * comps <= 0x7fffffffL, "mg_tensor_norm_grad: more than 65535 boxes");
    hipStream_t st = (hipStream_t)stream;
    const int CT = chan * comps, chunks = grad_chunks(nodes);
    double *sums = static_cast<double*>(workspace), *of_box = sums + (long)batch * CT * chunks;
    float2* coef = reinterpret_cast<float2*>(of_box + (long)batch * chan);
    int threads;
    const dim3 grid = apply_grid(batch, nodes, CT, &threads);
    hipLaunchKernelGGL(tensor_norm_grad_sums_kernel, dim3(grid.x, (unsigned)chunks, grid.z), dim3(threads), 0, st, dy, x, nodes, CT, sums);
    hipLaunchKernelGGL(tensor_norm_grad_fold_kernel, dim3((unsigned)groups, (unsigned)batch), dim3(256), 0, st, sums, chunks,
                       static_cast<const double*>(scratch), gamma, nodes, chan, groups, comps, eps, coef, of_box);
    hipLaunchKernelGGL(tensor_norm_grad_apply_kernel, grid, dim3(threads), 0, st, dy, x, batch, nodes, chan, groups, comps, gamma, coef, of_box,
                       dx, dgamma);
    return check_launch("mg_tensor_norm_grad");
}

int mg_tens_sigmoid(int inds, const float* x, long rows_times_chan, float* out, mg_stream_t stream) {
    MG_REQUIRE(inds >= 0 && inds <= 2 && rows_times_chan >= 0, "mg_tens_sigmoid: bad argument");
    if (rows_times_chan == 0) return MG_OK;
    MG_REQUIRE(x && out, "mg_tens_sigmoid: null pointer");
    const int T = inds == 0 ? 1 : (inds == 1 ? 3 : 9);
    hipLaunchKernelGGL(tens_sigmoid_kernel, dim3((unsigned)grid_for(rows_times_chan)), dim3(256), 0,
                       (hipStream_t)stream, x, rows_times_chan, T, out);
    return check_launch("mg_tens_sigmoid");
}

int mg_painn_update_pre(const float* lrv, int lrv_comp_major, const float* x_a, long rows, int n, float* ip, float* cat,
                        float* cat_rowmax, mg_stream_t stream) {
    MG_REQUIRE(cat_rowmax == nullptr || n <= 256, "mg_painn_update_pre: row maxima are emitted for n <= 256");
    MG_REQUIRE(rows >= 0 && n >= 0, "mg_painn_update_pre: negative size");
    if (rows * n == 0) return MG_OK;
    MG_REQUIRE(lrv && x_a && ip && cat, "mg_painn_update_pre: null pointer");
    MG_REQUIRE(rows <= 0x7fffffffL, "mg_painn_update_pre: more than 2^31 - 1 rows");
    const int threads = n >= 256 ? 256 : (int)ceil_div(n, kWave) * kWave;
    const dim3 grid((unsigned)rows, (unsigned)ceil_div(n, threads));
    if (lrv_comp_major)
        hipLaunchKernelGGL(painn_update_pre_kernel<true>, grid, dim3(threads), 0, (hipStream_t)stream, lrv, x_a, n, ip, cat,
                           cat_rowmax);
    else
        hipLaunchKernelGGL(painn_update_pre_kernel<false>, grid, dim3(threads), 0, (hipStream_t)stream, lrv, x_a, n, ip, cat,
                           cat_rowmax);
    return check_launch("mg_painn_update_pre");
}

int mg_painn_update_vec(const float* lrv, int lrv_comp_major, const float* y, const float* res_v, long rows, int n,
                        float* out_v, mg_stream_t stream) {
    MG_REQUIRE(rows >= 0 && n >= 0, "mg_painn_update_vec: negative size");
    if (rows * n == 0) return MG_OK;
    MG_REQUIRE(lrv && y && out_v, "mg_painn_update_vec: null pointer");
    MG_REQUIRE(rows <= 0x7fffffffL, "mg_painn_update_vec: more than 2^31 - 1 rows");
    const int threads = n >= 256 ? 256 : (int)ceil_div(n, kWave) * kWave;
    const dim3 grid((unsigned)rows, (unsigned)ceil_div(n, threads));
    const auto kernel = lrv_comp_major == 2 ? painn_update_vec_kernel<2> : (lrv_comp_major ? painn_update_vec_kernel<1> : painn_update_vec_kernel<0>);
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, (hipStream_t)stream, UpdateVec{lrv, y, res_v, out_v}, n);
    return check_launch("mg_painn_update_vec");
}

int mg_radial_encode(int kind, const float* r_ij, long n_edges, int n, float rmax, float* out, mg_stream_t stream) {
    MG_REQUIRE(kind == 1 || kind == 2, "mg_radial_encode: kind must be 1 (sq_radial_encode) or 2 (radial_encode_edge)");
    MG_REQUIRE(n_edges >= 0 && n >= 0 && rmax > 0.f, "mg_radial_encode: bad argument");
    if (n_edges * n == 0) return MG_OK;
    MG_REQUIRE(r_ij && out, "mg_radial_encode: null pointer");
    float c0, c1 = 0.f;
    if (kind == 1) {
        c0 = (float)(3.14159265358979323846 * 0.70710678118654752440);
        c1 = (float)pow((double)n, -0.7);
    } else {
        c0 = (float)3.14159265358979323846;
    }
    hipLaunchKernelGGL(radial_encode_kernel, dim3((unsigned)grid_for(n_edges * n)), dim3(256), 0, (hipStream_t)stream,
                       kind, r_ij, n_edges, n, rmax, c0, c1, out);
    return check_launch("mg_radial_encode");
}

}  // extern "C"
