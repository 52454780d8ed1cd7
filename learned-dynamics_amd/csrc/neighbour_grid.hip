// Periodic cell-list radius graph for gfx950.
//
// Pipeline (all on the caller's stream, no allocation, no host sync):
//   bin      wrap each atom into the box, cell id
//   sort     up to 16 workgroups per box, each sorting a slab of the box's cells:
//            counting sort by cell in LDS (histogram, scan, placement, rank by
//            atom id inside the cell, so that the cell-ordered array, and with it
//            every output row, is deterministic) -> cell_start.
//            Boxes of more than 16384 atoms or 4096 cells take four kernels instead
//            (histogram with global atomics, scan, place, order)
//   count    one workgroup per home cell: the 27 window cells are staged in LDS
//            once, each wave takes home atoms and sweeps the staged candidates
//            64 at a time, counting hits with ballot/popcount -> degree; the hits
//            themselves go, in window order, into the atom's row of a scratch
//            array (hit rows of a fixed capacity)
//            (boxes of at most 2048 atoms and 4096 cells: bin, sort and count are one kernel, box_search_kernel)
//   scan     degrees -> CSR row_ptr (+ per-box edge counts, statistics)
//   fill     copies the hit rows to row_ptr[i] (exact-size rows, no atomics per
//            edge, no geometry); a row with more hits than a hit row holds is
//            swept again by one wave.  graph_fill_kernel (mg_graph_fill; graph_fill_dealt_kernel for short
//            rows) is scan and fill in one, and writes int64 indices, edge vectors and the cell order as well
//
// fp32 recipe (this file is compiled with -ffp-contract=off):
//   w    = remainderf(x - box/2, box) + box/2                 (IEEE remainder)
//   cell = (int)(((float)ndiv * w) / box) % ndiv              (correctly rounded divide)
//   d    = remainder(w_i - w_j, box) per axis, evaluated as fma(-rint(t / box), box, t)
//          (|w_i - w_j| <= box, so the multiple is -1, 0 or 1 and the result is exact;
//          see count_kernel for why quotients within rounding of 1/2 do not matter)
//   d2   = fma(dz,dz, fma(dy,dy, dx*dx)) <= cutoff*cutoff, i != j
//   only the periodic 3x3x3 cell window is searched, with ndiv = ceil(box/cutoff):
//   when box/cutoff is not an integer the cells are narrower than the cutoff and
//   pairs two cells apart are not listed.
#include "common.hpp"
#include <mutex>
#include <type_traits>

namespace mg {
namespace {

// Built-in workspace of mg_neighbour_edges_static, for callers that cannot allocate one.  One copy per GPU, held
// from the moment the library is loaded until the process ends.  Host code never passes `scratch` itself anywhere:
// the name is a host-side handle, the device address comes from hipGetSymbolAddress (scratch_of_current_device).
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {nullptr};
std::mutex g_scratch_mutex;

// Device address of this GPU's copy of `scratch`; looked up once per device, with that device current.
int scratch_of_current_device(void** out) {
    int dev = -1;
    MG_HIP(hipGetDevice(&dev));
    MG_REQUIRE(dev >= 0 && dev < kMaxDevices, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        MG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        MG_REQUIRE(p != nullptr, "hipGetSymbolAddress returned a null address for the built-in workspace");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return MG_OK;
}

constexpr int kCandCapDense = 1024;   // candidates staged in LDS per home cell (16 KB), 4-wave workgroups
constexpr int kCandCapSparse = 512;   // sparse boxes: 1-wave workgroups, 8 KB
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;       // per thread
constexpr int kScanTile = kScanThreads * kScanItems;

struct Grid {
    int nx, ny, nz, ncells;   // per box
    float bx, by, bz;
    float r0sq;
    int batch, nodes;
};

constexpr int kNanBit = 1 << 30;    // in box_max; a cell holds fewer than 2^30 atoms
constexpr int kNanCell = 1 << 31;   // in cell_of: the atom has a NaN coordinate (consumers mask it out)

struct Workspace {
    float4* wrapped;    // A: (w.x, w.y, w.z, bits of box-local index)
    float4* sorted;     // A: same records in cell order
    int* cell_of;       // A: global cell id (batch offset included)
    int* slot;          // A
    int* placed;        // A: atom ids in cell order before ranking
    int* degree;        // A
    int* cell_count;    // C
    int* cell_start;    // C + 1
    int* block_sums;    // scan scratch (cell histogram)
    int* block_max;     // scan scratch
    int* deg_sums;      // sums / maxima of the degrees per tile of kScanTile rows
    int* deg_max;
    int* box_max;       // largest cell occupancy per workgroup of the sort, bit kNanBit: the box holds a NaN coordinate
                        // (without the per-box sort: one occupancy, one flag)
    void* hits;         // A x hit_cap: neighbours found by the count pass (box-local atom ids, window order);
                        // 16-bit entries when a box has at most 65536 atoms, else 32-bit
    int hit_cap;        // entries per hit row; rows with more hits are recomputed by the fill pass
    int hit_bytes;      // 2 or 4
    size_t bytes;
};

inline size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

Workspace carve(void* base, long A, long C, int hit_cap, int hit_bytes) {
    Workspace w{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void* p = base ? static_cast<char*>(base) + off : nullptr;
        off += align_up(bytes);
        return p;
    };
    const long scan_blocks = ceil_div((A > C ? A : C) + 1, kScanTile) + 1;
    w.wrapped = static_cast<float4*>(take(sizeof(float4) * A));
    w.sorted = static_cast<float4*>(take(sizeof(float4) * A));
    w.cell_of = static_cast<int*>(take(sizeof(int) * A));
    w.slot = static_cast<int*>(take(sizeof(int) * A));
    w.placed = static_cast<int*>(take(sizeof(int) * A));
    w.degree = static_cast<int*>(take(sizeof(int) * A));
    w.cell_count = static_cast<int*>(take(sizeof(int) * C));
    w.cell_start = static_cast<int*>(take(sizeof(int) * (C + 1)));
    w.block_sums = static_cast<int*>(take(sizeof(int) * scan_blocks));
    w.block_max = static_cast<int*>(take(sizeof(int) * scan_blocks));
    w.deg_sums = static_cast<int*>(take(sizeof(int) * scan_blocks));
    w.deg_max = static_cast<int*>(take(sizeof(int) * scan_blocks));
    w.box_max = static_cast<int*>(take(sizeof(int) * (A + 2)));           // (batch <= A)
    w.hits = take((size_t)hit_bytes * A * hit_cap);
    w.hit_cap = hit_cap;
    w.hit_bytes = hit_bytes;
    w.bytes = off;
    return w;
}

int make_grid(float cutoff, float bx, float by, float bz, int batch, int nodes, Grid* g) {
    MG_REQUIRE(cutoff > 0.f && bx > 0.f && by > 0.f && bz > 0.f, "cutoff and box must be positive");
    MG_REQUIRE(batch >= 0 && nodes >= 0, "negative batch or nodes");
    int nd[3];
    mg_neighbour_ndiv(cutoff, bx, by, bz, nd);
    if (nd[0] < 3 || nd[1] < 3 || nd[2] < 3)
        return fail(MG_ERR_BOX_TOO_SMALL, "box dimension must be greater than 3*cutoff");
    const long ncells = (long)nd[0] * nd[1] * nd[2];
    MG_REQUIRE(ncells * (batch > 0 ? batch : 1) < 0x7fffffffL, "too many cells (%ld per box)", ncells);
    MG_REQUIRE((long)batch * nodes < 0x7fffffffL, "batch*nodes does not fit int32");
    MG_REQUIRE((long)nd[0] * (batch > 0 ? batch : 1) <= 65535 && nd[1] <= 65535,
               "batch * cells along x (%ld) and cells along y (%d) must not exceed 65535", (long)nd[0] * batch, nd[1]);
    g->nx = nd[0]; g->ny = nd[1]; g->nz = nd[2]; g->ncells = (int)ncells;
    g->bx = bx; g->by = by; g->bz = bz;
    g->r0sq = cutoff * cutoff;
    g->batch = batch; g->nodes = nodes;
    return MG_OK;
}

// ---------------------------------------------------------------- device math
// The IEEE remainder is exact, so t - n box in one fma is the remainder bit for bit whenever n is its multiple, and a
// multiple that is off by one or more leaves at least box / 2: only results near box / 2 (and non-finite input) need
// the library's loop.
__device__ __forceinline__ float wrap_into_box(float x, float box) {
    const float half = 0.5f * box;
    const float t = x - half;
    const float r = __fmaf_rn(-rintf(t * (1.0f / box)), box, t);
    if (fabsf(r) < 0.4999f * box) return r + half;
    return remainderf(t, box) + half;
}

// (int)(correctly rounded quotient) % ndiv.  The quotient with a reciprocal is within a few ulp of the correctly
// rounded one: where both ends of that interval truncate to the same integer, so does the quotient.
__device__ __forceinline__ int cell_coord(float w, float box, int ndiv) {
    const float scaled = (float)ndiv * w;
    const float q = scaled * (1.0f / box);
    int c = (int)(q * 0.9999995f);
    if (!(c == (int)(q * 1.0000005f) && q >= 0.f)) c = (int)__fdiv_rn(scaled, box);
    if (c >= ndiv) c %= ndiv;
    return c < 0 ? 0 : c;   // only reachable with non-finite input
}

// torch's float `%` (floor-mod, b > 0): fmod, then move a result of the wrong sign by one period
__device__ __forceinline__ float floor_mod(float a, float b) {
    float m = fmodf(a, b);
    if (m < 0.f) m += b;
    return m;
}

// boxwrap(box, x_j - x_i), a floor-mod per axis.  fmod is exact, so one fma gives it bit for bit whenever the quotient
// was truncated to the right integer, which the result's range shows; fmodf itself (a loop over the exponents'
// difference) is left for the rest, behind one branch for the three axes.
struct Box3 {
    float x, y, z, ix, iy, iz;
};
__device__ __forceinline__ bool fast_wrap(float raw, float box, float inv_box, float* r) {
    const float half = 0.5f * box, a = raw + half;
    const float m = __fmaf_rn(-truncf(a * inv_box), box, a);
    *r = (m < 0.f ? m + box : m) - half;
    return fabsf(m) < box && (a < 0.f ? m <= 0.f : m >= 0.f);
}
__device__ __forceinline__ float3 wrapped_difference(const float3& xj, const float3& xi, const Box3& box) {
    const float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
    float3 r;
    const bool fast_x = fast_wrap(dx, box.x, box.ix, &r.x), fast_y = fast_wrap(dy, box.y, box.iy, &r.y);
    const bool fast_z = fast_wrap(dz, box.z, box.iz, &r.z);
    if (!(fast_x && fast_y && fast_z)) {
        r.x = floor_mod(dx + 0.5f * box.x, box.x) - 0.5f * box.x;
        r.y = floor_mod(dy + 0.5f * box.y, box.y) - 0.5f * box.y;
        r.z = floor_mod(dz + 0.5f * box.z, box.z) - 0.5f * box.z;
    }
    return r;
}
__device__ __forceinline__ Box3 box_of(float bx, float by, float bz) {
    return Box3{bx, by, bz, 1.0f / bx, 1.0f / by, 1.0f / bz};
}
__device__ __forceinline__ float3 load3(const float* p) { return make_float3(p[0], p[1], p[2]); }

__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        int t = __shfl_up(v, d);
        if (lane >= d) v += t;
    }
    return v;
}

// ------------------------------------------------------------------- kernels
// Clearing is done by a kernel, not a memset node, so that the sequence behaves
// the same when a caller records it into a HIP graph.
__global__ void __launch_bounds__(256) zero3_kernel(int* __restrict__ a, long na, int* __restrict__ b, long nb,
                                                    int* __restrict__ c, long nc) {
    const long stride = (long)gridDim.x * blockDim.x;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (long i = t; i < na; i += stride) a[i] = 0;
    for (long i = t; i < nb; i += stride) b[i] = 0;
    for (long i = t; i < nc; i += stride) c[i] = 0;
}

// HIST: also the histogram of cell sizes and each atom's slot in its cell (boxes too large for the per-box sort)
template <bool HIST>
__global__ void __launch_bounds__(256) bin_kernel(const float* __restrict__ x, Grid g, Workspace w) {
    const long A = (long)g.batch * g.nodes;
    const long a = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= A) return;
    const int b = (int)(a / g.nodes);
    const int i = (int)(a - (long)b * g.nodes);
    const float px = x[3 * a + 0], py = x[3 * a + 1], pz = x[3 * a + 2];
    const float wx = wrap_into_box(px, g.bx), wy = wrap_into_box(py, g.by), wz = wrap_into_box(pz, g.bz);
    const int cx = cell_coord(wx, g.bx, g.nx);
    const int cy = cell_coord(wy, g.by, g.ny);
    const int cz = cell_coord(wz, g.bz, g.nz);
    const int cell = ((b * g.nx + cx) * g.ny + cy) * g.nz + cz;
    const bool nan = px != px || py != py || pz != pz;
    w.wrapped[a] = make_float4(wx, wy, wz, __int_as_float(i));
    w.cell_of[a] = cell | (nan && !HIST ? kNanCell : 0);
    if (HIST) {
        w.slot[a] = atomicAdd(&w.cell_count[cell], 1);
        if (nan) atomicOr(&w.box_max[1], kNanBit);
    }
}

// Counting sort of a box by cell, entirely in LDS: histogram (LDS atomics), scan, placement, rank by atom id inside
// the cell.  A box is shared by gridDim.x workgroups: each takes a contiguous range of the box's cells (a slab),
// reads the cell of every atom of the box, counts the atoms of the slabs before its own (its place in the
// cell-ordered array) and sorts the atoms of its own slab.  Replaces the histogram / scan / place / order kernels
// for boxes of at most kSortNodes atoms and kSortCells cells.  Writes cell_start (global positions), sorted,
// box_max[b * slabs + slab].
constexpr int kSortThreads = 1024, kSortNodes = 16384, kSortCells = 4096;   // 2^14 atoms: 14 key bits
constexpr int kSortSlabsMax = 16;
__global__ void __launch_bounds__(kSortThreads) sort_box_kernel(Grid g, Workspace w) {
    constexpr int kPer = kSortNodes / kSortThreads, kCellsPer = kSortCells / kSortThreads;
    // cell sizes, then exclusive starts (start[cells of the slab] = its atoms), then a spare bin per lane
    __shared__ int start[kSortCells + 1 + kWave];
    // keys (cell << 14 | atom) in cell order: a key of a later cell compares greater than any key of this cell, so the
    // rank loop may read past the end of its cell without a bounds check (the array ends in 8 keys of INT_MAX)
    __shared__ int placed[kSortNodes + 8 + 1];   // (+ a spare word that takes the writes for atoms of other slabs)
    __shared__ int wave_sum[kSortThreads / kWave], wave_max[kSortThreads / kWave], wave_before[kSortThreads / kWave];
    __shared__ int wave_nan[kSortThreads / kWave];
    const int slab = blockIdx.x, slabs = gridDim.x;
    const int b = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    const long base = (long)b * g.nodes;
    const int cell_base = b * g.ncells;
    const int c_lo = (int)((long)slab * g.ncells / slabs), c_hi = (int)((long)(slab + 1) * g.ncells / slabs);
    const int ncs = c_hi - c_lo;              // cells of this slab
    for (int c = tid; c <= ncs + kWave; c += kSortThreads) start[c] = 0;
    __syncthreads();
    int cl[kPer], sl[kPer];                   // cell within the slab (-1: another slab's atom), slot within the cell
    int n_before = 0, nan = 0;
    // Straight-line code, so that the 16 loads (and then the 16 LDS atomics) of a thread are in flight together:
    // an index past the box reads the box's last atom and is discarded, an atom of another slab counts into a
    // spare bin of its lane.
    const int* cells = w.cell_of + base;
    const int last = g.nodes - 1;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = tid + kSortThreads * j;
        const int c = cells[i < g.nodes ? i : last];
        nan |= c;                             // (the sign bit)
        cl[j] = i < g.nodes ? (c & ~kNanCell) - cell_base : g.ncells;
    }
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int c = cl[j];
        n_before += c < c_lo ? 1 : 0;
        const bool own = c >= c_lo && c < c_hi;
        cl[j] = own ? c - c_lo : -1;
        sl[j] = atomicAdd(&start[own ? c - c_lo : ncs + 1 + lane], 1);
    }
    for (int d = kWave / 2; d > 0; d >>= 1) n_before += __shfl_xor(n_before, d);
    if (lane == 0) wave_before[wave] = n_before;
    const int any_nan = __any(nan < 0);
    if (lane == 0) wave_nan[wave] = any_nan;
    __syncthreads();
    // exclusive scan of the cell sizes: a thread owns kCellsPer consecutive cells
    int cnt[kCellsPer], sum = 0, mx = 0;
#pragma unroll
    for (int k = 0; k < kCellsPer; k++) {
        const int c = tid * kCellsPer + k;
        cnt[k] = c < ncs ? start[c] : 0;
        sum += cnt[k];
        mx = cnt[k] > mx ? cnt[k] : mx;
    }
    const int incl = wave_incl_scan(sum, lane);
    for (int d = kWave / 2; d > 0; d >>= 1) { const int t = __shfl_xor(mx, d); mx = t > mx ? t : mx; }
    if (lane == kWave - 1) wave_sum[wave] = incl;
    if (lane == 0) wave_max[wave] = mx;
    int before = 0;                           // atoms of this box in the slabs before this one
    for (int k = 0; k < kSortThreads / kWave; k++) before += wave_before[k];
    __syncthreads();
    int run = incl - sum;
    for (int k = 0; k < wave; k++) run += wave_sum[k];
    int mine = 0;                             // atoms of this slab
    for (int k = 0; k < kSortThreads / kWave; k++) mine += wave_sum[k];
#pragma unroll
    for (int k = 0; k < kCellsPer; k++) {
        const int c = tid * kCellsPer + k;
        if (c < ncs) {
            start[c] = run;
            w.cell_start[cell_base + c_lo + c] = (int)base + before + run;
        }
        run += cnt[k];
    }
    if (tid == 0) {
        start[ncs] = mine;
        int m = 0, any = 0;
        for (int k = 0; k < kSortThreads / kWave; k++) { m = wave_max[k] > m ? wave_max[k] : m; any |= wave_nan[k]; }
        w.box_max[b * slabs + slab] = m | (any ? kNanBit : 0);
        if (b == g.batch - 1 && slab == slabs - 1) w.cell_start[(long)g.batch * g.ncells] = g.batch * g.nodes;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = tid + kSortThreads * j;
        const bool own = cl[j] >= 0;
        const int first = start[own ? cl[j] : 0];
        placed[own ? first + sl[j] : kSortNodes + 8] = (cl[j] << 14) | i;
    }
    if (tid < 8) placed[mine + tid] = 0x7fffffff;
    __syncthreads();
    // position p of the slab holds atom (key & 16383) of cell (key >> 14); its final place is its rank by atom id
    // inside the cell.  Going by position keeps every lane busy (a slab has about gridDim.x times fewer atoms than
    // the box), and the atom's record is requested before the ranking, not after it.
    for (int p = tid; p < mine; p += kSortThreads) {
        const int key = placed[p];
        const int c = key >> 14;
        const float4 rec = w.wrapped[base + (key & (kSortNodes - 1))];
        const int lo = start[c], hi = start[c + 1];
        int rank = 0;
        for (int q0 = lo; q0 < hi; q0 += 8) {          // 8 independent LDS reads per trip, one wait
            int v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = placed[q0 + u];
#pragma unroll
            for (int u = 0; u < 8; u++) rank += v[u] < key ? 1 : 0;
        }
        w.sorted[base + before + lo + rank] = rec;
    }
}

__global__ void __launch_bounds__(256) place_kernel(Grid g, Workspace w) {
    const long A = (long)g.batch * g.nodes;
    const long a = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= A) return;
    w.placed[w.cell_start[w.cell_of[a]] + w.slot[a]] = (int)a;
}

// position p holds atom a of cell c; its final place is its rank by atom id inside c
__global__ void __launch_bounds__(256) order_kernel(Grid g, Workspace w) {
    const long A = (long)g.batch * g.nodes;
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= A) return;
    const int a = w.placed[p];
    const int c = w.cell_of[a];
    const int lo = w.cell_start[c], hi = w.cell_start[c + 1];
    int rank = 0;
    for (int q = lo; q < hi; q++) rank += (w.placed[q] < a) ? 1 : 0;
    w.sorted[lo + rank] = w.wrapped[a];
}

// --- two-kernel exclusive scan of n ints: out[0..n] (out[n] = total) -------

// block-wide exclusive scan of one value per thread (256 threads); returns the
// exclusive prefix and leaves the block total in *total
__device__ __forceinline__ int block_excl_scan(int v, int* total, int* lds /* >= 8 ints */) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int incl = wave_incl_scan(v, lane);
    if (lane == kWave - 1) lds[wave] = incl;
    __syncthreads();
    int off = 0, tot = 0;
    const int nw = blockDim.x / kWave;
    for (int k = 0; k < nw; k++) {
        const int s = lds[k];
        if (k < wave) off += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + incl - v;
}

// sums and maxima per tile; scanned (or null, or `in` itself): the sums inside the tile up to and with each entry
__global__ void __launch_bounds__(kScanThreads) scan_sums_kernel(const int* in, long n, int* block_sums, int* block_max, int* scanned) {
    __shared__ int lds[8];
    const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    int s = 0, m = 0, item[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        item[k] = (base + k < n) ? in[base + k] : 0;
        s += item[k];
        m = item[k] > m ? item[k] : m;
    }
    int total;
    int sum = block_excl_scan(s, &total, lds);
    if (scanned)
#pragma unroll
        for (int k = 0; k < kScanItems; k++) {
            sum += item[k];
            if (base + k < n) scanned[base + k] = sum;
        }
    // block max through the same LDS words
    for (int d = kWave / 2; d > 0; d >>= 1) { int t = __shfl_xor(m, d); m = t > m ? t : m; }
    if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        int mm = 0;
        for (int k = 0; k < kScanThreads / kWave; k++) mm = lds[k] > mm ? lds[k] : mm;
        block_sums[blockIdx.x] = total;
        block_max[blockIdx.x] = mm;
    }
}

// whole scan in one workgroup (n small): out[0..n], optional total / max.  Each lane scans a
// contiguous chunk serially, the chunk totals are scanned across the workgroup once.
constexpr int kScanSmallThreads = 1024;
__global__ void __launch_bounds__(kScanSmallThreads) scan_small_kernel(const int* __restrict__ in, int n,
                                                                       int* __restrict__ out, int* out_total, int* out_max) {
    __shared__ int lds[16];
    const int chunk = (n + kScanSmallThreads) / kScanSmallThreads;          // covers indices 0..n
    const int lo = threadIdx.x * chunk;
    const int hi = lo + chunk < n ? lo + chunk : n;
    int sum = 0, mx = 0;
    for (int k = lo; k < hi; k++) {
        const int v = in[k];
        sum += v;
        mx = v > mx ? v : mx;
    }
    int total;
    int run = block_excl_scan(sum, &total, lds);
    for (int k = lo; k < lo + chunk && k <= n; k++) {
        out[k] = run;
        if (k < n) run += in[k];
    }
    for (int d = kWave / 2; d > 0; d >>= 1) { int t = __shfl_xor(mx, d); mx = t > mx ? t : mx; }
    if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        int mm = 0;
        for (int k = 0; k < kScanSmallThreads / kWave; k++) mm = lds[k] > mm ? lds[k] : mm;
        if (out_total) *out_total = total;
        if (out_max) *out_max = mm;
    }
}

// nodes > 0: also edge_counts[b] = out[(b+1)*nodes] (inclusive prefix of edges per box)
// Every workgroup adds up the sums of the workgroups before it (at most a few thousand values: one strided pass)
// instead of waiting for a third kernel to scan them; workgroup 0 also reduces all of them to the totals.
__global__ void __launch_bounds__(kScanThreads) scan_apply_kernel(const int* __restrict__ in, long n,
                                                                  const int* __restrict__ block_sums,
                                                                  const int* __restrict__ block_max, int nblocks,
                                                                  int* __restrict__ out, int nodes,
                                                                  int* __restrict__ edge_counts, int* out_total,
                                                                  int* out_max, int* out_overflow,
                                                                  const int* __restrict__ box_max, int n_box,
                                                                  int* out_box_max) {
    __shared__ int lds[8];
    __shared__ long long before_lds[kScanThreads / kWave];
    __shared__ int max_lds[kScanThreads / kWave];
    long long before = 0, all = 0;
    int mx = 0;
    const bool totals = blockIdx.x == 0;
    const int upto = totals ? nblocks : (int)blockIdx.x;
    for (int k = threadIdx.x; k < upto; k += kScanThreads) {
        const int v = block_sums[k];
        all += v;
        if (k < (int)blockIdx.x) before += v;
        if (totals) { const int m = block_max[k]; mx = m > mx ? m : mx; }
    }
    for (int d = kWave / 2; d > 0; d >>= 1) {
        before += __shfl_xor(before, d);
        all += __shfl_xor(all, d);
        const int t = __shfl_xor(mx, d);
        mx = t > mx ? t : mx;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        before_lds[threadIdx.x / kWave] = totals ? all : before;
        max_lds[threadIdx.x / kWave] = mx;
    }
    __syncthreads();
    long long sum_w = 0;
    int max_w = 0;
    for (int k = 0; k < kScanThreads / kWave; k++) {
        sum_w += before_lds[k];
        max_w = max_lds[k] > max_w ? max_lds[k] : max_w;
    }
    const int block_offset = totals ? 0 : (int)sum_w;         // (an overflowing total is flagged by workgroup 0)
    if (totals && box_max != nullptr && threadIdx.x < kWave) {
        // largest cell occupancy over the boxes (the per-box sort leaves one value per box)
        int m = 0;
        for (int k = threadIdx.x; k < n_box; k += kWave) { const int v = box_max[k] & ~kNanBit; m = v > m ? v : m; }
        for (int d = kWave / 2; d > 0; d >>= 1) { const int t = __shfl_xor(m, d); m = t > m ? t : m; }
        if (threadIdx.x == 0) *out_box_max = m;
    }
    if (totals && threadIdx.x == 0) {
        if (out_total) *out_total = sum_w > 0x7fffffffLL ? 0x7fffffff : (int)sum_w;
        if (out_max) *out_max = max_w;
        if (out_overflow) *out_overflow = sum_w > 0x7fffffffLL ? 1 : 0;
    }
    const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    int v[kScanItems];
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        s += v[k];
    }
    int total;
    int run = block_excl_scan(s, &total, lds) + block_offset;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        if (base + k <= n) {
            out[base + k] = run;   // index n receives the grand total
            if (nodes > 0 && base + k > 0) {
                const unsigned idx = (unsigned)(base + k), q = idx / (unsigned)nodes;   // n < 2^31: 32-bit divide
                if (q * (unsigned)nodes == idx) edge_counts[q - 1] = run;
            }
        }
        run += v[k];
    }
}


// One workgroup per home cell.  The count pass stages the 27 window cells in LDS once (wrapped positions
// + atom ids), each wave takes home atoms and sweeps the staged candidates 64 at a time; the hits of a
// group go straight into the atom's hit row, behind the hits of the groups before it, so a hit row lists
// the neighbours in window order.  The fill pass is a copy of the hit rows to their places in the edge
// list and never touches the geometry again.  Windows larger than the LDS tile (kCandCap candidates) read
// their tail from global memory.
//
// The hot loop is straight-line code:
//   * the tile is padded to a multiple of 64 with candidates at +infinity (their distance test fails),
//     so no lane checks whether its candidate exists;
//   * a hit row is addressed through a buffer descriptor that covers exactly that row: entries past its
//     capacity are dropped by the bounds check of the store, the count goes on, and the fill pass finds
//     such rows by their degree;
//   * minimum image without compares: remainder(t, box) = t - rint(t / box) box, evaluated as
//     fma(-rint(t * (1 / box)), box, t).  For |t| <= box the multiple is -1, 0 or 1 and the fma is
//     exact, so the result is the IEEE remainder bit for bit unless t / box is within rounding of
//     +-1/2, where the other representative may be chosen; there |result| is about box / 2, which
//     exceeds the cutoff (the grid has at least 3 cells per axis, so box > 2 cutoff): such a pair is
//     listed by neither choice.
//   * a wrapped coordinate lies in [0, box] with BOTH ends possible (remainderf(x - box/2, box) +
//     box/2 gives exactly box for x = box, -box, 3 box, ... and for x within half an ulp below box),
//     and such an atom sits in cell 0 because the cell index is taken modulo ndiv.  Only a home cell
//     whose window holds neither cell 0 nor cell ndiv - 1 on any axis (coordinates 2 .. ndiv - 3,
//     ndiv >= 5) skips the minimum image altogether: there |w_i - w_j| < 2/5 box.
struct Window {
    int M;            // candidates in the 27 cells
    int self_base;    // the home cell's atoms are candidates self_base .. self_base + home_n - 1
    int home_lo, home_n;
};

// First wave: lane t < 27 looks cell t of the window up, a shuffle scan gives the prefix of the lengths.
// Returns false (uniformly) when the home cell is empty.
__device__ __forceinline__ bool window_ranges(const Grid& g, const Workspace& w, int b, int cx, int cy, int cz,
                                              int* range_start, int* range_prefix, Window* win) {
    if (threadIdx.x < kWave) {
        const int lane = threadIdx.x;
        const int t = lane < 27 ? lane : 26;
        const int dx = t / 9 - 1, dy = (t / 3) % 3 - 1, dz = t % 3 - 1;      // divisions by constants: multiplies
        int nx = cx + dx, ny = cy + dy, nz = cz + dz;                        // periodic neighbours without a division
        nx = nx < 0 ? nx + g.nx : (nx >= g.nx ? nx - g.nx : nx);
        ny = ny < 0 ? ny + g.ny : (ny >= g.ny ? ny - g.ny : ny);
        nz = nz < 0 ? nz + g.nz : (nz >= g.nz ? nz - g.nz : nz);
        const int nc = ((b * g.nx + nx) * g.ny + ny) * g.nz + nz;
        const int start = w.cell_start[nc];
        const int len = lane < 27 ? w.cell_start[nc + 1] - start : 0;
        int incl = len;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) {
            const int up = __shfl_up(incl, d);
            if (lane >= d) incl += up;
        }
        if (lane < 27) {
            range_start[lane] = start;
            range_prefix[lane + 1] = incl;
        }
        if (lane == 0) range_prefix[0] = 0;
    }
    __syncthreads();
    win->M = range_prefix[27];
    win->self_base = range_prefix[13];
    win->home_lo = range_start[13];
    win->home_n = range_prefix[14] - range_prefix[13];
    return win->home_n > 0;
}

// candidate k of the concatenated window -> address in the cell-ordered array
__device__ __forceinline__ int locate(const int* range_start, const int* range_prefix, int k) {
    int lo = 0, hi = 26;   // last range with prefix <= k
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (range_prefix[mid] <= k) lo = mid; else hi = mid - 1;
    }
    return range_start[lo] + (k - range_prefix[lo]);
}

// WRAP: bit 0 / 1 / 2 = apply the minimum image along x / y / z
template <int WRAP>
__device__ __forceinline__ bool within_cutoff(const float4& self, const float4& o, const Grid& g, float ibx, float iby,
                                              float ibz) {
    float dx = self.x - o.x, dy = self.y - o.y, dz = self.z - o.z;
    if (WRAP & 1) dx = __fmaf_rn(-rintf(dx * ibx), g.bx, dx);
    if (WRAP & 2) dy = __fmaf_rn(-rintf(dy * iby), g.by, dy);
    if (WRAP & 4) dz = __fmaf_rn(-rintf(dz * ibz), g.bz, dz);
    const float d2 = __fmaf_rn(dz, dz, __fmaf_rn(dy, dy, dx * dx));
    return d2 <= g.r0sq;
}

// hits below this lane in a ballot, plus `add`
__device__ __forceinline__ int hits_below(unsigned long long mask, int add) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)(mask & 0xffffffffull), (unsigned)add));
}

// HitT: unsigned short (boxes of at most 65536 atoms) or int
__device__ __forceinline__ void store_hit(__amdgpu_buffer_rsrc_t row, int id, int entry, unsigned short) {
    __builtin_amdgcn_raw_buffer_store_b16((short)id, row, entry << 1, 0, 0);
}
__device__ __forceinline__ void store_hit(__amdgpu_buffer_rsrc_t row, int id, int entry, int) {
    __builtin_amdgcn_raw_buffer_store_b32(id, row, entry << 2, 0, 0);
}

template <int kCandCap, typename HitT>
__global__ void __launch_bounds__(256) count_kernel(Grid g, Workspace w) {
    __shared__ float4 cand[kCandCap];
    __shared__ int range_start[27];
    __shared__ int range_prefix[28];

    // grid (nz, ny, nx * batch): the cell coordinates come from the workgroup id without a division chain
    const int cz = blockIdx.x, cy = blockIdx.y;
    const int b = blockIdx.z / g.nx, cx = blockIdx.z - b * g.nx;
    Window win;
    if (!window_ranges(g, w, b, cx, cy, cz, range_start, range_prefix, &win)) return;   // uniform
    const int M = win.M;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), nwaves = blockDim.x / kWave;   // (scalar)

    const int staged = M < kCandCap ? M : kCandCap;
    const int padded = (staged + kWave - 1) & ~(kWave - 1);        // <= kCandCap (a multiple of 64)
    const float inf = __int_as_float(0x7f800000);
    for (int k = threadIdx.x; k < padded; k += blockDim.x)
        cand[k] = k < staged ? w.sorted[locate(range_start, range_prefix, k)] : make_float4(inf, inf, inf, __int_as_float(-1));
    __syncthreads();

    // an axis needs the minimum image unless the window stays clear of cells 0 and ndiv - 1 (see above)
    const int wrap = ((g.nx < 5 || cx < 2 || cx > g.nx - 3) ? 1 : 0) | ((g.ny < 5 || cy < 2 || cy > g.ny - 3) ? 2 : 0) |
                     ((g.nz < 5 || cz < 2 || cz > g.nz - 3) ? 4 : 0);
    const float ibx = 1.0f / g.bx, iby = 1.0f / g.by, ibz = 1.0f / g.bz;
    const int node_base = b * g.nodes;
    const int row_bytes = w.hit_cap * (int)sizeof(HitT);
    HitT* const hits = static_cast<HitT*>(w.hits);

    const int self_base = __builtin_amdgcn_readfirstlane(win.self_base), home_n = __builtin_amdgcn_readfirstlane(win.home_n);
    for (int h = wave; h < home_n; h += nwaves) {
        const int k_self = self_base + h;              // uniform
        float4 self;
        if (k_self < kCandCap) self = cand[k_self];
        else self = w.sorted[win.home_lo + h];
        const int row = node_base + __builtin_amdgcn_readfirstlane(__float_as_int(self.w));
        // descriptor of this atom's hit row alone: a store past the row's capacity is dropped
        const __amdgpu_buffer_rsrc_t hit_row =
            __builtin_amdgcn_make_buffer_rsrc(hits + (long)row * w.hit_cap, 0, row_bytes, 0x00020000);
        // the home atom is itself a candidate and passes the distance test: its bit is taken out of the ballot of
        // its group with scalar instructions (no lane compares ids)
        const int self_group = k_self & ~(kWave - 1);
        const unsigned long long self_clear = ~(1ull << (k_self & (kWave - 1)));
        int running = 0;
        auto sweep = [&](auto wrap_tag) {
            constexpr int kWrap = decltype(wrap_tag)::value;
            for (int k0 = 0; k0 < padded; k0 += kWave) {
                const float4 o = cand[k0 + lane];
                unsigned long long mask = __ballot(within_cutoff<kWrap>(self, o, g, ibx, iby, ibz));
                if (k0 == self_group) mask &= self_clear;
                // (box-local atom ids: the fill pass adds the box's first row)
                if (__builtin_amdgcn_inverse_ballot_w64(mask))
                    store_hit(hit_row, __float_as_int(o.w), hits_below(mask, running), HitT{});
                running += __popcll(mask);
            }
        };
        switch (wrap) {                                // uniform over the workgroup
            case 0: sweep(std::integral_constant<int, 0>{}); break;
            case 1: sweep(std::integral_constant<int, 1>{}); break;
            case 2: sweep(std::integral_constant<int, 2>{}); break;
            case 3: sweep(std::integral_constant<int, 3>{}); break;
            case 4: sweep(std::integral_constant<int, 4>{}); break;
            case 5: sweep(std::integral_constant<int, 5>{}); break;
            case 6: sweep(std::integral_constant<int, 6>{}); break;
            default: sweep(std::integral_constant<int, 7>{}); break;
        }
        // candidates beyond the tile: from global memory
        for (int k0 = kCandCap; k0 < M; k0 += kWave) {
            const int k = k0 + lane;
            bool hit = false;
            int other = 0;
            if (k < M) {
                const float4 o = w.sorted[locate(range_start, range_prefix, k)];
                other = __float_as_int(o.w);
                hit = k != k_self && within_cutoff<7>(self, o, g, ibx, iby, ibz);
            }
            const unsigned long long mask = __ballot(hit);
            if (hit) store_hit(hit_row, other, hits_below(mask, running), HitT{});
            running += __popcll(mask);
        }
        if (lane == 0) w.degree[row] = running;
    }
}

// What the fill pass writes per edge: the int32 indices, and for a caller that asked for them their int64 copies and
// the edge vector boxwrap(box, x_j - x_i).
struct EdgeOut {
    int* src;
    int* dst;
    int64_t* src64;     // both or neither
    int64_t* dst64;
    float* r_ij;        // or null
    const float* x;     // unwrapped positions (with r_ij)

    // the arrays from edge e on
    __device__ __forceinline__ EdgeOut from(int e) const {
        return EdgeOut{src + e, dst + e, src64 ? src64 + e : nullptr, dst64 ? dst64 + e : nullptr, r_ij ? r_ij + 3 * (long)e : nullptr, x};
    }
    __device__ __forceinline__ void store(int e, int i, int j) const {
        src[e] = i;
        dst[e] = j;
        if (src64) {
            src64[e] = i;
            dst64[e] = j;
        }
    }
    __device__ __forceinline__ void store_vector(int e, const float3& r) const {
        float* to = r_ij + 3 * (long)e;
        to[0] = r.x;
        to[1] = r.y;
        to[2] = r.z;
    }
};

// Fill pass, slow path: one wave sweeps the window of atom `row` again (candidates from global memory, all axes with
// the minimum image) and writes its hits at out_pos, in window order.  For rows whose hit row was too short.
__device__ void refill_row(const Grid& g, const Workspace& w, int row, int out_pos, int capacity, const EdgeOut& out) {
    const int lane = threadIdx.x & (kWave - 1);
    const int b = row / g.nodes;
    const int id_self = row - b * g.nodes;
    const int node_base = b * g.nodes;
    const float4 self = w.wrapped[row];
    int c = (w.cell_of[row] & ~kNanCell) - b * g.ncells;
    const int cz = c % g.nz;
    c /= g.nz;
    const int cy = c % g.ny, cx = c / g.ny;
    const int t = lane < 27 ? lane : 26;
    const int dx = t / 9 - 1, dy = (t / 3) % 3 - 1, dz = t % 3 - 1;
    int nx = cx + dx, ny = cy + dy, nz = cz + dz;
    nx = nx < 0 ? nx + g.nx : (nx >= g.nx ? nx - g.nx : nx);
    ny = ny < 0 ? ny + g.ny : (ny >= g.ny ? ny - g.ny : ny);
    nz = nz < 0 ? nz + g.nz : (nz >= g.nz ? nz - g.nz : nz);
    const int nc = ((b * g.nx + nx) * g.ny + ny) * g.nz + nz;
    const int start = w.cell_start[nc];
    const int len = lane < 27 ? w.cell_start[nc + 1] - start : 0;
    const int incl = wave_incl_scan(len, lane);
    const int excl = incl - len;                       // lane t < 27: candidates before cell t of the window
    const int M = __shfl(incl, 26);
    const float ibx = 1.0f / g.bx, iby = 1.0f / g.by, ibz = 1.0f / g.bz;
    int cnt = 0;
    for (int k0 = 0; k0 < M; k0 += kWave) {
        const int k = k0 + lane;
        int lo = 0, hi = 26;                           // last cell of the window with excl <= k (5 halvings of 27)
#pragma unroll
        for (int it = 0; it < 5; it++) {
            const int mid = (lo + hi + 1) >> 1;
            const int pm = __shfl(excl, mid);
            if (pm <= k) lo = mid; else hi = mid - 1;
        }
        const int st = __shfl(start, lo), ex = __shfl(excl, lo);
        bool hit = false;
        int other = 0;
        if (k < M) {
            const float4 o = w.sorted[st + (k - ex)];
            other = __float_as_int(o.w);
            hit = other != id_self && within_cutoff<7>(self, o, g, ibx, iby, ibz);
        }
        const unsigned long long mask = __ballot(hit);
        const int pos = out_pos + hits_below(mask, cnt);
        if (hit && pos >= 0 && pos < capacity) {
            out.store(pos, row, node_base + other);
            if (out.r_ij)
                out.store_vector(pos, wrapped_difference(load3(out.x + 3 * (long)(node_base + other)), load3(out.x + 3 * (long)row),
                                                         box_of(g.bx, g.by, g.bz)));
        }
        cnt += __popcll(mask);
    }
}

// Fill pass: a workgroup takes kFillRows consecutive rows, whose edges are one contiguous range of the edge list; a
// thread takes every 256th edge of the range, finds its row among the staged row starts and copies one entry of
// that row's hits.  Edges beyond the capacity are dropped.
constexpr int kFillRows = 64;
template <typename HitT>
__global__ void __launch_bounds__(256) fill_kernel(Grid g, Workspace w, const int* __restrict__ row_ptr,
                                                   EdgeOut out, int capacity) {
    __shared__ int rp[kFillRows + 1];
    __shared__ int first_row[kFillRows];      // first row of the box that the row belongs to
    const long A = (long)g.batch * g.nodes;
    const long r0 = (long)blockIdx.x * kFillRows;
    const int nrows = A - r0 < kFillRows ? (int)(A - r0) : kFillRows;
    if ((int)threadIdx.x <= nrows) rp[threadIdx.x] = row_ptr[r0 + threadIdx.x];
    if ((int)threadIdx.x < nrows) first_row[threadIdx.x] = (int)((r0 + threadIdx.x) / g.nodes) * g.nodes;
    __syncthreads();
    const int cap = w.hit_cap;
    const HitT* __restrict__ hits = static_cast<const HitT*>(w.hits);
    const int e_hi = rp[nrows];
    for (int e = rp[0] + (int)threadIdx.x; e < e_hi; e += 256) {
        int lo = 0, hi = nrows - 1;                    // last row with rp <= e (6 halvings of 64)
#pragma unroll
        for (int it = 0; it < 6; it++) {
            const int mid = (lo + hi + 1) >> 1;
            if (rp[mid] <= e) lo = mid; else hi = mid - 1;
        }
        const int idx = e - rp[lo], deg = rp[lo + 1] - rp[lo];
        if (deg <= cap && idx >= 0 && idx < deg && e >= 0 && e < capacity)
            out.store(e, (int)(r0 + lo), first_row[lo] + (int)hits[(r0 + lo) * cap + idx]);
    }
    // rows with more hits than a hit row holds: a wave each
    const int wave = threadIdx.x / kWave;
    for (int r = wave; r < nrows; r += 256 / kWave)
        if (rp[r + 1] - rp[r] > cap) refill_row(g, w, (int)(r0 + r), rp[r], capacity, out);
}

// Small boxes: binning, sort and count in ONE kernel.  gridDim.x workgroups share a box; each bins and sorts the whole
// box in LDS (a few thousand clocks for at most kBoxNodes atoms: cheaper than the two launches and the round trip through
// memory it replaces) and then counts the home cells blockIdx.x * 8 + wave, + 8 gridDim.x, ...: a wave takes a home
// cell, its lanes hold one group of 64 candidates of the window at a time in registers, and every home atom of the cell
// sweeps them; lane h keeps the running count of home atom h.  Same hit rows, degrees and tables as the separate kernels.
// What bounds it is latency (a dozen dependent LDS phases); 2 launches per search instead of 6 + (see graph_fill_kernel).
constexpr int kBoxThreads = 512, kBoxNodes = 2048, kBoxCells = 4096, kBoxWaves = kBoxThreads / kWave;
template <int kPer, typename HitT>
__global__ void __launch_bounds__(kBoxThreads) box_search_kernel(const float* __restrict__ x, Grid g, Workspace w) {
    constexpr int kNodes = kPer * kBoxThreads;
    __shared__ float4 sorted[kNodes];
    __shared__ int placed[kNodes + 8];            // keys (cell << 11 | atom): see sort_box_kernel
    __shared__ int start[kBoxCells + 1];
    __shared__ int wave_sum[kBoxWaves], wave_max[kBoxWaves], wave_nan[kBoxWaves];
    const int part = blockIdx.x, parts = gridDim.x, b = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const long base = (long)b * g.nodes;
    const int cell_base = b * g.ncells;

    float4 rec[kPer];
    int cl[kPer], sl[kPer], nan = 0;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = tid + kBoxThreads * j;
        cl[j] = -1;
        if (i < g.nodes) {
            const float* p = x + 3 * (base + i);
            const float px = p[0], py = p[1], pz = p[2];
            nan |= (px != px || py != py || pz != pz) ? 1 : 0;
            rec[j] = make_float4(wrap_into_box(px, g.bx), wrap_into_box(py, g.by), wrap_into_box(pz, g.bz), __int_as_float(i));
            cl[j] = (cell_coord(rec[j].x, g.bx, g.nx) * g.ny + cell_coord(rec[j].y, g.by, g.ny)) * g.nz +
                    cell_coord(rec[j].z, g.bz, g.nz);
        }
    }
    for (int c = tid; c <= g.ncells; c += kBoxThreads) start[c] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; j++)
        if (cl[j] >= 0) sl[j] = atomicAdd(&start[cl[j]], 1);
    __syncthreads();
    // exclusive scan of the cell sizes: a thread owns `per` consecutive cells
    const int per = (g.ncells + kBoxThreads - 1) / kBoxThreads;
    int sum = 0, mx = 0;
    for (int k = 0; k < per; k++) {
        const int c = tid * per + k;
        const int v = c < g.ncells ? start[c] : 0;
        sum += v;
        mx = v > mx ? v : mx;
    }
    const int incl = wave_incl_scan(sum, lane);
    for (int d = kWave / 2; d > 0; d >>= 1) { const int t = __shfl_xor(mx, d); mx = t > mx ? t : mx; }
    const int any_nan = __any(nan);
    if (lane == kWave - 1) wave_sum[wave] = incl;
    if (lane == 0) { wave_max[wave] = mx; wave_nan[wave] = any_nan; }
    __syncthreads();
    int run = incl - sum;
    for (int k = 0; k < wave; k++) run += wave_sum[k];
    for (int k = 0; k < per; k++) {
        const int c = tid * per + k;
        if (c < g.ncells) {
            const int v = start[c];
            start[c] = run;
            run += v;
        }
    }
    if (tid == 0) start[g.ncells] = g.nodes;
    if (tid < 8) placed[g.nodes + tid] = 0x7fffffff;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; j++)
        if (cl[j] >= 0) placed[start[cl[j]] + sl[j]] = (cl[j] << 11) | (tid + kBoxThreads * j);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        if (cl[j] < 0) continue;
        const int key = (cl[j] << 11) | (tid + kBoxThreads * j);
        const int lo = start[cl[j]], hi = start[cl[j] + 1];
        int rank = 0;
        for (int q0 = lo; q0 < hi; q0 += 8) {
            int v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = placed[q0 + u];      // (q0 < nodes: at most 7 entries into the sentinels)
#pragma unroll
            for (int u = 0; u < 8; u++) rank += v[u] < key ? 1 : 0;
        }
        sorted[lo + rank] = rec[j];
        if (part == 0) {                          // (the fill pass sweeps rows that overflow their hit row again)
            w.wrapped[base + tid + kBoxThreads * j] = rec[j];
            w.cell_of[base + tid + kBoxThreads * j] = cell_base + cl[j];
        }
    }
    if (part == 0) {
        for (int c = tid; c < g.ncells; c += kBoxThreads) w.cell_start[cell_base + c] = (int)base + start[c];
        if (tid == 0) {
            int m = 0, any = 0;
            for (int k = 0; k < kBoxWaves; k++) { m = wave_max[k] > m ? wave_max[k] : m; any |= wave_nan[k]; }
            w.box_max[b] = m | (any ? kNanBit : 0);
            if (b == g.batch - 1) w.cell_start[(long)g.batch * g.ncells] = g.batch * g.nodes;
        }
    }
    __syncthreads();
    for (int p = tid + kBoxThreads * part; p < g.nodes; p += kBoxThreads * parts) w.sorted[base + p] = sorted[p];

    const float ibx = 1.0f / g.bx, iby = 1.0f / g.by, ibz = 1.0f / g.bz;
    HitT* const hits = static_cast<HitT*>(w.hits);
    const int row_bytes = w.hit_cap * (int)sizeof(HitT);
    for (int c = part * kBoxWaves + wave; c < g.ncells; c += parts * kBoxWaves) {        // uniform in the wave
        const int home_lo = __builtin_amdgcn_readfirstlane(start[c]), home_hi = __builtin_amdgcn_readfirstlane(start[c + 1]);
        if (home_lo == home_hi) continue;
        const int cz = c % g.nz, cxy = c / g.nz, cy = cxy % g.ny, cx = cxy / g.ny;
        const int t = lane < 27 ? lane : 26;
        const int dx = t / 9 - 1, dy = (t / 3) % 3 - 1, dz = t % 3 - 1;
        int nx = cx + dx, ny = cy + dy, nz = cz + dz;
        nx = nx < 0 ? nx + g.nx : (nx >= g.nx ? nx - g.nx : nx);
        ny = ny < 0 ? ny + g.ny : (ny >= g.ny ? ny - g.ny : ny);
        nz = nz < 0 ? nz + g.nz : (nz >= g.nz ? nz - g.nz : nz);
        const int nc = (nx * g.ny + ny) * g.nz + nz;
        const int st = start[nc];
        const int len = lane < 27 ? start[nc + 1] - st : 0;
        int pre = len;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) {
            const int up = __shfl_up(pre, d);
            if (lane >= d) pre += up;
        }
        const int excl = pre - len;
        const int M = __builtin_amdgcn_readlane(pre, 26);
        const bool inner = g.nx >= 5 && cx >= 2 && cx <= g.nx - 3 && g.ny >= 5 && cy >= 2 && cy <= g.ny - 3 && g.nz >= 5 &&
                           cz >= 2 && cz <= g.nz - 3;
        for (int h0 = home_lo; h0 < home_hi; h0 += kWave) {          // (one trip unless a cell holds more than 64 atoms)
            const int hn = home_hi - h0 < kWave ? home_hi - h0 : kWave;
            int counts = 0;                                          // lane h: hits of home atom h0 + h so far
            for (int k0 = 0; k0 < M; k0 += kWave) {
                const int k = k0 + lane;
                int lo = 0, hi = 26;                                 // last cell of the window with excl <= k
#pragma unroll
                for (int it = 0; it < 5; it++) {
                    const int mid = (lo + hi + 1) >> 1;
                    const int pm = __shfl(excl, mid);
                    if (pm <= k) lo = mid; else hi = mid - 1;
                }
                const int idx = __shfl(st, lo) + (k - __shfl(excl, lo));
                const bool valid = k < M;
                const float4 o = sorted[valid ? idx : home_lo];
                for (int h = 0; h < hn; h++) {
                    const float4 self = sorted[h0 + h];              // one address: a broadcast
                    const bool close = inner ? within_cutoff<0>(self, o, g, ibx, iby, ibz)
                                             : within_cutoff<7>(self, o, g, ibx, iby, ibz);
                    const unsigned long long mask = __ballot(close && valid && idx != h0 + h);
                    const int seen = __builtin_amdgcn_readlane(counts, h);
                    const int row = (int)base + __builtin_amdgcn_readfirstlane(__float_as_int(self.w));
                    const __amdgpu_buffer_rsrc_t hit_row =
                        __builtin_amdgcn_make_buffer_rsrc(hits + (long)row * w.hit_cap, 0, row_bytes, 0x00020000);
                    if (__builtin_amdgcn_inverse_ballot_w64(mask))
                        store_hit(hit_row, __float_as_int(o.w), hits_below(mask, seen), HitT{});
                    counts += lane == h ? __popcll(mask) : 0;
                }
            }
            if (lane < hn) w.degree[base + __float_as_int(sorted[h0 + lane].w)] = counts;
        }
    }
}

// The statistics of the whole graph, by the first workgroup before anything else: the host waits for them.
__device__ void graph_statistics(const Workspace& w, long A, int tiled, int n_box, int* stats) {
    __shared__ long long wave_all[4];
    __shared__ int wave_mx[4], wave_cell[4], wave_flag[4];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    long long all = 0;
    int mx = 0, cell = 0, flag = 0;
    const long n = tiled ? A / kScanTile + 1 : A;             // ceil((A + 1) / kScanTile) tiles
    const int* sums = tiled ? w.deg_sums : w.degree;
    const int* maxima = tiled ? w.deg_max : w.degree;
    for (long k = tid; k < n; k += 256) {
        all += sums[k];
        const int m = maxima[k];
        mx = m > mx ? m : mx;
    }
    for (int k = tid; k < n_box; k += 256) {
        const int v = w.box_max[k] & ~kNanBit;
        cell = v > cell ? v : cell;
        flag |= w.box_max[k] & kNanBit;
    }
    for (int d = kWave / 2; d > 0; d >>= 1) {
        all += __shfl_xor(all, d);
        int t = __shfl_xor(mx, d);
        mx = t > mx ? t : mx;
        t = __shfl_xor(cell, d);
        cell = t > cell ? t : cell;
        flag |= __shfl_xor(flag, d);
    }
    if (lane == 0) {
        wave_all[wave] = all;
        wave_mx[wave] = mx;
        wave_cell[wave] = cell;
        wave_flag[wave] = flag;
    }
    __syncthreads();
    if (tid == 0) {
        for (int k = 1; k < 4; k++) {
            all += wave_all[k];
            mx = wave_mx[k] > mx ? wave_mx[k] : mx;
            cell = wave_cell[k] > cell ? wave_cell[k] : cell;
            flag |= wave_flag[k];
        }
        // (a host may be polling these words: each is stored once, at system scope)
        const int words[4] = {all > 0x7fffffffLL ? 0x7fffffff : (int)all, cell, mx,
                              (all > 0x7fffffffLL ? 1 : 0) | (flag ? 4 : 0)};
#pragma unroll
        for (int k = 0; k < 4; k++) __hip_atomic_store(stats + k, words[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
// Row r0 + lane where scan_sums_kernel has left the sums inside the tile in the place of the degrees; a wave adds the tiles before by
// itself.  The rows r0 .. r0 + nrows - 1 lie in one tile.
struct FillRow { int degree, start; };
__device__ __forceinline__ FillRow row_of_tile(const Workspace& w, long r0, int lane, int nrows) {
    const int tile = (int)(r0 / kScanTile);
    int incl = 0, prev = 0, before = 0;
    if (lane < nrows) {
        incl = w.degree[r0 + lane];
        if ((r0 + lane) % kScanTile != 0) prev = w.degree[r0 + lane - 1];
    }
    for (int k = lane; k < tile; k += kWave) before += w.deg_sums[k];
    for (int d = kWave / 2; d > 0; d >>= 1) before += __shfl_xor(before, d);
    return FillRow{incl - prev, before + prev};
}
__device__ __forceinline__ void put_row(const Grid& g, long A, long r, const FillRow& own, int* row_ptr, int* edge_counts) {
    row_ptr[r] = own.start;
    const long next = r + 1;
    if (next == A) row_ptr[A] = own.start + own.degree;
    const unsigned q = (unsigned)next / (unsigned)g.nodes;                        // (next < 2^31: 32-bit divide)
    if (q * (unsigned)g.nodes == (unsigned)next) edge_counts[q - 1] = own.start + own.degree;
}

// Row pointer, statistics and edges of a whole graph in one kernel.  A workgroup takes `rows_per` consecutive rows and
// finds the position of its first edge by adding up the degrees of the rows before it: those of its tile of kScanTile
// rows and the sums of the tiles before (tiled: scan_sums_kernel has left them), or simply all of them (at most
// kDirectRows degrees from the L2: cheaper than a launch).  Workgroup 0 also reduces everything to the statistics.  The
// edge's int64 indices and its vector are written here, where i and j are in registers, instead of by three kernels that
// read the edge list back.  A wave takes RW rows, a lane an edge of each: what a row's edges are does not depend on where they go,
// so that its hits, its atom and the degrees of the rows before it are all requested at once, and the neighbours' atoms as
// soon as the hits are there.  6.8 M edges: 83 us (97 with the edges of 64 rows dealt out to the threads, whose rows had to be found,
// and a barrier after the sums).  Bound by the stores, 36 bytes per edge with everything asked for (44 us of them, 243 MB), and
// the two dependent loads before them, which wait behind the stores of other waves; 16-byte stores of four edges to a thread
// and eight waves per SIMD changed nothing or spilled.
constexpr long kDirectRows = 16384;
template <typename HitT, int RW>
__global__ void __launch_bounds__(256) graph_fill_kernel(Grid g, Workspace w, int tiled, int n_box, int* __restrict__ row_ptr,
                                                         int* __restrict__ edge_counts, int* stats, int capacity, EdgeOut out,
                                                         int* __restrict__ order) {
    constexpr int rows_per = 4 * RW;
    static_assert(rows_per <= kWave && kScanTile % rows_per == 0, "a wave holds the degrees of all rows, which lie in one tile");
    __shared__ int wave_before[4];
    const long A = (long)g.batch * g.nodes;
    const long r0 = (long)blockIdx.x * rows_per;
    const int nrows = A - r0 < rows_per ? (int)(A - r0) : rows_per;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int cap = w.hit_cap;
    const HitT* __restrict__ hits = static_cast<const HitT*>(w.hits);
    const float* __restrict__ x = out.x;
    if (blockIdx.x == 0) graph_statistics(w, A, tiled, n_box, stats);      // (before its own loads, which these would wait behind)
    int hit[RW];
    float3 xi[RW];
#pragma unroll
    for (int k = 0; k < RW; k++) {                    // (a wave's rows are scalars: so are their addresses)
        const int at = wave * RW + k;
        const long r = r0 + (at < nrows ? at : 0);
        hit[k] = lane < cap ? (int)hits[r * cap + lane] : 0;     // (past the row's degree: not used)
        if (x) xi[k] = load3(x + 3 * r);
    }
    FillRow own;                                                  // row r0 + lane
    if (tiled) {
        own = row_of_tile(w, r0, lane, nrows);
    } else {
        own.degree = lane < nrows ? w.degree[r0 + lane] : 0;
        int before = 0;
        for (long r = tid; r < r0; r += 256) before += w.degree[r];
        for (int d = kWave / 2; d > 0; d >>= 1) before += __shfl_xor(before, d);
        if (lane == 0) wave_before[wave] = before;
        const int incl = wave_incl_scan(own.degree, lane);        // (every wave by itself)
        __syncthreads();
        own.start = wave_before[0] + wave_before[1] + wave_before[2] + wave_before[3] + incl - own.degree;
    }
    const int my_degree = own.degree, my_start = own.start;

    const int my_box = (int)((unsigned)(r0 + (lane < nrows ? lane : 0)) / (unsigned)g.nodes) * g.nodes;      // first row of the row's box
    float3 xj[RW];
#pragma unroll
    for (int k = 0; k < RW; k++) {
        const int at = wave * RW + k, degree = __builtin_amdgcn_readlane(my_degree, at);
        hit[k] = lane < degree ? __builtin_amdgcn_readlane(my_box, at) + hit[k] : (int)r0;
        if (x) xj[k] = load3(x + 3 * (long)(degree <= cap ? hit[k] : (int)r0));
    }
    const Box3 box = box_of(g.bx, g.by, g.bz);
#pragma unroll
    for (int k = 0; k < RW; k++) {
        const int at = wave * RW + k, degree = __builtin_amdgcn_readlane(my_degree, at), start = __builtin_amdgcn_readlane(my_start, at);
        if (at >= nrows || start < 0) continue;
        const int row = (int)r0 + at;
        if (degree > cap) {
            refill_row(g, w, row, start, capacity, out);
            continue;
        }
        const EdgeOut here = out.from(start);
        const int room = capacity - start, n = degree < room ? degree : room;
        if (lane < n) {
            here.store(lane, row, hit[k]);
            if (x) here.store_vector(lane, wrapped_difference(xj[k], xi[k], box));
        }
        for (int t = lane + kWave; t < n; t += kWave) {
            const int j = __builtin_amdgcn_readlane(my_box, at) + (int)hits[(long)row * cap + t];
            here.store(t, row, j);
            if (x) here.store_vector(t, wrapped_difference(load3(x + 3 * (long)j), xi[k], box));
        }
    }
    if (wave == 0 && lane < nrows) put_row(g, A, r0 + lane, own, row_ptr, edge_counts);
    if (wave == 1 && lane < nrows && order) {
        const unsigned k = (unsigned)(r0 + lane);
        order[k] = (int)(k / (unsigned)g.nodes) * g.nodes + __float_as_int(w.sorted[k].w);
    }
}

// The same with the edges of 64 rows dealt out to the threads, which find their rows by bisection: for rows much shorter than a wave.
constexpr int kFillUnroll = 4;
template <typename HitT>
__global__ void __launch_bounds__(256) graph_fill_dealt_kernel(Grid g, Workspace w, int n_box, int* __restrict__ row_ptr,
                                                               int* __restrict__ edge_counts, int* stats, int capacity, EdgeOut out,
                                                               int* __restrict__ order) {
    constexpr int rows_per = kFillRows;
    __shared__ int rp[kFillRows + 1];
    __shared__ int first_row[kFillRows];      // first row of the box that the row belongs to
    __shared__ float3 x_row[kFillRows];
    const long A = (long)g.batch * g.nodes;
    const long r0 = (long)blockIdx.x * rows_per;
    const int nrows = A - r0 < rows_per ? (int)(A - r0) : rows_per;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    if (blockIdx.x == 0) graph_statistics(w, A, 1, n_box, stats);
    if (wave == 0) {
        const FillRow own = row_of_tile(w, r0, lane, nrows);
        if (lane < nrows) {
            rp[lane + 1] = own.start + own.degree;
            put_row(g, A, r0 + lane, own, row_ptr, edge_counts);
        }
        if (lane == 0) rp[0] = own.start;
        if (lane >= nrows && lane < rows_per) rp[lane + 1] = 0x7fffffff;
    }
    if (wave == 1 && lane < nrows) {
        const unsigned k = (unsigned)(r0 + lane);
        const int first = (int)(k / (unsigned)g.nodes) * g.nodes;
        first_row[lane] = first;
        if (order) order[k] = first + __float_as_int(w.sorted[k].w);
    }
    if (wave == 2 && lane < nrows && out.r_ij) x_row[lane] = load3(out.x + 3 * (r0 + lane));
    __syncthreads();
    const int cap = w.hit_cap;
    const HitT* __restrict__ hits = static_cast<const HitT*>(w.hits);
    const int e_hi = rp[nrows];
    const Box3 box = box_of(g.bx, g.by, g.bz);
    for (int e0 = rp[0] + tid; e0 < e_hi; e0 += 256 * kFillUnroll) {
        int row[kFillUnroll], j[kFillUnroll];
        bool ok[kFillUnroll];
#pragma unroll
        for (int u = 0; u < kFillUnroll; u++) {
            const int e = e0 + 256 * u;
            int lo = 0;                                // last row with rp <= e (rp ends in INT_MAX past the last row)
            for (int step = rows_per >> 1; step > 0; step >>= 1) lo += rp[lo + step] <= e ? step : 0;
            lo = lo < nrows ? lo : nrows - 1;          // (a position past the last edge: discarded below, but it must not
                                                       // name a row that is not staged, its atom is read all the same)
            const int idx = e - rp[lo], deg = rp[lo + 1] - rp[lo];
            ok[u] = e < e_hi && deg <= cap && idx >= 0 && idx < deg && e >= 0 && e < capacity;
            row[u] = lo;
            j[u] = ok[u] ? (int)hits[(r0 + lo) * cap + idx] : 0;
        }
        float3 xj[kFillUnroll];
#pragma unroll
        for (int u = 0; u < kFillUnroll; u++) {
            j[u] += first_row[row[u]];
            if (out.r_ij) xj[u] = load3(out.x + 3 * (long)j[u]);
        }
#pragma unroll
        for (int u = 0; u < kFillUnroll; u++)
            if (ok[u]) out.store(e0 + 256 * u, (int)r0 + row[u], j[u]);
        if (out.r_ij) {
#pragma unroll
            for (int u = 0; u < kFillUnroll; u++) {
                const float3 r = wrapped_difference(xj[u], x_row[row[u]], box);
                if (ok[u]) out.store_vector(e0 + 256 * u, r);
            }
        }
    }
    for (int r = wave; r < nrows; r += 4)
        if (rp[r + 1] - rp[r] > cap) refill_row(g, w, (int)(r0 + r), rp[r], capacity, out);
}

// order[k] = global id of the k-th atom in cell order (cells x-major, atoms by id inside a cell)
__global__ void __launch_bounds__(256) cell_order_kernel(Grid g, Workspace w, int* __restrict__ order) {
    const long A = (long)g.batch * g.nodes;
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= A) return;
    order[k] = (int)(k / g.nodes) * g.nodes + __float_as_int(w.sorted[k].w);
}

__global__ void __launch_bounds__(256) wrap_cells_kernel(const float* __restrict__ x, Grid g,
                                                         float* __restrict__ wrapped, int* __restrict__ cell) {
    const long A = (long)g.batch * g.nodes;
    const long a = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= A) return;
    const float wx = wrap_into_box(x[3 * a + 0], g.bx);
    const float wy = wrap_into_box(x[3 * a + 1], g.by);
    const float wz = wrap_into_box(x[3 * a + 2], g.bz);
    wrapped[3 * a + 0] = wx; wrapped[3 * a + 1] = wy; wrapped[3 * a + 2] = wz;
    cell[a] = (cell_coord(wx, g.bx, g.nx) * g.ny + cell_coord(wy, g.by, g.ny)) * g.nz + cell_coord(wz, g.bz, g.nz);
}

__global__ void __launch_bounds__(256) pad_kernel(const int* __restrict__ row_ptr, const int* __restrict__ dst,
                                                  long A, int nodes, int nmax, int* __restrict__ neighbours,
                                                  int* __restrict__ counts) {
    // one wave per node
    const long a = ((long)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const int lane = threadIdx.x & (kWave - 1);
    if (a >= A) return;
    const int lo = row_ptr[a], n = row_ptr[a + 1] - lo;
    const int node_base = (int)(a / nodes) * nodes;
    if (lane == 0) counts[a] = n;
    for (int k = lane; k < n && k < nmax; k += kWave) neighbours[a * nmax + k] = dst[lo + k] - node_base;
}

__global__ void __launch_bounds__(256) padded_read_kernel(const int* __restrict__ counts,
                                                          const int* __restrict__ neighbours,
                                                          const float* __restrict__ x, long A, int nodes, int nmax,
                                                          int chan, float* __restrict__ edge) {
    // flat over (node, slot, chan)
    const long total = A * nmax * chan;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const int c = (int)(t % chan);
        const long as = t / chan;
        const int j = (int)(as % nmax);
        const long a = as / nmax;
        float v = 0.f;
        if (j < counts[a]) {
            const long nb = (a / nodes) * nodes + neighbours[a * nmax + j];
            v = x[nb * chan + c];
        }
        edge[t] = v;
    }
}

__global__ void __launch_bounds__(256) padded_reduce_kernel(const int* __restrict__ counts,
                                                            const float* __restrict__ edge, long A, int nmax,
                                                            int chan, float* __restrict__ out) {
    const long total = A * chan;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const int c = (int)(t % chan);
        const long a = t / chan;
        const int n = counts[a] < nmax ? counts[a] : nmax;
        float s = 0.f;
        for (int j = 0; j < n; j++) s += edge[(a * nmax + j) * chan + c];
        out[t] = s;
    }
}


__global__ void __launch_bounds__(256) edge_vectors_kernel(const float* __restrict__ x, const int* __restrict__ src,
                                                           const int* __restrict__ dst, long E, float bx, float by,
                                                           float bz, float* __restrict__ r_ij,
                                                           int8_t* __restrict__ shift) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const float3 xi = load3(x + 3 * (long)src[e]), xj = load3(x + 3 * (long)dst[e]);
    const float3 r = wrapped_difference(xj, xi, box_of(bx, by, bz));
    r_ij[3 * e + 0] = r.x;
    r_ij[3 * e + 1] = r.y;
    r_ij[3 * e + 2] = r.z;
    if (shift) {
        shift[3 * e + 0] = (int8_t)rintf(__fdiv_rn((xj.x - xi.x) - r.x, bx));
        shift[3 * e + 1] = (int8_t)rintf(__fdiv_rn((xj.y - xi.y) - r.y, by));
        shift[3 * e + 2] = (int8_t)rintf(__fdiv_rn((xj.z - xi.z) - r.z, bz));
    }
}

int run_scan(const int* in, long n, int* out, Workspace& w, int* out_total, int* out_max, int* out_overflow,
             hipStream_t st, int nodes = 0, int* edge_counts = nullptr) {
    if (n <= 16384 && nodes == 0 && out_overflow == nullptr) {
        hipLaunchKernelGGL(scan_small_kernel, dim3(1), dim3(kScanSmallThreads), 0, st, in, (int)n, out, out_total, out_max);
        return check_launch("neighbour scan");
    }
    const int nblocks = (int)ceil_div(n + 1, kScanTile);
    hipLaunchKernelGGL(scan_sums_kernel, dim3(nblocks), dim3(kScanThreads), 0, st, in, n, w.block_sums, w.block_max, (int*)nullptr);
    hipLaunchKernelGGL(scan_apply_kernel, dim3(nblocks), dim3(kScanThreads), 0, st, in, n, w.block_sums, w.block_max,
                       nblocks, out, nodes, edge_counts, out_total, out_max, out_overflow, (const int*)nullptr, 0,
                       (int*)nullptr);
    return check_launch("neighbour scan");
}

// The graph truncated at `capacity` edges: row pointers and per-box counts above the capacity are lowered to it, so
// that every kernel that walks the edges through row_ptr stays inside edge arrays of that many entries.  stats[0]
// keeps the true count; bit 1 of stats[3] says that edges were dropped.
__global__ void __launch_bounds__(256) clamp_row_ptr_kernel(int* __restrict__ row_ptr, long n_ptr,
                                                            int* __restrict__ edge_counts, int batch, int capacity,
                                                            int* __restrict__ stats) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_ptr && row_ptr[i] > capacity) row_ptr[i] = capacity;
    if (i < batch && edge_counts[i] > capacity) edge_counts[i] = capacity;
    if (i == 0 && stats[0] > capacity) stats[3] |= 2;
}

int pairs_block_size(const Grid& g);
// workgroups that share the sort of one box: one per 1024 atoms (box_max has batch * nodes entries, so slabs <= nodes)
int sort_slabs(const Grid& g) {
    const int s = g.nodes / 1024;
    return s < 1 ? 1 : (s > kSortSlabsMax ? kSortSlabsMax : s);
}
// one workgroup per cell, laid out so that the kernels read the cell coordinates off the workgroup id
dim3 cell_grid(const Grid& g) { return dim3((unsigned)g.nz, (unsigned)g.ny, (unsigned)(g.nx * g.batch)); }
// Hit rows.  An entry is a box-local atom id: 16 bits when a box has at most 65536 atoms.  The host knows the mean
// density only, and a row that is too short costs a second sweep of the atom's window in the fill pass, so a row has
// kHitCapMax entries (enough for any density short of a dense liquid with a long cutoff: 512 bytes of address space
// per atom, of which a search touches what its neighbour counts need) whenever the workspace is as large as
// mg_neighbour_workspace_bytes says; a smaller workspace (the library's built-in one) gets the longest rows that
// fit, down to kHitCapMin entries.  Count, fill and cell-order calls derive the same layout from the same
// (batch, nodes, box, workspace size).
constexpr int kHitCapMax = 256, kHitCapMin = 32;
int hit_entry_bytes(const Grid& g) { return g.nodes <= 65536 ? 2 : 4; }

// Workspace layout for a buffer of `workspace_bytes` (0: the preferred size).  Returns false when not even the
// shortest rows fit; *needed is then the smallest size that works.
bool layout(const Grid& g, void* base, size_t workspace_bytes, Workspace* w, size_t* needed) {
    const long A = (long)g.batch * g.nodes, C = (long)g.batch * g.ncells;
    const int eb = hit_entry_bytes(g);
    int cap = kHitCapMax;
    if (workspace_bytes != 0 && A > 0) {
        const size_t fixed = carve(nullptr, A, C, 0, eb).bytes + 512;      // alignment of the base and of the rows
        const size_t room = workspace_bytes > fixed ? workspace_bytes - fixed : 0;
        long fit = (long)(room / ((size_t)eb * (size_t)A));
        fit &= ~7L;                                     // rows stay 16-byte aligned
        if (fit < kHitCapMin) {
            if (needed) *needed = carve(nullptr, A, C, kHitCapMin, eb).bytes + 256;
            return false;
        }
        cap = fit < kHitCapMax ? (int)fit : kHitCapMax;
    }
    *w = carve(base, A, C, cap, eb);
    if (workspace_bytes != 0 && w->bytes + 256 > workspace_bytes) {     // (A == 0: the fixed arrays alone)
        if (needed) *needed = w->bytes + 256;
        return false;
    }
    return true;
}

int pairs_block_size(const Grid& g) {
    // sparse boxes: one wave per cell and a tile of 256 candidates are plenty (10 % faster than four waves at 1.2
    // atoms per cell).  Only the mean is known here: 16384 atoms clumped in a ball inside a box of 8000 cells (2 per
    // cell on average, 22 where they are) overflow that tile and take 0.30 ms with one wave against 0.18 ms with four,
    // hence the low threshold.
    const double mean_occ = (double)g.nodes / (double)g.ncells;
    return mean_occ <= 2.0 ? 64 : 256;
}


// boxes small enough for box_search_kernel
bool whole_box_search(const Grid& g) { return g.nodes <= kBoxNodes && g.ncells <= kBoxCells; }
bool per_box_sort(const Grid& g) { return g.nodes <= kSortNodes && g.ncells <= kSortCells; }
// words of box_max that the search leaves
int box_max_entries(const Grid& g) { return whole_box_search(g) ? g.batch : per_box_sort(g) ? g.batch * sort_slabs(g) : 2; }

template <int kPer, typename HitT>
void launch_box_search(const float* x, const Grid& g, const Workspace& w, hipStream_t st) {
    // workgroups per box: one home cell per wave while the whole search stays within two workgroups per CU
    const int most = g.batch >= 512 ? 1 : 512 / g.batch;
    int parts = (g.ncells + kBoxWaves - 1) / kBoxWaves;
    parts = parts > most ? most : parts;
    hipLaunchKernelGGL((box_search_kernel<kPer, HitT>), dim3((unsigned)parts, (unsigned)g.batch), dim3(kBoxThreads), 0, st, x,
                       g, w);
}

// cell-ordered atoms, hit rows and degrees of every atom (batch * nodes > 0)
int enqueue_search(const float* x, const Grid& g, const Workspace& w0, hipStream_t st) {
    Workspace w = w0;
    const long A = (long)g.batch * g.nodes, C = (long)g.batch * g.ncells;
    if (whole_box_search(g)) {                     // (at most 2048 atoms per box: 16-bit hit rows)
        if (g.nodes <= kBoxThreads) launch_box_search<1, unsigned short>(x, g, w, st);
        else if (g.nodes <= 2 * kBoxThreads) launch_box_search<2, unsigned short>(x, g, w, st);
        else launch_box_search<4, unsigned short>(x, g, w, st);
        return check_launch("neighbour search");
    }
    const unsigned ablocks = (unsigned)ceil_div(A, 256);
    if (per_box_sort(g)) {
        hipLaunchKernelGGL(bin_kernel<false>, dim3(ablocks), dim3(256), 0, st, x, g, w);
        hipLaunchKernelGGL(sort_box_kernel, dim3((unsigned)sort_slabs(g), (unsigned)g.batch), dim3(kSortThreads), 0, st, g, w);
    } else {
        hipLaunchKernelGGL(zero3_kernel, dim3((unsigned)(ceil_div(C, 256) < 1024 ? ceil_div(C, 256) : 1024)), dim3(256),
                           0, st, w.box_max, 2L, (int*)nullptr, 0L, w.cell_count, C);
        hipLaunchKernelGGL(bin_kernel<true>, dim3(ablocks), dim3(256), 0, st, x, g, w);
        if (int s = run_scan(w.cell_count, C, w.cell_start, w, nullptr, w.box_max, nullptr, st)) return s;
        hipLaunchKernelGGL(place_kernel, dim3(ablocks), dim3(256), 0, st, g, w);
        hipLaunchKernelGGL(order_kernel, dim3(ablocks), dim3(256), 0, st, g, w);
    }
    const bool narrow = w.hit_bytes == 2;
    if (pairs_block_size(g) == 64) {
        if (narrow) hipLaunchKernelGGL((count_kernel<kCandCapSparse, unsigned short>), cell_grid(g), dim3(64), 0, st, g, w);
        else hipLaunchKernelGGL((count_kernel<kCandCapSparse, int>), cell_grid(g), dim3(64), 0, st, g, w);
    } else {
        if (narrow) hipLaunchKernelGGL((count_kernel<kCandCapDense, unsigned short>), cell_grid(g), dim3(256), 0, st, g, w);
        else hipLaunchKernelGGL((count_kernel<kCandCapDense, int>), cell_grid(g), dim3(256), 0, st, g, w);
    }
    return check_launch("neighbour search");
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_neighbour_ndiv(float cutoff, float box_x, float box_y, float box_z, int ndiv[3]) {
    ndiv[0] = (int)ceilf(box_x / cutoff);
    ndiv[1] = (int)ceilf(box_y / cutoff);
    ndiv[2] = (int)ceilf(box_z / cutoff);
    return MG_OK;
}

int mg_neighbour_workspace_bytes(int batch, int nodes, float cutoff, float box_x, float box_y, float box_z,
                                 size_t* bytes) {
    MG_REQUIRE(bytes != nullptr, "bytes is null");
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    Workspace w;
    layout(g, nullptr, 0, &w, nullptr);
    *bytes = w.bytes + 256;
    return MG_OK;
}

int mg_neighbour_count(const float* x, int batch, int nodes, float cutoff, float box_x, float box_y,
                       float box_z, void* workspace, size_t workspace_bytes, int* row_ptr,
                       int* edge_counts, int* stats, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    MG_REQUIRE(row_ptr && stats && workspace, "mg_neighbour_count: null pointer");
    MG_REQUIRE(batch == 0 || edge_counts, "mg_neighbour_count: edge_counts is null");
    const long A = (long)batch * nodes;
    void* base = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255));
    Workspace w;
    size_t needed = 0;
    if (workspace_bytes == 0 || !layout(g, base, workspace_bytes, &w, &needed))
        return fail(MG_ERR_WORKSPACE, "mg_neighbour_count: workspace has %zu bytes, at least %zu needed", workspace_bytes,
                    needed);
    hipStream_t st = (hipStream_t)stream;
    if (A == 0) {
        hipLaunchKernelGGL(zero3_kernel, dim3(1), dim3(256), 0, st, stats, 4L, row_ptr, 1L, edge_counts, (long)batch);
        return check_launch("mg_neighbour_count");
    }
    MG_REQUIRE(x != nullptr, "mg_neighbour_count: x is null");
    const int deg_tiles = (int)ceil_div(A + 1, kScanTile);
    if (int s = enqueue_search(x, g, w, st)) return s;
    hipLaunchKernelGGL(scan_sums_kernel, dim3((unsigned)deg_tiles), dim3(kScanThreads), 0, st, (const int*)w.degree, A,
                       w.deg_sums, w.deg_max, (int*)nullptr);
    hipLaunchKernelGGL(scan_apply_kernel, dim3((unsigned)deg_tiles), dim3(kScanThreads), 0, st, (const int*)w.degree, A,
                       (const int*)w.deg_sums, (const int*)w.deg_max, deg_tiles, row_ptr, nodes, edge_counts, stats + 0,
                       stats + 2, stats + 3, (const int*)w.box_max, box_max_entries(g), stats + 1);
    return check_launch("mg_neighbour_count");
}

int mg_neighbour_fill(const void* workspace, size_t workspace_bytes, int batch, int nodes, float cutoff,
                      float box_x, float box_y, float box_z, const int* row_ptr, int n_edges, int* src,
                      int* dst, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    MG_REQUIRE(n_edges >= 0, "mg_neighbour_fill: negative n_edges");
    const long A = (long)batch * nodes;
    if (A == 0 || n_edges == 0) return MG_OK;
    MG_REQUIRE(workspace && row_ptr && src && dst, "mg_neighbour_fill: null pointer");
    void* base = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255));
    Workspace w;
    size_t needed = 0;
    if (workspace_bytes == 0 || !layout(g, base, workspace_bytes, &w, &needed))
        return fail(MG_ERR_WORKSPACE, "mg_neighbour_fill: workspace has %zu bytes, at least %zu needed", workspace_bytes,
                    needed);
    const EdgeOut out{src, dst, nullptr, nullptr, nullptr, nullptr};
    if (w.hit_bytes == 2)
        hipLaunchKernelGGL(fill_kernel<unsigned short>, dim3((unsigned)ceil_div(A, kFillRows)), dim3(256), 0,
                           (hipStream_t)stream, g, w, row_ptr, out, n_edges);
    else
        hipLaunchKernelGGL(fill_kernel<int>, dim3((unsigned)ceil_div(A, kFillRows)), dim3(256), 0, (hipStream_t)stream, g,
                           w, row_ptr, out, n_edges);
    return check_launch("mg_neighbour_fill");
}

int mg_graph_search(const float* x, int batch, int nodes, float cutoff, float box_x, float box_y, float box_z,
                    void* workspace, size_t workspace_bytes, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    if ((long)batch * nodes == 0) return MG_OK;
    MG_REQUIRE(x && workspace, "mg_graph_search: null pointer");
    void* base = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255));
    Workspace w;
    size_t needed = 0;
    if (workspace_bytes == 0 || !layout(g, base, workspace_bytes, &w, &needed))
        return fail(MG_ERR_WORKSPACE, "mg_graph_search: workspace has %zu bytes, at least %zu needed", workspace_bytes, needed);
    hipStream_t st = (hipStream_t)stream;
    if (int s = enqueue_search(x, g, w, st)) return s;
    const long A = (long)batch * nodes;
    if (A > kDirectRows)
        hipLaunchKernelGGL(scan_sums_kernel, dim3((unsigned)ceil_div(A + 1, kScanTile)), dim3(kScanThreads), 0, st,
                           (const int*)w.degree, A, w.deg_sums, w.deg_max, w.degree);
    return check_launch("mg_graph_search");
}

int mg_graph_fill(const float* x, const void* workspace, size_t workspace_bytes, int batch, int nodes, float cutoff,
                  float box_x, float box_y, float box_z, int* row_ptr, int* edge_counts, int* stats, int capacity, int* src,
                  int* dst, int64_t* src64, int64_t* dst64, float* r_ij, int* order, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    MG_REQUIRE(capacity >= 0, "mg_graph_fill: negative capacity");
    MG_REQUIRE(row_ptr && stats, "mg_graph_fill: null pointer");
    MG_REQUIRE((src64 == nullptr) == (dst64 == nullptr), "mg_graph_fill: src64 and dst64 go together");
    const long A = (long)batch * nodes;
    hipStream_t st = (hipStream_t)stream;
    if (A == 0) {
        hipLaunchKernelGGL(zero3_kernel, dim3(1), dim3(256), 0, st, stats, 4L, row_ptr, 1L, edge_counts, (long)batch);
        return check_launch("mg_graph_fill");
    }
    MG_REQUIRE(workspace && edge_counts && (capacity == 0 || (src && dst)) && (r_ij == nullptr || x),
               "mg_graph_fill: null pointer");
    void* base = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255));
    Workspace w;
    size_t needed = 0;
    if (workspace_bytes == 0 || !layout(g, base, workspace_bytes, &w, &needed))
        return fail(MG_ERR_WORKSPACE, "mg_graph_fill: workspace has %zu bytes, at least %zu needed", workspace_bytes, needed);
    const EdgeOut out{src, dst, src64, dst64, r_ij, r_ij ? x : nullptr};
    const int tiled = A > kDirectRows ? 1 : 0;
    // Few rows: one to a wave, so that a small graph still spreads over the chip (337 atoms: 4.3 us, 9 with eight); otherwise eight, whose
    // loads are in flight together (131 072 rows of 52 edges: one 107, four 88, eight 83 us)
    auto launch = [&](auto hit, auto rw) {
        hipLaunchKernelGGL((graph_fill_kernel<decltype(hit), decltype(rw)::value>), dim3((unsigned)ceil_div(A, 4 * decltype(rw)::value)),
                           dim3(256), 0, st, g, w, tiled, box_max_entries(g), row_ptr, edge_counts, stats, capacity, out, order);
    };
    // Beyond 16 384 rows (us of this kernel, a wave to a row / dealt out, and of the kernel before both, whose rows were dealt out, in
    // brackets).  Rows that fill less than half of a wave's lanes are dealt out: 4 edges a row, 20 000 rows 9.2 / 6.5, 131 072 38 / 15;
    // 26 edges, 32 768 rows 14.9 / 14.2, 131 072 49 / 35 (39).  Longer rows take a wave each up to 32 768 (20 000 of 52 16.3 / 22.4,
    // 32 768 22 / 24), and are dealt out beyond (65 536 of 40 32 / 28 (30), of 80 58 / 47 (49); 98 304 of 52 60 / 55 (58)), up to where
    // the edges outgrow the 256 MB of the memory-side cache: there whole waves write fewer pieces, if a row is one piece (131 072 of
    // 52 98 / 107 (110), of 80 195 / 186 (189); 262 144 of 40 198 / 206 (209), of 80 409 / 409).
    // 4097 to 16 384 rows take a wave each (4200 of 16 12.3 (14.4), of 52 13.3 (21.7); 16 384 24.1 (26.5) and 26.1 (34); of 4 edges,
    // where the sums over the rows before are all there is, 12.4 (11.0) and 24.0 (22.2)).
    const double mean = 4.18879 * cutoff * cutoff * cutoff * nodes / ((double)box_x * box_y * box_z);
    const bool wave_rows = mean > 32 && (A <= 32768 || (mean <= kWave && A * mean >= 6.0e6));
    const bool dealt = tiled && !wave_rows;
    auto with_rows = [&](auto hit) {
        if (A <= 4096) launch(hit, std::integral_constant<int, 1>{});
        else if (!dealt) launch(hit, std::integral_constant<int, 8>{});
        else
            hipLaunchKernelGGL(graph_fill_dealt_kernel<decltype(hit)>, dim3((unsigned)ceil_div(A, kFillRows)), dim3(256), 0, st, g, w,
                               box_max_entries(g), row_ptr, edge_counts, stats, capacity, out, order);
    };
    if (w.hit_bytes == 2) with_rows((unsigned short)0);
    else with_rows((int)0);
    return check_launch("mg_graph_fill");
}

int mg_neighbour_edges(const float* x, int batch, int nodes, float cutoff, float box_x, float box_y, float box_z,
                       void* workspace, size_t workspace_bytes, int* row_ptr, int* edge_counts, int* stats,
                       int capacity, int* src, int* dst, mg_stream_t stream) {
    MG_REQUIRE(capacity >= 0, "mg_neighbour_edges: negative capacity");
    MG_REQUIRE(capacity == 0 || (src && dst), "mg_neighbour_edges: src / dst is null");
    if (int s = mg_neighbour_count(x, batch, nodes, cutoff, box_x, box_y, box_z, workspace, workspace_bytes, row_ptr,
                                   edge_counts, stats, stream))
        return s;
    if (int s = mg_neighbour_fill(workspace, workspace_bytes, batch, nodes, cutoff, box_x, box_y, box_z, row_ptr,
                                  capacity, src, dst, stream))
        return s;
    const long n_ptr = (long)batch * nodes + 1;
    if (n_ptr == 1) return MG_OK;
    // after the fill pass (which places edges by the exact row_ptr): the caller's view is the graph cut at capacity
    hipLaunchKernelGGL(clamp_row_ptr_kernel, dim3((unsigned)ceil_div(n_ptr, 256)), dim3(256), 0, (hipStream_t)stream,
                       row_ptr, n_ptr, edge_counts, batch, capacity, stats);
    return check_launch("mg_neighbour_edges");
}

int mg_neighbour_edges_static(const float* x, int batch, int nodes, float cutoff, float box_x, float box_y,
                              float box_z, int* row_ptr, int* edge_counts, int* stats, int capacity, int* src,
                              int* dst, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    Workspace probe;
    size_t need = 0;
    if (!layout(g, nullptr, kScratchBytes, &probe, &need))
        return fail(MG_ERR_WORKSPACE,
                    "mg_neighbour_edges_static: this search needs at least %zu bytes of workspace (%zu per atom), the "
                    "built-in one holds %zu; use mg_neighbour_edges with a workspace of your own",
                    need, need / (size_t)((long)batch * nodes > 0 ? (long)batch * nodes : 1), kScratchBytes);
    void* ws = nullptr;
    if (int s = scratch_of_current_device(&ws)) return s;
    // every array of the workspace that must start at zero (the cell histogram) is cleared by a kernel inside
    // mg_neighbour_count; everything else is written before it is read, so what the previous call left is harmless
    return mg_neighbour_edges(x, batch, nodes, cutoff, box_x, box_y, box_z, ws, kScratchBytes, row_ptr, edge_counts,
                              stats, capacity, src, dst, stream);
}

int mg_neighbour_cell_order(const void* workspace, size_t workspace_bytes, int batch, int nodes, float cutoff,
                            float box_x, float box_y, float box_z, int* order, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    const long A = (long)batch * nodes;
    if (A == 0) return MG_OK;
    MG_REQUIRE(workspace && order, "mg_neighbour_cell_order: null pointer");
    void* base = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~uintptr_t(255));
    Workspace w;
    size_t needed = 0;
    if (workspace_bytes == 0 || !layout(g, base, workspace_bytes, &w, &needed))
        return fail(MG_ERR_WORKSPACE, "mg_neighbour_cell_order: workspace has %zu bytes, at least %zu needed",
                    workspace_bytes, needed);
    hipLaunchKernelGGL(cell_order_kernel, dim3((unsigned)ceil_div(A, 256)), dim3(256), 0, (hipStream_t)stream, g, w,
                       order);
    return check_launch("mg_neighbour_cell_order");
}

int mg_neighbour_wrap_cells(const float* x, int batch, int nodes, float cutoff, float box_x, float box_y,
                            float box_z, float* wrapped, int* cell, mg_stream_t stream) {
    Grid g;
    if (int s = make_grid(cutoff, box_x, box_y, box_z, batch, nodes, &g)) return s;
    const long A = (long)batch * nodes;
    if (A == 0) return MG_OK;
    MG_REQUIRE(x && wrapped && cell, "mg_neighbour_wrap_cells: null pointer");
    hipLaunchKernelGGL(wrap_cells_kernel, dim3((unsigned)ceil_div(A, 256)), dim3(256), 0, (hipStream_t)stream, x, g,
                       wrapped, cell);
    return check_launch("mg_neighbour_wrap_cells");
}

int mg_neighbour_pad(const int* row_ptr, const int* dst, int batch, int nodes, int neighboursmax,
                     int* neighbours, int* counts, mg_stream_t stream) {
    MG_REQUIRE(batch >= 0 && nodes >= 0 && neighboursmax >= 0, "mg_neighbour_pad: negative size");
    const long A = (long)batch * nodes;
    if (A == 0) return MG_OK;
    MG_REQUIRE(row_ptr && counts && (neighboursmax == 0 || neighbours), "mg_neighbour_pad: null pointer");
    hipLaunchKernelGGL(pad_kernel, dim3((unsigned)ceil_div(A * kWave, 256)), dim3(256), 0, (hipStream_t)stream,
                       row_ptr, dst, A, nodes, neighboursmax, neighbours, counts);
    return check_launch("mg_neighbour_pad");
}

int mg_padded_edges_read(const int* counts, const int* neighbours, const float* x, int batch, int nodes,
                         int neighboursmax, int chan, float* edge_data, mg_stream_t stream) {
    MG_REQUIRE(batch >= 0 && nodes >= 0 && neighboursmax >= 0 && chan >= 0, "mg_padded_edges_read: negative size");
    const long A = (long)batch * nodes, total = A * neighboursmax * chan;
    if (total == 0) return MG_OK;
    MG_REQUIRE(counts && neighbours && x && edge_data, "mg_padded_edges_read: null pointer");
    const long blocks = ceil_div(total, 256);
    hipLaunchKernelGGL(padded_read_kernel, dim3((unsigned)(blocks < 65536 * 16 ? blocks : 65536 * 16)), dim3(256), 0,
                       (hipStream_t)stream, counts, neighbours, x, A, nodes, neighboursmax, chan, edge_data);
    return check_launch("mg_padded_edges_read");
}

int mg_padded_edges_reduce(const int* counts, const float* edge_data, int batch, int nodes, int neighboursmax,
                           int chan, float* out, mg_stream_t stream) {
    MG_REQUIRE(batch >= 0 && nodes >= 0 && neighboursmax >= 0 && chan >= 0, "mg_padded_edges_reduce: negative size");
    const long A = (long)batch * nodes, total = A * chan;
    if (total == 0) return MG_OK;
    MG_REQUIRE(counts && out && (neighboursmax == 0 || edge_data), "mg_padded_edges_reduce: null pointer");
    const long blocks = ceil_div(total, 256);
    hipLaunchKernelGGL(padded_reduce_kernel, dim3((unsigned)(blocks < 65536 * 16 ? blocks : 65536 * 16)), dim3(256),
                       0, (hipStream_t)stream, counts, edge_data, A, neighboursmax, chan, out);
    return check_launch("mg_padded_edges_reduce");
}

int mg_edge_vectors(const float* x, const int* src, const int* dst, long n_edges, float box_x, float box_y,
                    float box_z, float* r_ij, int8_t* shift, mg_stream_t stream) {
    MG_REQUIRE(n_edges >= 0, "mg_edge_vectors: negative n_edges");
    if (n_edges == 0) return MG_OK;
    MG_REQUIRE(x && src && dst && r_ij, "mg_edge_vectors: null pointer");
    MG_REQUIRE(box_x > 0.f && box_y > 0.f && box_z > 0.f, "mg_edge_vectors: box must be positive");
    hipLaunchKernelGGL(edge_vectors_kernel, dim3((unsigned)ceil_div(n_edges, 256)), dim3(256), 0,
                       (hipStream_t)stream, x, src, dst, n_edges, box_x, box_y, box_z, r_ij, shift);
    return check_launch("mg_edge_vectors");
}

}  // extern "C"
