// grid.hip -- what a catalogue goes through before its pairs are counted: the pass that takes it over
// (copy, bounding box, weight statistics) and the GPU cell grid (counting sort of points by cell, cell
// start offsets).  Replaces the kd-tree build (kdtree2.F90:611-1012) and its r-ball queries: a pair
// kernel reads each neighbour cell row as one contiguous range of the sorted points.
#include <algorithm>

#include "gs_device.h"
#include "gs_kernels.h"

namespace gs {

using namespace dev;

// ---------------------------------------------------------------- catalogue
// One pass over a catalogue handed over: copies it (where src and dst differ) and reduces its bounding box,
// the largest data and random weight and the first invalid weight.  The last block to finish reduces the
// blocks' partials, so that one launch and one wait give the host everything (with k_wsum, where there
// are weights); before, the copies, the check, the sums and the bounding box were seven launches and three
// waits.  Bound by memory where it is large (each coordinate and weight is read and written once: 600k points 32 us),
// by the chain load, reduction, release, reduction where it is small (60k points 11 us; with one load in flight, a
// reduction per quantity and a release by every wave 19).
// The thread count is a multiple of 3, so that every thread's coordinates share one axis.
constexpr int kIngestThreads = 192;

// the maxima of v over the block, in every thread of it; all nine at once, so that their shuffles overlap
__device__ __forceinline__ void block_reduce_max(double (&v)[9], double (*red)[9])
{
    for (int off = 32; off > 0; off >>= 1)
        for (int q = 0; q < 9; ++q) v[q] = fmax(v[q], __shfl_down(v[q], off, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 9; ++q) red[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
    for (int q = 0; q < 9; ++q) {
        v[q] = red[0][q];
        for (int k = 1; k < kIngestThreads / 64; ++k) v[q] = fmax(v[q], red[k][q]);
    }
}

__global__ __launch_bounds__(kIngestThreads) void k_ingest(const double* __restrict__ xyz, const double* __restrict__ w,
                                                           const int32_t* __restrict__ buf, int64_t n, int64_t n_data,
                                                           double* xyz_out, double* w_out, int32_t* buf_out,
                                                           IngestScratch* sc, CatalogueStats* out)
{
    __shared__ double red[kIngestThreads / 64][9];
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, step = gridDim.x * (int64_t)blockDim.x;
    const int axis = (int)(t % 3);
    double mn = 1e308, mx = -1e308;
    // four loads in flight: a store between them could change what they read, for all the compiler knows
    for (int64_t i = t; i < 3 * n; i += 4 * step) {
        double v[4];
        for (int k = 0; k < 4; ++k) v[k] = i + k * step < 3 * n ? xyz[i + k * step] : 0.0;
        for (int k = 0; k < 4; ++k)
            if (i + k * step < 3 * n) {
                if (xyz_out != xyz) xyz_out[i + k * step] = v[k];
                mn = fmin(mn, v[k]);
                mx = fmax(mx, v[k]);
            }
    }
    double wm[2] = {0.0, 0.0};
    unsigned long long bad = ~0ull;
    if (w)
        for (int64_t i = t; i < n; i += 4 * step) {
            double v[4];
            for (int k = 0; k < 4; ++k) v[k] = i + k * step < n ? w[i + k * step] : 0.0;
            for (int k = 0; k < 4; ++k) {
                const int64_t at = i + k * step;
                if (at >= n) break;
                if (w_out != w) w_out[at] = v[k];
                if (!(v[k] >= 0.0) || !isfinite(v[k])) bad = bad < (unsigned long long)at ? bad : (unsigned long long)at;
                else if (at < n_data) wm[0] = fmax(wm[0], v[k]);
                else wm[1] = fmax(wm[1], v[k]);
            }
        }
    if (buf && buf_out != buf)
        for (int64_t i = t; i < n; i += step) buf_out[i] = buf[i];

    // lowest values negated; the index of a bad weight as a double: exact below 2^53
    double v[9];
    for (int k = 0; k < 3; ++k) {
        v[k] = axis == k ? -mn : -1e308;
        v[3 + k] = axis == k ? mx : -1e308;
    }
    v[6] = wm[0];
    v[7] = wm[1];
    v[8] = bad == ~0ull ? -1e308 : -(double)bad;
    block_reduce_max(v, red);
    if (threadIdx.x == 0)
        for (int q = 0; q < 9; ++q) sc[blockIdx.x].v[q] = v[q];
    if (!last_block(&out->ticket)) return;
    for (int q = 0; q < 9; ++q) v[q] = -1e308;
    for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x) {
        double x[9];
        for (int q = 0; q < 9; ++q) x[q] = load_agent(&sc[b].v[q]);
        for (int q = 0; q < 9; ++q) v[q] = fmax(v[q], x[q]);
    }
    block_reduce_max(v, red);
    if (threadIdx.x == 0)
        for (int q = 0; q < 9; ++q) out->v[q] = q < 3 || q == 8 ? -v[q] : v[q];
    // without weights there is no k_wsum to hand the statistics to the host
    if (!w && threadIdx.x == 0)
        for (int q = 0; q < 9; ++q) out->host->v[q] = out->v[q];
}

// Exact fixed-point sums of the data and the random weights (wsum_fixed at the scale of the largest weight),
// then the statistics to the host.
__global__ __launch_bounds__(256) void k_wsum(const double* __restrict__ w, int64_t n, int64_t n_data,
                                              IngestScratch* sc, CatalogueStats* out)
{
    __shared__ unsigned long long red[4][4];
    const int k = wsum_scale(fmax(out->v[6], out->v[7]));
    unsigned long long a[4] = {0, 0, 0, 0};     // data lo, hi, randoms lo, hi
    if (out->v[8] >= 1e308)                     // no invalid weight
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
            uint64_t lo, hi;
            wsum_fixed(w[i], k, lo, hi);
            const int o = i < n_data ? 0 : 2;
            add128(a[o], a[o + 1], lo, hi);
        }
    auto block_sum = [&]() {                    // the block's sum of a, in thread 0
        for (int off = 32; off > 0; off >>= 1)
            for (int q = 0; q < 4; q += 2) {
                const unsigned long long l = __shfl_down(a[q], off, 64), h = __shfl_down(a[q + 1], off, 64);
                add128(a[q], a[q + 1], l, h);
            }
        __syncthreads();
        if ((threadIdx.x & 63) == 0)
            for (int q = 0; q < 4; ++q) red[threadIdx.x >> 6][q] = a[q];
        __syncthreads();
        if (threadIdx.x == 0)
            for (int v = 1; v < 4; ++v)
                for (int q = 0; q < 4; q += 2) add128(a[q], a[q + 1], red[v][q], red[v][q + 1]);
    };
    block_sum();
    if (threadIdx.x == 0)
        for (int q = 0; q < 4; ++q) sc[blockIdx.x].s[q] = a[q];
    if (!last_block(&out->ticket)) return;
    for (int q = 0; q < 4; ++q) a[q] = 0;
    for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x)
        for (int q = 0; q < 4; q += 2) add128(a[q], a[q + 1], load_agent(&sc[b].s[q]), load_agent(&sc[b].s[q + 1]));
    block_sum();
    if (threadIdx.x == 0) {
        for (int q = 0; q < 4; ++q) out->host->s[q] = a[q];
        for (int q = 0; q < 9; ++q) out->host->v[q] = out->v[q];
    }
}

hipError_t launch_ingest(const double* xyz, const double* w, const int32_t* buf, int64_t n, int64_t n_data,
                         double* xyz_out, double* w_out, int32_t* buf_out, IngestScratch* scratch, CatalogueStats* stats,
                         hipStream_t st)
{
    const int nblk = (int)std::min<int64_t>(std::max<int64_t>((3 * n + 12 * kIngestThreads - 1) / (12 * kIngestThreads), 1),
                                            kIngestBlocks);
    hipLaunchKernelGGL(k_ingest, dim3(nblk), dim3(kIngestThreads), 0, st, xyz, w, buf, n, n_data, xyz_out, w_out, buf_out,
                       scratch, stats);
    if (w) {
        const int wblk = (int)std::min<int64_t>(std::max<int64_t>((n + 1023) / 1024, 1), kIngestBlocks);
        hipLaunchKernelGGL(k_wsum, dim3(wblk), dim3(256), 0, st, w_out, n, n_data, scratch, stats);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- exclusive scan
// Three-phase scan of int32 counts: each block scans 1024 entries in LDS and
// emits its total; the totals are scanned recursively; offsets are added back.
constexpr int kScanBlock = 1024;

__global__ __launch_bounds__(256) void k_scan_block(const int32_t* __restrict__ in, int64_t n,
                                                    int32_t* __restrict__ out, int32_t* __restrict__ sums)
{
    __shared__ int32_t s[kScanBlock];
    __shared__ int32_t wsum[4];
    const int64_t base = (int64_t)blockIdx.x * kScanBlock;
    const int t = threadIdx.x;
    int v[4];
    int run = 0;
    for (int k = 0; k < 4; ++k) {
        int64_t i = base + t * 4 + k;
        v[k] = i < n ? in[i] : 0;
        run += v[k];
    }
    // inclusive scan of per-thread totals across the block (wave64 shuffles, then across 4 waves)
    int x = run;
    const int lane = t & 63, w = t >> 6;
    for (int off = 1; off < 64; off <<= 1) {
        int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int wpre = 0;
    for (int k = 0; k < w; ++k) wpre += wsum[k];
    int excl = wpre + x - run;
    for (int k = 0; k < 4; ++k) {
        s[t * 4 + k] = excl;
        excl += v[k];
    }
    __syncthreads();
    for (int k = 0; k < 4; ++k) {
        int64_t i = base + t * 4 + k;
        if (i < n) out[i] = s[t * 4 + k];
    }
    if (t == 255) sums[blockIdx.x] = excl;
}

__global__ __launch_bounds__(256) void k_scan_add(int32_t* __restrict__ out, int64_t n, const int32_t* __restrict__ offs)
{
    const int64_t base = (int64_t)blockIdx.x * kScanBlock;
    const int32_t o = offs[blockIdx.x];
    for (int k = threadIdx.x; k < kScanBlock; k += blockDim.x) {
        int64_t i = base + k;
        if (i < n) out[i] += o;
    }
}

hipError_t exclusive_scan(const int32_t* in, int32_t* out, int64_t n, int32_t* scratch, hipStream_t st)
{
    // scratch must hold scan_scratch_size(n) int32
    if (n <= 0) return hipSuccess;
    int64_t nb = (n + kScanBlock - 1) / kScanBlock;
    int32_t* sums = scratch;
    int32_t* sums_scanned = scratch + nb;
    hipLaunchKernelGGL(k_scan_block, dim3((unsigned)nb), dim3(256), 0, st, in, n, out, sums);
    if (nb > 1) {
        hipError_t e = exclusive_scan(sums, sums_scanned, nb, scratch + 2 * nb, st);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_scan_add, dim3((unsigned)nb), dim3(256), 0, st, out, n, sums_scanned);
    }
    return hipGetLastError();
}

int64_t scan_scratch_size(int64_t n)
{
    int64_t tot = 0;
    while (n > 1) {
        int64_t nb = (n + kScanBlock - 1) / kScanBlock;
        tot += 2 * nb;
        n = nb;
    }
    return tot + 2;
}

// ---------------------------------------------------------------- cells
// Counting sort of the points into cells, a cell's data points before its randoms (consecutive neighbours
// then mostly share a class), in three launches: the counts of data and randoms per cell, each point
// keeping its rank in its count; the exclusive scan of the counts, by blocks, with the blocks' offsets
// scanned by the last block; the scatter, which adds the offsets where it needs them and writes the final
// cell starts beside.  The order inside a count follows the atomics' order; every count and fixed-point sum
// computed from the sorted arrays is independent of it.  One grid, or one per region of a batch.
// Scan: 1,000,001 counts 13 us (with scalar loads, blocks of 2048 and a release by every wave 70).
constexpr int kCellScan = 4096;     // counts per block of the scan, 8 per thread

__device__ __forceinline__ int cell_coord(double v, double lo, double inv_h, int dim)
{
    int c = (int)floor((v - lo) * inv_h);
    return c < 0 ? 0 : (c >= dim ? dim - 1 : c);
}

__device__ __forceinline__ int region_of(const int32_t* off, int nreg, int64_t i)
{
    int lo = 0, hi = nreg - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
}

struct PointCell {
    int cx, row, cell;      // x cell and x-row (over all regions), cell
    bool random;
};

__device__ __forceinline__ PointCell point_cell(const GridArgs& a, int64_t i)
{
    double lo[3] = {a.g.lo[0], a.g.lo[1], a.g.lo[2]};
    int nx = a.g.dim[0], ny = a.g.dim[1], nz = a.g.dim[2], cell0 = 0, row0 = 0;
    int64_t p0 = 0, nd = a.n_data;
    if (a.nreg > 0) {
        const RegionDesc& R = a.regions[region_of(a.off, a.nreg, i)];
        for (int k = 0; k < 3; ++k) lo[k] = R.lo[k];
        nx = R.dim[0]; ny = R.dim[1]; nz = R.dim[2];
        cell0 = R.cell_base;
        row0 = R.row_base;
        p0 = R.pt_base;
        nd = R.n_data;
    }
    const double inv_h = 1.0 / a.g.h, inv_hx = 1.0 / a.g.hx;
    const double x = a.xyz[3 * i + 0], y = a.xyz[3 * i + 1], z = a.xyz[3 * i + 2];
    PointCell c;
    if (x != x || y != y || z != z) {
        // A point that is not a number has no pairs.  It goes behind all cells, to an x-row of its own, so that no
        // chunk of points has its coordinates relative to it.  (A single grid: regions have no such points.)
        c.cx = 0;
        c.row = ny * nz;
        c.cell = (int)a.ncell;
        c.random = false;
        return c;
    }
    c.cx = cell_coord(x, lo[0], inv_hx, nx);
    const int cy = cell_coord(y, lo[1], inv_h, ny);
    const int cz = cell_coord(z, lo[2], inv_h, nz);
    const int row = cz * ny + cy;
    c.row = row0 + row;
    c.cell = cell0 + row * nx + c.cx;
    c.random = i - p0 >= nd;
    return c;
}

__global__ __launch_bounds__(256) void k_cell_rank(GridArgs a)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * blockDim.x) {
        const PointCell c = point_cell(a, i);
        a.rank[i] = atomicAdd(&a.count[2 * (int64_t)c.cell + (c.random ? 1 : 0)], 1);
    }
}

__global__ __launch_bounds__(kCellScan / 8) void k_cell_scan(int32_t* __restrict__ v, int64_t n, int32_t* __restrict__ boff,
                                                   unsigned* ticket)
{
    constexpr int kThreads = kCellScan / 8, kWaves = kThreads / 64;
    __shared__ int32_t wsum[kWaves];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    // exclusive prefix of x over the block's threads; *total: the block's sum
    auto block_scan = [&](int x, int* total) {
        int inc = x;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(inc, off, 64);
            if (lane >= off) inc += y;
        }
        __syncthreads();
        if (lane == 63) wsum[wv] = inc;
        __syncthreads();
        int pre = 0, all = 0;
        for (int k = 0; k < kWaves; ++k) {
            if (k < wv) pre += wsum[k];
            all += wsum[k];
        }
        *total = all;
        return pre + inc - x;
    };
    const int64_t base = (int64_t)blockIdx.x * kCellScan + threadIdx.x * 8;
    int x[8] = {0, 0, 0, 0, 0, 0, 0, 0}, sum = 0, total;
    const bool whole = base + 8 <= n;       // a thread's 8 counts in two 16-byte accesses
    if (whole) {
        *(int4*)x = *(const int4*)(v + base);
        *(int4*)(x + 4) = *(const int4*)(v + base + 4);
    } else {
        for (int k = 0; k < 8; ++k)
            if (base + k < n) x[k] = v[base + k];
    }
    for (int k = 0; k < 8; ++k) sum += x[k];
    int run = block_scan(sum, &total);
    for (int k = 0; k < 8; ++k) {
        const int t = x[k];
        x[k] = run;
        run += t;
    }
    if (whole) {
        *(int4*)(v + base) = *(const int4*)x;
        *(int4*)(v + base + 4) = *(const int4*)(x + 4);
    } else {
        for (int k = 0; k < 8; ++k)
            if (base + k < n) v[base + k] = x[k];
    }
    if (threadIdx.x == 0) __hip_atomic_store(&boff[blockIdx.x], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!last_block(ticket)) return;
    int carry = 0;
    for (int b0 = 0; b0 < (int)gridDim.x; b0 += kThreads) {
        const int b = b0 + threadIdx.x;
        const int t = b < (int)gridDim.x ? load_agent(&boff[b]) : 0;
        const int e = block_scan(t, &total);
        if (b < (int)gridDim.x) boff[b] = carry + e;
        carry += total;
    }
}

__global__ __launch_bounds__(256) void k_cell_scatter(GridArgs a)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, step = gridDim.x * (int64_t)blockDim.x;
    auto start = [&](int64_t k) { return a.count[k] + a.boff[k / kCellScan]; };
    for (int64_t i = t; i < a.n; i += step) {
        const PointCell c = point_cell(a, i);
        const int pos = start(2 * (int64_t)c.cell + (c.random ? 1 : 0)) + a.rank[i];
        a.pw[pos] = make_double4(a.xyz[3 * i], a.xyz[3 * i + 1], a.xyz[3 * i + 2], a.w ? a.w[i] : 1.0);
        a.cell[pos] = make_int2(c.cx, c.row);
        a.flags[pos] = (c.random ? 1u : 0u) | ((a.buf && a.buf[i] == 1) ? 2u : 0u);
        a.orig[pos] = (int32_t)i;
    }
    for (int64_t c = t; c <= a.ncell; c += step) a.cell_start[c] = start(2 * c);
}

int64_t cell_scan_blocks(int64_t ncell) { return (2 * ncell + 1 + kCellScan - 1) / kCellScan; }

static int blocks_for(int64_t n)
{
    int64_t b = (n + 255) / 256;
    if (b > 65535) b = 65535;
    return (int)(b < 1 ? 1 : b);
}

hipError_t launch_cell_sort(const GridArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL(k_cell_rank, dim3(blocks_for(a.n)), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_cell_scan, dim3((unsigned)cell_scan_blocks(a.ncell)), dim3(kCellScan / 8), 0, st, a.count, 2 * a.ncell + 1,
                       a.boff, a.ticket);
    hipLaunchKernelGGL(k_cell_scatter, dim3(blocks_for(std::max<int64_t>(a.n, a.ncell + 1))), dim3(256), 0, st, a);
    return hipGetLastError();
}

// Work chunks of the full-stencil adjoint kernel: up to `group` consecutive points of one x-row of
// cells (fixed cy, cz).  nch[r] = chunks of row r; nch[nrow] = 0.
__global__ __launch_bounds__(256) void k_row_chunks(const int32_t* __restrict__ start, int nx, int nrow, int group,
                                                    int32_t* __restrict__ nch)
{
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r <= nrow; r += gridDim.x * blockDim.x) {
        int v = 0;
        if (r < nrow) v = (start[(r + 1) * nx] - start[r * nx] + group - 1) / group;
        nch[r] = v;
    }
}

hipError_t launch_row_chunks(const int32_t* start, int nx, int nrow, int group, int32_t* nch, hipStream_t st)
{
    hipLaunchKernelGGL(k_row_chunks, dim3(blocks_for(nrow + 1)), dim3(256), 0, st, start, nx, nrow, group, nch);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* __restrict__ p, int64_t n, uint32_t v)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

hipError_t launch_fill_u32(void* p, int64_t n, uint32_t v, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_u32, dim3(std::min(blocks_for(n), 2048)), dim3(256), 0, st, (uint32_t*)p, n, v);
    return hipGetLastError();
}

}  // namespace gs
