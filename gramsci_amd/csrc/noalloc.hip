// noalloc.hip -- gs_count_2pcf_noalloc: the 2PCF count of a catalogue already in
// device memory, with every device buffer it needs (the sorted copy of the
// catalogue, the cell grid, scan scratch, kernel parameters, histogram
// accumulators, work counters, reduction partials) carved out of one
// file-scope device array.  The call allocates no device memory, for callers
// that cannot allocate (code under HIP graph capture, serving loops, harnesses
// that forbid hipMalloc).  The kernels are those of gs_count_2pcf.
//
// Limits: at most kNoAllocMaxPoints points and kNoAllocMaxCells grid cells
// (the cell edge is widened until the grid fits).  Each GPU that runs the
// library holds the array (about 43 MB) until the process ends.  Every call on
// a GPU uses that GPU's one array: calls that overlap on one GPU race.
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "gs_api_internal.h"
#include "gs_kernels.h"

namespace gs {
namespace {

constexpr int64_t kNoAllocMaxPoints = (int64_t)1 << 19;
constexpr int64_t kNoAllocMaxCells = (int64_t)1 << 20;
constexpr int64_t kScanBlocks = 1040;              // >= cell_scan_blocks(kNoAllocMaxCells)
constexpr int64_t kMaxHist = 3 * (int64_t)kMaxBins * kMaxBins;   // histogram entries [3][nb][nm]

constexpr size_t al(size_t b) { return (b + 255) / 256 * 256; }

// byte offsets of the parts of the array
constexpr size_t kOffPw = 0;
constexpr size_t kOffCell = kOffPw + al(kNoAllocMaxPoints * sizeof(double4));
constexpr size_t kOffFlags = kOffCell + al(kNoAllocMaxPoints * sizeof(int2));
constexpr size_t kOffOrig = kOffFlags + al(kNoAllocMaxPoints * 4);
constexpr size_t kOffRank = kOffOrig + al(kNoAllocMaxPoints * 4);
constexpr size_t kOffCellStart = kOffRank + al(kNoAllocMaxPoints * 4);
constexpr size_t kOffBoff = kOffCellStart + al((kNoAllocMaxCells + 1) * 4);
constexpr size_t kOffParams = kOffBoff + al(kScanBlocks * 4);
// what a launch clears: the work counters and the ticket of the scan, the outputs' copies (pair_copies: one,
// or at most 131,072 words), the cell counts (as many of them as the call needs)
constexpr size_t kOffQueue = kOffParams + al(sizeof(BinDesc) + 16 + kMaxRows * sizeof(Row));
constexpr size_t kOffWork = kOffQueue + al((64 * kQueuePad + 1) * 4);
constexpr size_t kOffIngest = kOffWork + al((6 * kMaxHist + 8 + 131072) * 8) + al((2 * kNoAllocMaxCells + 1) * 4);
constexpr size_t kNoAllocBytes = kOffIngest + al(kIngestBlocks * sizeof(IngestScratch));

// The array.  In host code its name stands for the symbol, not for a device address: host code
// uses the address hipGetSymbolAddress returns for the current device (scratch_base below).
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
std::mutex g_mu;
unsigned char* g_base[kMaxDevices] = {};

// The array's address on `device` (which must be current), looked up once per device.
int scratch_base(int device, unsigned char** out)
{
    if (device < 0 || device >= kMaxDevices) return fail(GS_ENODEV, "device %d out of range", device);
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_base[device]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        g_base[device] = (unsigned char*)ptr;
    }
    *out = g_base[device];
    return GS_OK;
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" int gs_count_2pcf_noalloc(gs_ctx* c, const gs_params* p, const double* d_xyz, const double* d_w,
                                     const int32_t* d_buf, int64_t n_data, int64_t n_rand, uint64_t* cnt,
                                     double* wsum, double* n2, double* n3, gs_stats* st)
{
    if (!c) return fail(GS_EINVAL, "NULL context");
    int rc = check_params(p, 2);
    if (rc) return rc;
    const int64_t n = n_data + n_rand;
    if (n_data < 0 || n_rand < 0 || (!d_xyz && n > 0)) return fail(GS_EINVAL, "bad catalogue (NULL or sizes)");
    if (n > kNoAllocMaxPoints)
        return fail(GS_ELIMIT, "gs_count_2pcf_noalloc holds at most %lld points (got %lld)",
                    (long long)kNoAllocMaxPoints, (long long)n);
    if ((rc = ctx_set_device(c))) return rc;
    CtxView v = view(c);
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    unsigned char* base;
    if ((rc = scratch_base(device, &base))) return rc;
    const hipStream_t s = v.stream;

    // ---- weights and bounding box: the context's pass over a new catalogue, which copies nothing here
    CatalogueInfo info;
    if ((rc = ctx_catalogue_info(c, d_xyz, d_w, d_buf, n, n_data, (double*)d_xyz, (double*)d_w, (int32_t*)d_buf,
                                 (IngestScratch*)(base + kOffIngest), &info)))
        return rc;

    // ---- grid (as gs_count_2pcf, with the cell edge widened to fit kNoAllocMaxCells)
    const int nb = p->nbins, nm = p->nmu;
    const bool weighted = d_w != nullptr;
    const int nbt = 3 * nb * nm;
    const PairGrid q = pair_grid(n, info.bbox, p->rmax, p->cell_div, kNoAllocMaxCells);
    std::vector<Row> rows = half_stencil(q.h, q.h / q.sx, p->rmax, q.mst);
    if ((int)rows.size() > kMaxRows) return fail(GS_ELIMIT, "stencil too large");
    GridDesc g;
    if ((rc = grid_desc(info.bbox, q.h, q.sx, kNoAllocMaxCells, &g))) return rc;
    if (cell_scan_blocks(g.ncell) > kScanBlocks) return fail(GS_ELIMIT, "scan scratch too small");

    // ---- bins, launch shape, parameters, cleared accumulators
    double xmax = 0, t64[kMaxBins + 2];
    for (int k = 0; k < 6; ++k) xmax = std::max(xmax, std::fabs(info.bbox[k]));
    const int copies = pair_copies(1, nbt);
    const size_t nwork = (size_t)copies * pair_copy_words(1, nbt), nout = 3 * (size_t)nbt + 4;
    const size_t rows_off = (sizeof(BinDesc) + 15) / 16 * 16, blob = rows_off + rows.size() * sizeof(Row);
    const size_t out_off = al(blob);
    HostBuf& H = ctx_host(c);
    if ((rc = ctx_thresholds(c, *p, t64)) || (rc = H.reserve(out_off + nout * 8))) return rc;
    BinDesc& B = *(BinDesc*)H.ptr;
    if ((rc = fill_pair_bins(*p, t64, q, xmax, info.wmax_d, info.wmax_r, B))) return rc;
    std::copy(rows.begin(), rows.end(), (Row*)(H.ptr + rows_off));
    const PairVariant var{nb, nm, p->precision == GS_FP64 || B.wide, weighted, p->log_bins != 0, d_buf != nullptr};
    PairShape shape;
    if ((rc = pair2_shape(var, &shape))) return rc;
    unsigned char* dB = base + kOffParams;
    unsigned long long* work = (unsigned long long*)(base + kOffWork);
    const size_t count_off = kOffWork + al(nwork * 8);
    e = hipMemcpyAsync(dB, H.ptr, blob, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return hip_fail(e, "parameter upload");
    // the array keeps the previous call's contents: clear what starts at zero (with a fill kernel)
    (void)hipEventRecord(v.ev[0], s);
    e = launch_fill_u32(base + kOffQueue, (int64_t)(count_off + (2 * (size_t)g.ncell + 1) * 4 - kOffQueue) / 4, 0u, s);
    GridArgs ga{};
    ga.xyz = d_xyz;
    ga.w = d_w;
    ga.buf = d_buf;
    ga.n = n;
    ga.n_data = n_data;
    ga.ncell = g.ncell;
    ga.g = g;
    ga.rank = (int32_t*)(base + kOffRank);
    ga.count = (int32_t*)(base + count_off);
    ga.boff = (int32_t*)(base + kOffBoff);
    ga.ticket = (unsigned*)(base + kOffQueue) + 64 * kQueuePad;
    ga.pw = (double4*)(base + kOffPw);
    ga.cell = (int2*)(base + kOffCell);
    ga.flags = (uint32_t*)(base + kOffFlags);
    ga.orig = (int32_t*)(base + kOffOrig);
    ga.cell_start = (int32_t*)(base + kOffCellStart);
    if (e == hipSuccess && n > 0) e = launch_cell_sort(ga, s);
    if (e != hipSuccess) return hip_fail(e, "grid build");

    PairArgs a{};
    a.pw = ga.pw;
    a.cell = ga.cell;
    a.flags = ga.flags;
    a.cell_start = ga.cell_start;
    a.rows = (const Row*)(dB + rows_off);
    a.bins = (const BinDesc*)dB;
    a.queue = (int32_t*)(base + kOffQueue);
    a.out_cnt = work;
    a.out_w = work + 2 * nbt;
    a.out_stats = work + 6 * nbt;
    a.copies = copies;
    a.copy_stride = pair_copy_words(1, nbt);
    a.g = g;
    a.g.m = q.mst;
    a.nrows = (int)rows.size();
    (void)hipEventRecord(v.ev[2], s);
    if (n > 0) {
        e = pair_launch(a, var, shape, q, n, v.n_cu, s);
        if (e != hipSuccess) return hip_fail(e, "pair kernel launch");
    }
    (void)hipEventRecord(v.ev[3], s);
    unsigned long long* const h_out = (unsigned long long*)(H.ptr + out_off);
    e = launch_pair_reduce(work, copies, 1, nbt, nm, weighted, h_out, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_fail(e, "pair kernel");
    combine2(h_out, nb, nm, B, weighted, info.wsum_d, info.wsum_r, cnt, wsum, n2, n3, st);
    if (st) {
        float ms_grid = 0, ms_count = 0;
        (void)hipEventElapsedTime(&ms_grid, v.ev[0], v.ev[2]);
        (void)hipEventElapsedTime(&ms_count, v.ev[2], v.ev[3]);
        st->ms_grid = ms_grid;
        st->ms_count = ms_count;
        st->ms_kernel_avg = ms_count;
        st->cell_div = q.mst;
    }
    return GS_OK;
}
