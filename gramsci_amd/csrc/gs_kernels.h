// gs_kernels.h -- launch interfaces of the HIP kernels (host side).
#pragma once

#include "gs_common.h"

namespace gs {

// grid.hip
// What the pass over a new catalogue finds: v = bounding box (3 lowest, 3 highest), largest data and random
// weight, index of the first invalid (negative or non-finite) weight (1e308: none); s = exact fixed-point
// sums of the data and the random weights (lo, hi each).  Lives in device memory, with a pointer to the
// pinned host copy that the last kernel fills in.
struct CatalogueStats {
    double v[9];
    unsigned long long s[4];
    unsigned ticket;            // blocks done (zero between launches)
    CatalogueStats* host;
};
struct IngestScratch {          // one per block
    double v[9];
    unsigned long long s[4];
};
constexpr int kIngestBlocks = 1024;
// copies xyz, w, buf (w, buf may be NULL) to xyz_out, w_out, buf_out (or nothing where they are the same) and
// fills *stats and its host copy
hipError_t launch_ingest(const double* xyz, const double* w, const int32_t* buf, int64_t n, int64_t n_data,
                         double* xyz_out, double* w_out, int32_t* buf_out, IngestScratch* scratch, CatalogueStats* stats,
                         hipStream_t st);

// Counting sort of a catalogue (input order) into the cells of a grid, or of each region's grid.
struct GridArgs {
    const double *xyz, *w;
    const int32_t* buf;
    int64_t n, n_data, ncell;
    GridDesc g;                 // lo, dim: single grid; h, hx
    const RegionDesc* regions;  // batch (nreg > 0)
    const int32_t* off;         // nreg+1 first point of each region
    int32_t nreg;
    int32_t* rank;              // [n] scratch
    int32_t* count;             // [2 ncell + 1] scratch: data and randoms per cell, points in none; zero before
    int32_t* boff;              // [cell_scan_blocks(ncell)] scratch
    unsigned* ticket;           // zero before and after
    // the sorted catalogue: point and raw weight, x cell and x-row (over all regions), flags, input index
    double4* pw;
    int2* cell;
    uint32_t* flags;
    int32_t *orig, *cell_start; // cell_start[ncell + 1]
};
int64_t cell_scan_blocks(int64_t ncell);
hipError_t launch_cell_sort(const GridArgs& a, hipStream_t st);

hipError_t exclusive_scan(const int32_t* in, int32_t* out, int64_t n, int32_t* scratch, hipStream_t st);
int64_t scan_scratch_size(int64_t n);
hipError_t launch_row_chunks(const int32_t* start, int nx, int nrow, int group, int32_t* nch, hipStream_t st);
hipError_t launch_fill_u32(void* p, int64_t n, uint32_t v, hipStream_t st);

// domain decomposition (decompose.hip)
hipError_t launch_region_box(const float* xyz, const int32_t* reg, int64_t n, int nreg, int32_t* keys, hipStream_t st);
hipError_t launch_region_flag(const float* xyz, int64_t n, const float* ext, int32_t* flag, hipStream_t st);
hipError_t launch_region_scatter(const float* xyz, int64_t n, const float* box, const int32_t* flag, const int32_t* pos,
                                 int32_t* idx, int32_t* buf, hipStream_t st);

// The half-stencil walk of the pair and adjoint kernels (gs_pair_tiles.h).
struct WalkArgs {
    const double4* pw;          // sorted points: x, y, z, raw weight
    const int2* cell;           // sorted: x cell, x-row of cells (over all regions)
    const uint32_t* flags;      // sorted: bit0 random, bit1 never-apex
    const int32_t* cell_start;  // ncell+1
    const Row* rows;            // half stencil
    const BinDesc* bins;        // device copy
    int32_t* queue;             // 64 work counters (dev::ItemQueue), zeroed before launch
    GridDesc g;
    int32_t n;                  // points
    int32_t nrows;
    int32_t group;              // points per chunk: 16, 32 or 64
    int32_t lg_parts;           // log2 of the work items per chunk
    int32_t cap_cells;          // largest extent of a piece of a chunk in x cells, less one
    const RegionDesc* regions;  // batched regions (nreg > 0): per-region grids
    const int32_t* row_base;    // nreg+1 first x-row of each region
    int32_t nreg;
};

// Arguments of the persistent 2PCF pair kernel (pair2.hip).
struct PairArgs : WalkArgs {
    unsigned long long* out_cnt;    // [2][3][nb][nm]: plane 0 counts for both directions, plane 1 for one
    unsigned long long* out_w;      // [2][3][nb][nm][2] 128-bit fixed point (lo, hi)
    unsigned long long* out_stats;  // [0] candidates, [1] rechecks, [2] overflow pairs
    int64_t copy_stride;        // words between the copies of the outputs (pair_copy_words)
    int32_t copies;             // power of two <= 64; work-group b adds to copy b mod copies
    int32_t reps;               // LDS histogram replicas (power of two <= 32)
    int32_t planes;             // with buffer points: 2 if the LDS histogram has a plane per direction count
};

// Copies of `words` words that fit 1 MiB, at most 64 (a power of two, at least 1).
inline int output_copies(int64_t words)
{
    int c = 1;
    while (c < 64 && 2 * c * words <= 131072) c *= 2;
    return c;
}
// One copy of the pair kernel's outputs: [nreg][2][nbt] counts, [nreg][2][nbt][2] sums, 4 statistics.
inline int64_t pair_copy_words(int64_t nreg, int64_t nbt) { return 6 * nreg * nbt + 4; }
inline int pair_copies(int64_t nreg, int64_t nbt) { return output_copies(pair_copy_words(nreg, nbt)); }

// The pair kernel's variant: histogram, precision, unit or given weights, bins, buffer points or none.
struct PairVariant {
    int nb, nm;
    bool fp64, weighted, logb, buf;
};

// Arguments of the persistent 3PCF triplet kernel (triplet3.hip).
// Histogram cell h = (cfg * nm + mu) * 4 + class.
struct TripArgs {
    const double4* pw;
    const uint32_t* flags;
    const int32_t* orig;        // original input index of each sorted point (RSD: find_normal argument order)
    const int32_t* cell_start;
    const Row* rows;            // full stencil
    const BinDesc* bins;
    const uint16_t* cfg_tab;    // [nb][nb][nb] -> 0-based configuration (unused when equi)
    const uint8_t* ntab;        // RSD: [nm][nm] 0-based find_normal bin of (mu(k1), mu(k2))
    int32_t* queue;             // work counters (ItemQueue)
    int32_t* err;               // set to 1 if an apex has more than kmax neighbours
    // outputs, `copies` of them copy_words() apart; work-group b adds to copy b mod copies
    unsigned long long* out_cnt;    // [nreg][ncfg][nm][4]
    unsigned long long* out_w;      // [nreg][ncfg][nm][4][2]
    unsigned long long* out_stats;  // candidates, rechecks, overflow, units, evaluated pairs
    int64_t copy_stride;
    int32_t copies;             // power of two <= 64
    GridDesc g;
    int32_t nrows;
    int32_t n_items;            // apexes (all points; buffer points are skipped)
    int32_t ncfg;               // configurations (nb for equi: the configuration is the common bin)
    int32_t nm;                 // mu bins (1: isotropic)
    int32_t equi;               // only triangles whose three sides share one bin
    int32_t reps;
    int32_t kmax;
    int32_t lds_hist;           // histogram in LDS (else global atomics)
    // batched regions (nreg > 0): each apex uses its region's grid (regions[r].lo/dim/cell_base,
    // g.h shared) and adds to its region's histogram, out_cnt/out_w + r * [ncfg][nm][4]
    int32_t nreg;
    const RegionDesc* regions;
    // two-pass runs: with ovf set, an apex with more than kmax neighbours is appended to
    // ovf (count in *ovf_n) and skipped instead of raising err; with items set, work item
    // t is apex items[t] (the second pass over those apexes, with a larger kmax)
    int32_t* ovf;
    int32_t* ovf_n;
    const int32_t* items;
    const int32_t* n_items_dev;     // if set, the number of work items is read here (captured second pass)
    int32_t log_bins;               // selects the kernel variant (log or linear bin estimate)
    int32_t wg;                     // threads per work-group (one apex each): 64, 128 or 256 (0: 256)
    int32_t batch;                  // apexes taken per queue fetch (0: 1)
    // neighbour counts beyond every LDS list: with ovf_kmax set, the largest neighbour count of a
    // queued apex is kept there (atomic max); with glist set, each work-group keeps its apex's
    // neighbour list in device memory at glist + blockIdx.x * glist_stride bytes (kmax entries)
    // instead of LDS, and the histogram goes to global memory
    int32_t* ovf_kmax;
    void* glist;
    int64_t glist_stride;
    // triplet_matrix.hip: tables, and the three bins of each configuration (a byte each); buffer points present
    const struct TripMatrix* matrix;
    const uint32_t* cfg_bins;
    int32_t buf;
};
// Tables of the matrix kernel (fill_triplet_matrix), for coordinates scaled by a power of two such that rmax is
// in [1, 2): a squared side s is certainly in slot k (0: below the bins, nb + 1: above) if s - ok[k].x, as a
// float's bits, is below those of ok[k].y; its slot is estimated by f(s) ua + ub, f = sqrt (linear) or log2 (log).
struct TripMatrix {
    double scale;
    double t_top;               // kept neighbours of an apex: t64[0] < s < t_top (beyond, up to t64[nb+1]: overflow)
    double inv_h, inv_hx;       // 1 / cell edges
    float2 ok[kMaxBins + 2];
    float ua, ub;
};
// teams: waves of a work-group that take an apex each, or 1
size_t triplet_matrix_lds(const TripArgs& a, int nb, int teams);
hipError_t launch_triplet_matrix(const TripArgs& a, int nb, bool wave, int nblocks, hipStream_t st);
int triplet_matrix_occupancy(const TripArgs& a, int nb, bool wave);
// One copy of the triplet kernel's outputs (nh histogram entries over all regions): counts, sums, 8 statistics.
inline int64_t triplet_copy_words(int64_t nh) { return 3 * nh + 8; }
// Sums the copies into out (device or pinned host memory): entries [0, nplain) as 64-bit integers, then nwide
// two-word integers, then ntail 64-bit ones.
hipError_t launch_sum_copies(const unsigned long long* in, int copies, int64_t stride, int64_t nplain, int64_t nwide,
                             int64_t ntail, unsigned long long* out, hipStream_t st);
// bytes per neighbour of a device-memory neighbour list (glist) of the triplet kernel
size_t triplet3_glist_entry_bytes(const TripArgs& a, bool fp64, bool weighted);
size_t triplet3_lds_bytes(const TripArgs& a, int nb, bool fp64, bool weighted);
size_t triplet3_queue_bytes(const TripArgs& a, bool weighted);
hipError_t launch_triplet3(const TripArgs& a, int nb, bool fp64, bool weighted, int nblocks, hipStream_t st);
int triplet3_occupancy(const TripArgs& a, int nb, bool fp64, bool weighted);
// neighbour counts of the apexes t * stride (t < nsample) of a single catalogue, -1 for buffer points, then the
// numbers of their candidates
hipError_t launch_nbr_count(const TripArgs& a, int stride, int nsample, int after_only, int32_t* out,
                            hipStream_t st);

// Arguments of the persistent 4PCF quad kernel (quad4.hip).
struct QuadArgs {
    const double4* pw;
    const uint32_t* flags;
    const int32_t* orig;        // original input index of each sorted point
    const int32_t* cell_start;
    const Row* rows;            // full stencil
    const BinDesc* bins;
    const uint16_t* cfg_tab;    // [nb]^4 -> 1-based perimeter configuration, 0 = not sorted
    int32_t* queue;             // work counters (ItemQueue)
    int32_t* err;
    // outputs, `copies` of them copy_stride words apart; work-group b adds to copy b mod copies
    int64_t copy_stride;
    int32_t copies;             // power of two <= 64
    unsigned long long* out_cnt;    // [ncell][16]
    double* out_w;              // weighted: [ncell][16] quad products, [6][ncell][4] disc pair (tetra: triple) products
    unsigned long long* out_stats;
    GridDesc g;
    int32_t nrows;
    int32_t n_items;
    int32_t ncell;
    int32_t kmax;
    int32_t lds_hist;           // counts in LDS (else global atomics)
    int32_t tetra;              // regular tetrahedra only (all six sides in one bin; cell = that bin)
    // two-pass runs, as for the triplet kernel: with ovf set, an apex with more than kmax
    // neighbours is queued (count in *ovf_n) and skipped; with items set, work item t is apex items[t]
    int32_t* ovf;
    int32_t* ovf_n;
    const int32_t* items;
    const int32_t* n_items_dev; // if set, the number of work items is read here
    int32_t batch;              // apexes taken per queue fetch (0: 1)
    int32_t bin_masks;          // a mask per bin and neighbour of the quads' last points, else one per neighbour
    int32_t lds_w;              // weighted sums in LDS (else global atomics; device-memory lists: always those)
    // as for the triplet kernel: with ovf_kmax set, the largest neighbour count of a queued apex is
    // kept there; with glist set, each work-group keeps its apex's neighbour list (kmax entries, a
    // power of two) at glist + blockIdx.x * glist_stride bytes of device memory, with no link matrix
    // (the neighbour-neighbour bins are evaluated where they are needed)
    int32_t* ovf_kmax;
    void* glist;
    int64_t glist_stride;
};
// bytes per neighbour of a device-memory neighbour list (glist) of the quad kernel: x, y, z, w,
// key, permutation, packed bin, and the sort's staging copy of x, y, z, w and the packed bin
constexpr size_t kQuadGlistEntryBytes = 4 * 8 + 3 * 4 + 4 * 8 + 4;
// kmax: 64, 128 or 256; wave: one wave per apex (kmax 64)
size_t quad4_lds_bytes(const QuadArgs& a, int nb, bool weighted, bool wave);
hipError_t launch_quad4(const QuadArgs& a, int nb, bool weighted, bool wave, int nblocks, hipStream_t st);
int quad4_occupancy(const QuadArgs& a, int nb, bool weighted, bool wave);
hipError_t launch_sum_copies_f64(const double* in, int copies, int64_t stride, int64_t n, double* out, hipStream_t st);

// Arguments of the persistent 2PCF adjoint kernel (adjoint.hip).
struct AdjArgs {
    const double4* pw;
    const int2* cell;           // sorted: x cell, x-row
    const uint32_t* flags;
    const int32_t* orig;
    const int32_t* cell_start;
    const int32_t* row_chunk;
    const Row* rows;            // full stencil
    const BinDesc* bins;
    const double* g2;           // dL/dN2 [nb][nm]
    const double* g3;           // dL/dN3 [nb][nm]
    int32_t* queue;
    double* G;                  // dL/dwn per point, original order
    unsigned long long* out_stats;
    GridDesc g;
    int32_t nrows;
    int32_t n_chunks;
    double inv_wd, inv_wr;
};
// Arguments of the half-stencil FP32 adjoint kernel: per sorted point a fixed-point sum Ghi * 2^32 + Glo of
// G * 2^F (zeroed before launch), with the dL/dN tables scaled by g_scale and the normalised weights by
// w_scale (g_scale * w_scale = 2^F).
struct AdjHalfArgs : WalkArgs {
    const double* g2;           // dL/dN2 [nb][nm]
    const double* g3;           // dL/dN3 [nb][nm]
    unsigned long long* Glo;
    long long* Ghi;
    unsigned long long* out_stats;  // candidates, rechecks
    double inv_wd, inv_wr, g_scale, w_scale;
};
size_t adjoint2_lds_bytes(int nb, int nm, bool fp64);
hipError_t launch_adjoint2(const AdjArgs& a, int nb, int nm, bool fp64, bool rsd, int nblocks, hipStream_t st);
int adjoint2_occupancy(int nb, int nm, bool fp64, bool rsd);
// half-stencil FP32 adjoint (rows: half stencil): every unordered pair once, its term added to both ends
size_t adjoint2h_lds_bytes(int nb, int nm, bool buf);
hipError_t launch_adjoint2h(const AdjHalfArgs& a, int nb, int nm, bool logb, bool buf, int nblocks, hipStream_t st);
int adjoint2h_occupancy(int nb, int nm, bool logb, bool buf);
// G[orig[k]] = (Ghi[k] * 2^32 + Glo[k]) * 2^-F (the sums as doubles, original order)
hipError_t launch_adj_fx(const unsigned long long* Glo, const long long* Ghi, const int32_t* orig, int64_t n, int F,
                         double* G, hipStream_t st);
// part: 2 nblk + 2; stats: the pair kernel's two counters and a zero ticket; host_stats: pinned host memory
hipError_t launch_adj_partials(const double* G, const double* w, int64_t n, int64_t n_data, double inv_wd,
                               double inv_wr, double* part, int nblk, unsigned long long* stats,
                               unsigned long long* host_stats, hipStream_t st);
hipError_t launch_adj_finish(const double* G, int64_t n, int64_t n_data, const double* sums, double inv_wd,
                             double inv_wr, double* out, hipStream_t st);

// largest dynamic LDS of the pair kernel (160 KiB less its static part)
constexpr size_t kPairLdsMax = 160 * 1024 - 32;
// Dynamic LDS bytes of the pair kernel for these parameters and work-group size wg (a multiple of 64, <= 1024).
size_t pair2_lds_bytes(int nb, int nm, int planes, int reps, bool weighted, bool batched, int wg);
hipError_t launch_pair2(const PairArgs& a, const PairVariant& v, int nblocks, int wg, hipStream_t st);
// its unit-weight variants (pair2_unit.hip)
hipError_t launch_pair2_unit(const PairArgs& a, const PairVariant& v, size_t lds, int nblocks, int wg, hipStream_t st);
int pair2_unit_occupancy(const PairVariant& v, size_t lds, int wg);
// copies -> [nreg][nbt] counts and [nreg][nbt][2] sums over ordered pairs, 4 statistics
hipError_t launch_pair_reduce(const unsigned long long* in, int copies, int nreg, int nbt, int nm, bool weighted,
                              unsigned long long* out, hipStream_t st);
// Work-groups of wg threads per CU the pair kernel can keep resident (0 if it cannot run).
int pair2_occupancy(const PairVariant& v, int planes, int reps, bool batched, int wg);

}  // namespace gs
