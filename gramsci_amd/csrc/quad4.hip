// quad4.hip -- persistent 4PCF quad kernel.
//
// Replaces create_graph (gramsci.F90:288-348) + query_4pcf_all2 (:662-861).
// For every apex i that is not a buffer point and has more than 3 kept
// neighbours (:675), and every k1 < k2 < k3 of its neighbours in ascending
// ORIGINAL index (the reference's neighbour lists are sorted by id,
// sorting_module.F90:36-47), with all three cross sides kept
// (find_dist :685,692,694), the quad is binned at
//     cell = (bintable(ind1, ind4, ind5, ind3), ind2, ind6)
// where ind1..3 are the apex sides, ind4 = (k1,k2), ind5 = (k2,k3) and
// ind6 = (k1,k3); bintable is only filled for non-decreasing perimeters
// (:1402-1420), so other orientations are dropped (:701).
//
// A team per apex, persistent over apexes (k_quad4):
//   1. gather the kept neighbours into LDS (indices by ballots, then records with all lanes busy);
//   2. sort them by original index (rank sort, one thread per neighbour);
//   3. evaluate every neighbour-neighbour side: a K x K matrix of bins, from which each row's bit masks;
//   4. for every linked (k1, k2) the k3 are the bits of an intersection of masks.
// Teams are single waves for at most 64 neighbours and unit weights, else work-groups (64, 128 or 256).  Apexes with more
// neighbours than an LDS list holds run in k_quad4_big, with lists in device memory and no matrix.
// Counts go to an LDS histogram [cell][16 random patterns] (or straight to
// global memory when it does not fit); weighted runs add FP64 sums of the
// quad products per pattern and of the six disc pair products (:754-818).
//
// What bounds it: latency and lane use.  A sparse sample has 10 to 60 neighbours an apex, 100 candidates, 2,000
// linked triples and some tens of quads, so a work-group of 256 threads per apex spent its time in barriers with most
// lanes idle, and a lane scanned every k3 > k2 for the few that close a quad.  One wave needs no barrier, and the
// masks give exactly the quads.  50k + 100k points, rmax 20 of box 500, 3 bins: 3.60 -> 0.97 ms
// in the kernels (by work-groups alone 1.84); weighted, 20k + 40k points, 2 bins, 92 quads an apex 12.3 -> 0.7.
//
// With `tetra` the kernel is query_graph_tetrahedron (:548-660) instead: no
// minimum neighbour count, only quads whose six sides share one bin b
// (cell = b), and the disc sums are triple products that include the weight
// of the point whose random status selects the term (:590-631).
#include "gs_device.h"
#include "gs_kernels.h"

namespace gs {

using namespace dev;

// LDS byte layout shared by host and device
namespace {

struct QuadLds {
    size_t t64, tab, hist, sums, lists, masks, rows, team, total;
};

// km: list entries (64, 128, 256); teams of a work-group; big: k_quad4_big, without lists
__host__ __device__ inline QuadLds quad_lds(const QuadArgs& a, int nb, bool weighted, int km, int teams, bool big)
{
    QuadLds l;
    size_t b = 0;
    l.t64 = b;
    b += ((size_t)(nb + 2) * 8 + 15) / 16 * 16;
    l.tab = b;
    if (!a.tetra) b += ((size_t)nb * nb * nb * nb * 2 + 15) / 16 * 16;      // perimeter table
    l.hist = b;
    if (a.lds_hist) b += (size_t)a.ncell * 16 * 4;
    l.sums = b;
    if (weighted && a.lds_w && !big) b += (size_t)a.ncell * 40 * 8;
    l.lists = b;
    // stencil rows (after the links where they are longer), then coordinates, beside them original and sorted index,
    // later the masks; weights; bins, random flags; links
    const size_t per = (size_t)km / 8 * (a.tetra ? 1 : 1 + (a.bin_masks ? nb : 1));
    const size_t rows = ((size_t)a.nrows * 12 + 15) / 16 * 16;
    l.masks = km * (per > 32 ? per : 32);
    l.team = big ? 0 : l.masks + km * ((weighted ? 8 : 0) + 2) + (size_t)km * (km + 4);
    l.rows = !big && rows <= (size_t)km * 24 ? 0 : l.team;
    if (l.rows == l.team) l.team += rows;
    l.total = b + teams * l.team;
    return l;
}

}  // namespace

// the FP64 sums of one quad: the product per pattern ([ncell][16]), then the six disc pair products and their
// conditions ([6][ncell][4]), gramsci.F90:710, :754-818; the tetrahedron's terms also carry the conditioning
// point's weight (:590-631)
__device__ __forceinline__ void add_quad_sums(double* ow, int ncell, int cell, int pat, int ri, int r1, int r2, int r3,
                                              double wi, double w1, double w2, double w3, bool tetra)
{
    atomicAdd(&ow[(size_t)cell * 16 + pat], wi * w1 * w2 * w3);
    double* od = ow + (size_t)ncell * 16;
    const double fi = tetra ? wi : 1.0, f1 = tetra ? w1 : 1.0, f3 = tetra ? w3 : 1.0;
    if (ri) {
        atomicAdd(&od[((size_t)3 * ncell + cell) * 4 + (r1 | r2 << 1)], w1 * w2 * fi);
        atomicAdd(&od[((size_t)4 * ncell + cell) * 4 + (r3 | r2 << 1)], w3 * w2 * fi);
        atomicAdd(&od[((size_t)5 * ncell + cell) * 4 + (r3 | r1 << 1)], w3 * w1 * fi);
    }
    if (r3) {
        atomicAdd(&od[((size_t)1 * ncell + cell) * 4 + (ri | r2 << 1)], wi * w2 * f3);
        atomicAdd(&od[((size_t)0 * ncell + cell) * 4 + (ri | r1 << 1)], wi * w1 * f3);
    }
    if (r1) atomicAdd(&od[((size_t)2 * ncell + cell) * 4 + (ri | r3 << 1)], wi * w3 * f1);
}

// The apex's neighbour list in device memory (a.glist), for apexes with more neighbours than an LDS list holds: one
// work-group per apex; the neighbour-neighbour bins are evaluated where needed (no matrix), and the quads run in
// segments with the LDS counts drained after each.
template <bool W>
__global__ __launch_bounds__(kWG) void k_quad4_big(QuadArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const int nb = B.nb;
    const int kmax = a.kmax;
    const int ncell = a.ncell;
    const bool lh = a.lds_hist != 0;
    const bool tetra = a.tetra != 0;
    const int tid = threadIdx.x;

    const QuadLds l = quad_lds(a, nb, W, 64, 1, true);
    double* t64 = (double*)(smem + l.t64);
    uint16_t* tab = (uint16_t*)(smem + l.tab);
    uint32_t* hc = (uint32_t*)(smem + l.hist);
    // the apex's stencil rows: first point, number of points, and candidate number of the first point
    int32_t* rw_js = (int32_t*)(smem + l.lists);
    int32_t* rw_len = rw_js + a.nrows;
    int32_t* rw_off = rw_len + a.nrows;
    unsigned char* p = (unsigned char*)a.glist + (size_t)blockIdx.x * (size_t)a.glist_stride;
    double* nx_ = (double*)p;
    double* ny_ = nx_ + kmax;
    double* nz_ = ny_ + kmax;
    double* nw_ = nz_ + kmax;
    int32_t* key = (int32_t*)(nw_ + kmax);   // original index (sort key)
    int32_t* pk = key + kmax;                // sort permutation, then bin | rand << 8 in sorted order
    int32_t* jl = pk + kmax;                 // bin | rand << 8 in gather order
    uint8_t* L = (uint8_t*)(jl + kmax);      // the sort's staging area

    __shared__ int s_item, s_k, s_over, s_ncand;

    if (lh)
        for (int k = tid; k < ncell * 16; k += kWG) hc[k] = 0;
    for (int k = tid; k < nb + 2; k += kWG) t64[k] = B.t64[k];
    if (!tetra)
        for (int k = tid; k < nb * nb * nb * nb; k += kWG) tab[k] = a.cfg_tab[k];
    __syncthreads();

    const int nxg = a.g.dim[0], nyg = a.g.dim[1], nzg = a.g.dim[2];
    const double inv_h = 1.0 / a.g.h, inv_hx = 1.0 / a.g.hx;
    unsigned long long units = 0, binned = 0, over = 0, cand = 0;
    const int nb2 = nb * nb;
    // the work-group's copy of the outputs
    const size_t copy = (size_t)(blockIdx.x & (unsigned)(a.copies - 1)) * (size_t)a.copy_stride;
    unsigned long long* const out_cnt = a.out_cnt + copy;
    double* const out_w = a.out_w + copy;

    // adds the LDS counts to the global counts and clears them (all threads of the work-group)
    auto drain_counts = [&]() {
        for (int k = tid; k < ncell * 16; k += kWG) {
            const uint32_t v = hc[k];
            if (v) {
                atomicAdd(&out_cnt[k], (unsigned long long)v);
                hc[k] = 0;
            }
        }
    };
    // work items: batches of consecutive apexes, fetched by wave 0
    const int n_items = a.n_items_dev ? *a.n_items_dev : a.n_items;
    const int bsz = max(a.batch, 1);
    ItemQueue items(a.queue, (n_items + bsz - 1) / bsz, 1);
    int b_next = 0, b_end = 0;      // the rest of the current batch (work-group uniform)
    while (true) {
        if (tid == 0) {
            s_k = 0;
            s_over = 0;
        }
        const bool fetch = b_next >= b_end;
        if (fetch && tid < kWave) {
            const int b = items.next(tid, 0);
            if (tid == 0) s_item = b;
        }
        __syncthreads();
        if (fetch) {
            const int b = s_item;
            if (b < 0) break;
            b_next = b * bsz;
            b_end = min(n_items, b_next + bsz);
        }
        const int item = b_next++;
        const int apex = a.items ? a.items[item] : item;
        const uint32_t fa = a.flags[apex];
        if (fa & 2u) {
            __syncthreads();
            continue;
        }
        const double4 Pa = a.pw[apex];
        const int cx = min(max((int)floor((Pa.x - a.g.lo[0]) * inv_hx), 0), nxg - 1);
        const int cy = min(max((int)floor((Pa.y - a.g.lo[1]) * inv_h), 0), nyg - 1);
        const int cz = min(max((int)floor((Pa.z - a.g.lo[2]) * inv_h), 0), nzg - 1);

        const unsigned long long cand0 = cand, over0 = over;   // restored if the apex is queued
        // ---- 1. gather: the stencil rows' point ranges are read in parallel (one row per thread) into
        // LDS and numbered by a prefix sum over the rows; the candidates of all rows are then numbered
        // consecutively and thread t takes numbers t, t + 256, ... (every thread busy even where rows
        // are short)
        for (int r = tid; r < a.nrows; r += kWG) {
            const Row rw = a.rows[r];
            const int by = cy + rw.dy, bz = cz + rw.dz;
            const int bx0 = max(cx + rw.x0, 0), bx1 = min(cx + rw.x1, nxg - 1);
            int js = 0, len = 0;
            if (by >= 0 && by < nyg && bz >= 0 && bz < nzg && bx0 <= bx1) {
                const int rb = (bz * nyg + by) * nxg;
                js = a.cell_start[rb + bx0];
                len = a.cell_start[rb + bx1 + 1] - js;
            }
            rw_js[r] = js;
            rw_len[r] = len;
        }
        __syncthreads();
        if (tid < 64) {         // exclusive prefix of the row lengths, 64 rows at a time (wave 0)
            int run = 0;
            for (int b0 = 0; b0 < a.nrows; b0 += 64) {
                const int x = b0 + tid < a.nrows ? rw_len[b0 + tid] : 0;
                int inc = x;
                for (int off = 1; off < 64; off <<= 1) {
                    const int y = __shfl_up(inc, off, 64);
                    if (tid >= off) inc += y;
                }
                if (b0 + tid < a.nrows) rw_off[b0 + tid] = run + inc - x;
                run += __shfl(inc, 63, 64);
            }
            if (tid == 0) s_ncand = run;
        }
        __syncthreads();
        const int ncand = s_ncand;
        int row = 0, row_end = a.nrows > 0 ? rw_len[0] : 0, j0 = a.nrows > 0 ? rw_js[0] : 0;
        {
            for (int next = tid; next < ncand; next += kWG) {
                while (next >= row_end) {           // the row holding candidate number next
                    ++row;
                    const int row_beg = rw_off[row];
                    row_end = row_beg + rw_len[row];
                    j0 = rw_js[row] - row_beg;
                }
                const int j = j0 + next;
                ++cand;
                const double4 Pj = a.pw[j];
                const int b = bin_of(exact_s(Pa.x, Pa.y, Pa.z, Pj.x, Pj.y, Pj.z), t64, nb);
                if (b < 0) continue;
                if (b == nb) { ++over; continue; }
                const int pos = atomicAdd(&s_k, 1);
                if (pos >= kmax) { s_over = 1; continue; }
                nx_[pos] = Pj.x; ny_[pos] = Pj.y; nz_[pos] = Pj.z; nw_[pos] = Pj.w;
                key[pos] = a.orig[j];
                jl[pos] = (int)(b | ((a.flags[j] & 1u) << 8));   // packed, moved by the sort below
            }
        }
        __syncthreads();
        const int K = min(s_k, kmax);
        if (s_over) {
            if (a.ovf) {
                // left to a later pass with room for all its neighbours (s_k counted every one)
                if (tid == 0) {
                    a.ovf[atomicAdd(a.ovf_n, 1)] = apex;
                    if (a.ovf_kmax) atomicMax(a.ovf_kmax, s_k);
                }
                cand = cand0;       // the later pass counts this apex's candidates
                over = over0;
                __syncthreads();
                continue;
            }
            if (tid == 0) atomicExch(a.err, 1);
        }
        if (K <= (tetra ? 2 : 3)) {        // gramsci.F90:675 (the tetrahedron query has no such skip)
            __syncthreads();
            continue;
        }

        // ---- 2. sort by original index
        // bitonic sort of (key, slot), then gather (slot pk[u] -> position u) through the device-memory
        // list's staging area
        double* tmp = (double*)L;
        int np2 = 1;
        while (np2 < K) np2 <<= 1;
        for (int k = tid; k < np2; k += kWG) pk[k] = k;           // slot permutation
        __syncthreads();
        for (int size = 2; size <= np2; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int t = tid; t < np2 / 2; t += kWG) {
                    const int lo = 2 * t - (t & (stride - 1));
                    const int hi = lo + stride;
                    const bool up = ((lo & size) == 0);
                    const int sa = pk[lo], sb = pk[hi];
                    const int ka = sa < K ? key[sa] : 0x7fffffff;
                    const int kb = sb < K ? key[sb] : 0x7fffffff;
                    if ((ka > kb) == up) { pk[lo] = sb; pk[hi] = sa; }
                }
                __syncthreads();
            }
        }
        for (int u = tid; u < K; u += kWG) {
            const int sl = pk[u];
            tmp[u] = nx_[sl];
            tmp[K + u] = ny_[sl];
            tmp[2 * K + u] = nz_[sl];
            tmp[3 * K + u] = nw_[sl];
            ((int*)(tmp + 4 * K))[u] = jl[sl];
        }
        __syncthreads();
        for (int u = tid; u < K; u += kWG) {
            nx_[u] = tmp[u]; ny_[u] = tmp[K + u]; nz_[u] = tmp[2 * K + u]; nw_[u] = tmp[3 * K + u];
            pk[u] = ((int*)(tmp + 4 * K))[u];
        }
        __syncthreads();

        // ---- 3. neighbour-neighbour side bins (find_dist), evaluated where they are needed
        auto link = [&](int x, int y) -> int {       // x < y: bin + 1 of side (x, y), 0 if not kept
            const int b = bin_of(exact_s(nx_[x], ny_[x], nz_[x], nx_[y], ny_[y], nz_[y]), t64, nb);
            return (b >= 0 && b < nb) ? b + 1 : 0;
        };

        // ---- 4. quads: linked (k1, k2) over the lanes, k3 > k2 scanned by the lane
        const int ri = (int)(fa & 1u);
        const double wi = Pa.w;
        const long long P = (long long)K * (K - 1) / 2;
        int u = 0;
        long long rem = tid;
        while (u < K - 1 && rem >= K - 1 - u) { rem -= K - 1 - u; ++u; }
        // segments of at most 2^30 / K pairs (each adds fewer than K counts), with the u32 LDS counts drained after
        // each, and after every apex
        const long long seg = max((long long)kWG, ((1ll << 30) / max(K, 1)) / kWG * kWG);
        long long pi = tid;
        for (long long s0 = 0; s0 < P; s0 += seg) {
        if (s0 > 0) {
            __syncthreads();
            if (lh) drain_counts();
            __syncthreads();
        }
        const long long s1 = min(P, s0 + seg);
        for (; pi < s1; pi += kWG) {
            const int v = u + 1 + (int)rem;
            const int ind4 = link(u, v);
            const int p1 = pk[u], p2 = pk[v];
            const int ind1 = (p1 & 255) + 1, ind2 = (p2 & 255) + 1;
            if (ind4 && (!tetra || (ind2 == ind1 && ind4 == ind1))) {     // tetra: gramsci.F90:564-567
                units += (unsigned long long)(K - 1 - v);
                const int r1 = (p1 >> 8) & 1, r2 = (p2 >> 8) & 1;
                for (int k3 = v + 1; k3 < K; ++k3) {
                    const int ind5 = link(v, k3);
                    if (!ind5) continue;
                    const int ind6 = link(u, k3);
                    if (!ind6) continue;
                    const int p3 = pk[k3];
                    const int ind3 = (p3 & 255) + 1;
                    int cell;
                    if (tetra) {
                        if (ind3 != ind1 || ind5 != ind1 || ind6 != ind1) continue;   // :571-579
                        cell = ind1 - 1;
                    } else {
                        const int cfg = tab[(((ind1 - 1) * nb + (ind4 - 1)) * nb + (ind5 - 1)) * nb + (ind3 - 1)];
                        if (cfg == 0) continue;
                        cell = (cfg - 1) * nb2 + (ind2 - 1) * nb + (ind6 - 1);
                    }
                    const int r3 = (p3 >> 8) & 1;
                    const int pat = ri | (r1 << 1) | (r2 << 2) | (r3 << 3);
                    ++binned;
                    if (lh) atomicAdd(&hc[cell * 16 + pat], 1u);
                    else atomicAdd(&out_cnt[(size_t)cell * 16 + pat], 1ull);
                    if constexpr (W) {
                        add_quad_sums(out_w, ncell, cell, pat, ri, r1, r2, r3, wi, nw_[u], nw_[v], nw_[k3], tetra);
                    }
                }
            }
            rem += kWG;
            while (u < K - 1 && rem >= K - 1 - u) { rem -= K - 1 - u; ++u; }
        }
        }
        __syncthreads();
        if (lh) drain_counts();
    }
    __syncthreads();
    // statistics: summed over the work-group, then added to its copy of the outputs
    __shared__ unsigned long long s_stat[5];
    if (tid < 5) s_stat[tid] = 0;
    __syncthreads();
    const unsigned long long st[5] = {cand, 0, over, units, binned};
    for (int q = 0; q < 5; ++q) {
        unsigned long long v = st[q];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if ((tid & 63) == 0 && v) atomicAdd(&s_stat[q], v);
    }
    __syncthreads();
    if (tid < 5 && s_stat[tid]) atomicAdd(&a.out_stats[copy + tid], s_stat[tid]);
}

// Apexes with at most KM = 64 NW neighbours, one team (WAVE: a wave, else the work-group) each.  Sets of neighbours
// are masks of NW 64-bit words:
//   M[u]     the neighbours k > u linked to u (a kept side);
//   T[b][v]  the neighbours k > v with b <= ind5 <= ind3 (ind5 the bin of their side to v, ind3 that of their side to
//            the apex),
// so that the k3 of all quads of a linked pair (u, v) are the bits of T[ind4][v] & M[u].  Those are BIN's 1 + nb
// masks a neighbour.  Without BIN there is one T[v], of 1 <= ind5 <= ind3, and ind5 >= ind4 is tested bit by bit; or
// (tetra) T[v] alone, of ind5 = ind3 = ind2, the one bin of all sides, and the k3 are the bits of T[v] & T[u].  The masks
// come from the rows of link bytes, four at a time: with bytes below 128, (x | 0x80) - y keeps bit 7 exactly where
// x >= y, and a dot product of the bytes' bits packs them.  Sums of weighted quads go to LDS where they fit (a.lds_w).
template <bool W, int NW, bool WAVE, bool BIN>
__global__ __launch_bounds__(kWG) void k_quad4(QuadArgs a)
{
    static_assert(!WAVE || (NW == 1 && !W), "a wave holds one neighbour per lane");
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const int nb = scalar(B.nb), nb2 = nb * nb, ncell = a.ncell;
    const bool lh = a.lds_hist != 0, lw = W && a.lds_w != 0, tetra = !BIN && a.tetra != 0;
    const int tid = threadIdx.x, lane = tid & 63, wv = scalar(tid >> 6);
    constexpr int teams = WAVE ? kWG / kWave : 1, tn = WAVE ? kWave : kWG, KM = 64 * NW, LD = KM + 4;
    const int tl = WAVE ? lane : tid;
    auto sync = [&]() {
        if constexpr (WAVE) wave_sync();
        else __syncthreads();
    };

    const QuadLds l = quad_lds(a, nb, W, KM, teams, false);
    double* t64 = (double*)(smem + l.t64);
    uint16_t* tab = (uint16_t*)(smem + l.tab);
    uint32_t* hc = (uint32_t*)(smem + l.hist);
    double* hw = (double*)(smem + l.sums);  // [ncell][16] products, [6][ncell][4] disc terms
    unsigned char* p = smem + l.lists + (WAVE ? wv : 0) * l.team;
    int32_t* rw_js = (int32_t*)(p + l.rows);
    int32_t* rw_len = rw_js + a.nrows;
    int32_t* rw_off = rw_len + a.nrows;
    double* xs = (double*)p;                // the sorted neighbours, their indices; from step 3b on the masks
    double* ys = xs + KM;
    double* zs = ys + KM;
    int32_t* key = (int32_t*)(zs + KM);
    int32_t* jl = key + KM;
    unsigned long long* M = (unsigned long long*)p;     // [NW][KM] (not tetra)
    unsigned long long* T = M + (tetra ? 0 : NW * KM);  // [BIN: nb][NW][KM]
    p += l.masks;
    double* ws = (double*)p;
    if (W) p += KM * 8;
    uint8_t* A = (uint8_t*)p;               // bin + 1 of the apex's sides
    uint8_t* rnd = A + KM;                  // random points
    uint8_t* L = rnd + KM;                  // [KM][LD] bin + 1 of side (u, v), u < v; 0: not kept.  An odd number of
                                            // words a row: lanes reading a column fall on all banks

    __shared__ int s_item, s_k, s_ncand;
    if (lh)
        for (int k = tid; k < ncell * 16; k += kWG) hc[k] = 0;
    if (lw)
        for (int k = tid; k < ncell * 40; k += kWG) hw[k] = 0.0;
    for (int k = tid; k < nb + 2; k += kWG) t64[k] = B.t64[k];
    if (!tetra)
        for (int k = tid; k < nb2 * nb2; k += kWG) tab[k] = a.cfg_tab[k];
    for (int k = tl; k < (KM * LD + 2 * KM) / 4; k += tn) ((uint32_t*)A)[k] = 0;    // bytes stay below 128
    if (tid == 0) s_k = 0;
    __syncthreads();

    const size_t copy = (size_t)(blockIdx.x & (unsigned)(a.copies - 1)) * (size_t)a.copy_stride;
    unsigned long long* const out_cnt = a.out_cnt + copy;
    double* const out_w = a.out_w + copy;
    auto drain_counts = [&](int t, int step) {
        for (int k = opaque(t); k < ncell * 16; k += step) {
            const uint32_t v = atomicExch(&hc[k], 0u);
            if (v) atomicAdd(&out_cnt[k], (unsigned long long)v);
        }
    };
    const double t_lo = scalar(B.t64[0]), t_hi = scalar(B.t64[nb + 1]);
    const float ua = B.ua, ub = B.ub, nbm1f = (float)(nb - 1);
    const bool logb = B.log_bins != 0;
    const int nx = a.g.dim[0], ny = a.g.dim[1], nz = a.g.dim[2];
    const double inv_h = scalar(1.0 / a.g.h), inv_hx = scalar(1.0 / a.g.hx);
    unsigned long long units = 0, bound = 0, cand = 0;
    unsigned long long binned = 0;
    unsigned over = 0;
    const int n_items = scalar(a.n_items_dev ? *a.n_items_dev : a.n_items);
    const int bsz = max(a.batch, 1);
    ItemQueue items(a.queue, (n_items + bsz - 1) / bsz, 1);

    // exact bin of a kept s (nb: overflow), as adjust_bin
    auto bin_kept = [&](double s) {
        int b = (int)__builtin_amdgcn_fmed3f(bin_estimate((float)s, logb, ua, ub), 0.0f, nbm1f);
        while (b > 0 && s < t64[b]) --b;
        while (b < nb && s >= t64[b + 1]) ++b;
        return b;
    };

    auto visit_apex = [&](const int item) {
        const int apex = scalar(a.items ? a.items[item] : item);
        const uint32_t fa = (uint32_t)scalar((int)a.flags[apex]);
        if (fa & 2u) return;
        double4 Pa = a.pw[apex];
        Pa.x = scalar(Pa.x); Pa.y = scalar(Pa.y); Pa.z = scalar(Pa.z);
        const int cx = min(max((int)floor((Pa.x - a.g.lo[0]) * inv_hx), 0), nx - 1);
        const int cy = min(max((int)floor((Pa.y - a.g.lo[1]) * inv_h), 0), ny - 1);
        const int cz = min(max((int)floor((Pa.z - a.g.lo[2]) * inv_h), 0), nz - 1);
        // ---- 1. the stencil rows' candidates, numbered consecutively; the kept ones' indices by ballots
        int ncand = 0;
        if (WAVE || tid < kWave) {
            for (int b0 = 0; b0 < a.nrows; b0 += kWave) {
                const int r = b0 + lane;
                int js = 0, len = 0;
                if (r < a.nrows) {
                    const Row rw = a.rows[r];
                    const int by = cy + rw.dy, bz = cz + rw.dz;
                    const int bx0 = max(cx + rw.x0, 0), bx1 = min(cx + rw.x1, nx - 1);
                    if (by >= 0 && by < ny && bz >= 0 && bz < nz && bx0 <= bx1) {
                        const int rb = (bz * ny + by) * nx;
                        js = a.cell_start[rb + bx0];
                        len = a.cell_start[rb + bx1 + 1] - js;
                    }
                }
                int inc = len;
                for (int off = 1; off < kWave; off <<= 1) {
                    const int y = __shfl_up(inc, off, 64);
                    if (lane >= off) inc += y;
                }
                if (r < a.nrows) {
                    rw_js[r] = js;
                    rw_len[r] = len;
                    rw_off[r] = ncand + inc - len;
                }
                ncand += scalar(__shfl(inc, 63, 64));
            }
            if (!WAVE && tid == 0) s_ncand = ncand;
        }
        sync();
        if (!WAVE) ncand = scalar(s_ncand);
        int K = 0;
        unsigned n_over = 0;
        {
            int row = 0, row_end = a.nrows > 0 ? rw_len[0] : 0, j0 = a.nrows > 0 ? rw_js[0] : 0;
            for (int base = 0; base < ncand; base += tn) {
                const int next = base + tl;
                bool kept = false;
                int j = 0;
                if (next < ncand) {
                    while (next >= row_end) {
                        ++row;
                        const int beg = rw_off[row];
                        row_end = beg + rw_len[row];
                        j0 = rw_js[row] - beg;
                    }
                    j = j0 + next;
                    const double4 Pj = a.pw[j];
                    const double s = exact_s(Pa.x, Pa.y, Pa.z, Pj.x, Pj.y, Pj.z);
                    kept = s > t_lo && s < t_hi;
                    if (kept && s >= t64[nb]) {     // the reference's out-of-range bin
                        kept = false;
                        ++n_over;
                    }
                }
                const unsigned long long m = __builtin_amdgcn_ballot_w64(kept);
                int pos = K;
                if constexpr (!WAVE) {
                    int at = 0;
                    if (lane == 0 && m) at = atomicAdd(&s_k, (int)__popcll(m));
                    pos = scalar(at);
                }
                pos += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (kept && pos < KM) jl[pos] = j;
                K += (int)__popcll(m);
            }
        }
        sync();
        if constexpr (!WAVE) {
            K = scalar(s_k);
            __syncthreads();
            if (tid == 0) s_k = 0;
        }
        if (K > KM) {
            // left to the next pass, which also counts its candidates and overflows
            if (tl == 0) {
                a.ovf[atomicAdd(a.ovf_n, 1)] = apex;
                if (a.ovf_kmax) atomicMax(a.ovf_kmax, K);
            }
            sync();
            return;
        }
        cand += (unsigned)ncand;
        over += n_over;
        if (K <= (tetra ? 2 : 3)) {                 // gramsci.F90:675 (the tetrahedron query has no such skip)
            sync();
            return;
        }
        // ---- 2. thread u: neighbour u, to its place in the order of the original indices
        double4 P = make_double4(0, 0, 0, 0);
        int ku = 0x7fffffff, pk = 0;
        if (tl < K) {
            const int j = jl[tl];
            P = a.pw[j];
            ku = a.orig[j];
            pk = bin_kept(exact_s(Pa.x, Pa.y, Pa.z, P.x, P.y, P.z)) + 1;
            pk |= (int)(a.flags[j] & 1u) << 8;
        }
        if (tl < KM) key[tl] = ku;                  // from K on: above all others
        sync();
        if (tl < K) {
            int rank = 0;
            for (int j = 0; j < K; j += 4) {
                const int4 k4 = *(const int4*)&key[j];
                rank += (k4.x < ku ? 1 : 0) + (k4.y < ku ? 1 : 0) + (k4.z < ku ? 1 : 0) + (k4.w < ku ? 1 : 0);
            }
            xs[rank] = P.x; ys[rank] = P.y; zs[rank] = P.z;
            if constexpr (W) ws[rank] = P.w;
            A[rank] = (uint8_t)pk;
            rnd[rank] = (uint8_t)(pk >> 8);
        }
        sync();
        // ---- 3a. links.  The pairs u < v are numbered in folded rows of K: row r holds (r, r + 1 + c) for
        // c < K - 1 - r, then (K - 2 - r, c).
        const int np = K * (K - 1) / 2, dq = tn / K, dr = tn - dq * K, r00 = tl / K, c00 = tl - r00 * K;
        {
            int r = r00, c = c00;
            for (int pi = tl; pi < np; pi += tn) {
                const bool first = c < K - 1 - r;
                const int u = first ? r : K - 2 - r, v = first ? r + 1 + c : c;
                const double s = exact_s(xs[u], ys[u], zs[u], xs[v], ys[v], zs[v]);
                int b = -1;
                if (s > t_lo && s < t_hi) b = bin_kept(s);
                L[u * LD + v] = (uint8_t)(b >= 0 && b < nb ? b + 1 : 0);
                c += dr;
                const bool carry = c >= K;
                c -= carry ? K : 0;
                r += dq + (carry ? 1 : 0);
            }
        }
        sync();
        // ---- 3b. thread u: its row's masks
        if (tl < K) {
            const uint32_t* Lr = (const uint32_t*)(L + tl * LD);
            const uint32_t* Aw = (const uint32_t*)A;
            for (int w = 0; w < NW; ++w) {
                const int k0 = 64 * w, left = K - k0, words = min(max((left + 3) >> 2, 0), 16);
                unsigned long long above = left >= 64 ? ~0ull : (left > 0 ? (1ull << left) - 1 : 0ull);
                above &= tl < k0 ? ~0ull : (tl < k0 + 63 ? ~0ull << (tl - k0 + 1) : 0ull);
                auto mask_of = [&](auto&& pick) {
                    uint32_t lo = 0, hi = 0;
                    for (int q = 0; q < words; ++q) {
                        // bit 7 of each byte -> 4 bits
                        const uint32_t x = pick(Lr[16 * w + q], Aw[16 * w + q]);
                        const uint32_t bits = __builtin_amdgcn_udot4((x >> 7) & 0x01010101u, 0x08040201u, 0u, false);
                        if (q < 8) lo |= bits << (4 * q); else hi |= bits << (4 * (q - 8));
                    }
                    return (((unsigned long long)hi << 32) | lo) & above;
                };
                constexpr uint32_t kHigh = 0x80808080u, kOne = 0x01010101u;
                if (tetra) {
                    const uint32_t bb = A[tl] * kOne;
                    T[w * KM + tl] = mask_of([&](uint32_t x, uint32_t y) { return ~(((x ^ bb) | (y ^ bb)) + 0x7f7f7f7fu); });
                    continue;
                }
                M[w * KM + tl] = mask_of([&](uint32_t x, uint32_t) { return x + 0x7f7f7f7fu; });
                for (int b = 1; b <= (BIN ? nb : 1); ++b) {
                    const uint32_t bb = (uint32_t)b * kOne;
                    T[((b - 1) * NW + w) * KM + tl] =
                        mask_of([&](uint32_t x, uint32_t y) { return ((y | kHigh) - x) & ((x | kHigh) - bb); });
                }
            }
        }
        sync();
        // ---- 4. quads of the linked pairs
        const int ri = (int)(fa & 1u);
        {
            int r = r00, c = c00;
            for (int pi = tl; pi < np; pi += tn) {
                const bool first = c < K - 1 - r;
                const int u = first ? r : K - 2 - r, v = first ? r + 1 + c : c;
                const int ind4 = L[u * LD + v], ind1 = A[u], ind2 = A[v];
                if (ind4 && (!tetra || (ind2 == ind1 && ind4 == ind1))) {       // tetra: gramsci.F90:564-567
                    units += (unsigned)(K - 1 - v);
                    // perimeters that do not begin ind1 <= ind4 have no configuration (:701)
                    const unsigned long long* Tv = T + (BIN ? (size_t)(ind4 - 1) * NW * KM : 0);
                    const unsigned long long* Mu = (tetra ? T : M) + u;
                    if (ind4 >= ind1)
                        for (int w = NW == 1 ? 0 : (v + 1) >> 6; w < NW; ++w) {
                            unsigned long long m = Tv[w * KM + v] & Mu[w * KM];
                            while (m) {
                                const int k3 = 64 * w + (int)__builtin_ctzll(m);
                                m &= m - 1;
                                const int ind5 = L[v * LD + k3], ind6 = L[u * LD + k3], ind3 = A[k3];
                                if (!BIN && ind5 < ind4) continue;
                                const int r1 = rnd[u], r2 = rnd[v], r3 = rnd[k3];
                                int cell = ind1 - 1;
                                if (!tetra) {
                                    const int cfg = tab[(((ind1 - 1) * nb + (ind4 - 1)) * nb + (ind5 - 1)) * nb + (ind3 - 1)];
                                    cell = (cfg - 1) * nb2 + (ind2 - 1) * nb + (ind6 - 1);
                                }
                                const int pat = ri | (r1 << 1) | (r2 << 2) | (r3 << 3);
                                ++binned;
                                if (lh) atomicAdd(&hc[cell * 16 + pat], 1u);
                                else atomicAdd(&out_cnt[(size_t)cell * 16 + pat], 1ull);
                                if constexpr (W)
                                    add_quad_sums(lw ? hw : out_w, ncell, cell, pat, ri, r1, r2, r3, Pa.w, ws[u], ws[v],
                                                  ws[k3], tetra);
                            }
                        }
                }
                c += dr;
                const bool carry = c >= K;
                c -= carry ? K : 0;
                r += dq + (carry ? 1 : 0);
            }
        }
        // the u32 counts are shared by the work-group's teams; an apex adds fewer than 2^22
        bound += (unsigned)(K * (K - 1) * (K - 2) / 6);
        if (lh && bound > (1ull << 28)) {
            sync();
            drain_counts(tl, tn);
            bound = 0;
        }
        sync();
    };

    while (true) {
        if (tid < kWave) {
            const int b = items.next(lane, 0);
            if (tid == 0) s_item = b;
        }
        __syncthreads();
        const int b = scalar(s_item);
        if (b < 0) break;
        const int lo = b * bsz, hi = min(n_items, lo + bsz);
        for (int it = lo + (WAVE ? wv : 0); it < hi; it += teams) visit_apex(it);
        __syncthreads();
    }
    __syncthreads();
    if (lh) drain_counts(tid, kWG);
    if (lw)
        for (int k = opaque(tid); k < ncell * 40; k += kWG)
            if (hw[k] != 0.0) atomicAdd(&out_w[k], hw[k]);
    if (tl != 0) cand = 0;                          // kept by the team's threads alike
    __shared__ unsigned long long s_stat[5];
    if (tid < 5) s_stat[tid] = 0;
    __syncthreads();
    const unsigned long long st[5] = {cand, 0, (unsigned long long)over, units, binned};
    for (int q = 0; q < 5; ++q) {
        unsigned long long v = st[q];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if (lane == 0 && v) atomicAdd(&s_stat[q], v);
    }
    __syncthreads();
    if (tid < 5 && s_stat[tid]) atomicAdd(&a.out_stats[copy + tid], s_stat[tid]);
}

template <bool BIN>
static void (*quad_kernel_lds(const QuadArgs& a, bool weighted, bool wave))(QuadArgs)
{
    if (wave) return k_quad4<false, 1, true, BIN>;      // unit weights
    if (a.kmax <= 64) return weighted ? k_quad4<true, 1, false, BIN> : k_quad4<false, 1, false, BIN>;
    if (a.kmax <= 128) return weighted ? k_quad4<true, 2, false, BIN> : k_quad4<false, 2, false, BIN>;
    return weighted ? k_quad4<true, 4, false, BIN> : k_quad4<false, 4, false, BIN>;
}

static void (*quad_kernel(const QuadArgs& a, bool weighted, bool wave))(QuadArgs)
{
    if (a.glist) return weighted ? k_quad4_big<true> : k_quad4_big<false>;
    return a.bin_masks ? quad_kernel_lds<true>(a, weighted, wave) : quad_kernel_lds<false>(a, weighted, wave);
}

size_t quad4_lds_bytes(const QuadArgs& a, int nb, bool weighted, bool wave)
{
    return quad_lds(a, nb, weighted, a.kmax, wave ? kWG / kWave : 1, a.glist != nullptr).total;
}

hipError_t launch_quad4(const QuadArgs& a, int nb, bool weighted, bool wave, int nblocks, hipStream_t st)
{
    const size_t lds = quad4_lds_bytes(a, nb, weighted, wave);
    auto kern = quad_kernel(a, weighted, wave);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(kWG), lds, st, a);
    return hipGetLastError();
}

int quad4_occupancy(const QuadArgs& a, int nb, bool weighted, bool wave)
{
    const size_t lds = quad4_lds_bytes(a, nb, weighted, wave);
    auto kern = quad_kernel(a, weighted, wave);
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return 1;
    int n = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, kWG, lds);
    return (e == hipSuccess && n > 0) ? n : 1;
}

// sums the copies of n doubles
__global__ __launch_bounds__(256) void k_sum_copies_f64(const double* __restrict__ in, int copies, int64_t stride, int64_t n,
                                                        double* __restrict__ out)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t e = blockIdx.x * (int64_t)(blockDim.x / kWave) + threadIdx.x / kWave;
    if (e >= n) return;
    double v = lane < copies ? in[(size_t)lane * (size_t)stride + e] : 0.0;
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) out[e] = v;
}

hipError_t launch_sum_copies_f64(const double* in, int copies, int64_t stride, int64_t n, double* out, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sum_copies_f64, dim3((unsigned)((n + kWG / kWave - 1) / (kWG / kWave))), dim3(kWG), 0, st, in, copies,
                       stride, n, out);
    return hipGetLastError();
}

}  // namespace gs
