// pcf34.cpp -- C ABI for the 3PCF and 4PCF paths (gs_count_3pcf, gs_count_3pcf_equi,
// gs_count_4pcf, gs_count_4pcf_tetra):
// grid, stencil, configuration tables, kernel launch and the host-side
// combination of exact class counts / sums into the reference's N2, N3,
// discN, discR.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "gs_api_internal.h"
#include "gs_kernels.h"

using namespace gs;

namespace gs {

void extra_release(GsExtra& x)
{
    x.params.release();
    x.out.release();
    x.queue.release();
    x.dbl.release();
    x.i32.release();
    x.big.release();
    x.big_zero.release();
}

// bintable for the 3PCF (gramsci.F90:1459-1474), 0-based configuration of a
// sorted triple in the i <= j <= k enumeration, for every permutation.
std::vector<uint16_t> table3(int nb)
{
    std::vector<uint16_t> t((size_t)nb * nb * nb, 0);
    int cfg = 0;
    for (int i = 0; i < nb; ++i)
        for (int j = i; j < nb; ++j)
            for (int k = j; k < nb; ++k) {
                const int p[6][3] = {{i, j, k}, {i, k, j}, {j, i, k}, {j, k, i}, {k, i, j}, {k, j, i}};
                for (auto& q : p) t[((size_t)q[0] * nb + q[1]) * nb + q[2]] = (uint16_t)cfg;
                ++cfg;
            }
    return t;
}

// The triplet kernel's table: 4 * configuration (the histogram index of the configuration's class 0).
// Empty when 4 * configurations does not fit 16 bits (then the table would not fit in LDS either).
std::vector<uint16_t> table3_hist(int nb)
{
    const long ncfg = (long)nb * (nb + 1) * (nb + 2) / 6;
    if (4 * ncfg > 65535) return {};
    std::vector<uint16_t> t = table3(nb);
    for (auto& x : t) x = (uint16_t)(4 * x);
    return t;
}

// bintable for the 4PCF (gramsci.F90:1402-1420): 1-based configuration for
// non-decreasing quadruples only, 0 elsewhere.
static std::vector<uint16_t> table4(int nb)
{
    std::vector<uint16_t> t((size_t)nb * nb * nb * nb, 0);
    int cfg = 0;
    for (int i = 0; i < nb; ++i)
        for (int j = i; j < nb; ++j)
            for (int k = j; k < nb; ++k)
                for (int l = k; l < nb; ++l) t[(((size_t)i * nb + j) * nb + k) * nb + l] = (uint16_t)(++cfg);
    return t;
}

static void fill_stats(gs_stats* st, hipEvent_t* ev, const unsigned long long* s, int m)
{
    if (!st) return;
    memset(st, 0, sizeof(*st));
    float ms_grid = 0, ms_count = 0;
    (void)hipEventElapsedTime(&ms_grid, ev[0], ev[1]);
    (void)hipEventElapsedTime(&ms_count, ev[2], ev[3]);
    st->ms_grid = ms_grid;
    st->ms_count = ms_count;
    st->ms_kernel_avg = ms_count;
    st->n_candidates = s[0];
    st->n_recheck = s[1];
    st->n_overflow = s[2];
    st->n_units = s[3];
    st->n_binned = s[4];
    st->n_evaluated = s[3];
    st->cell_div = m;
}

}  // namespace gs

// ====================================================================== 3PCF

namespace gs {

// find_normal (gramsci.F90:1611-1625) tabulated over its two int8 arguments,
// 0-based: mu11/mu22 are default reals (mu1-0.5 in single precision, the
// division by the double mu_scale and "- 1.0" in double, rounded to single on
// assignment), the rest of the expression is single precision left to right,
// and floor()+1 is stored in an int8 before the clamp.  A negative radicand
// (NaN) ends in bin 1 whatever integer its floor converts to.
std::vector<uint8_t> normal_table(int nm)
{
    std::vector<uint8_t> t((size_t)nm * nm, 0);
    const double mu_scale = (double)(0.5f * (float)nm);
    for (int a = 1; a <= nm; ++a)
        for (int b = 1; b <= nm; ++b) {
            const float x = (float)((double)((float)a - 0.5f) / mu_scale - 1.0);
            const float y = (float)((double)((float)b - 0.5f) / mu_scale - 1.0);
            volatile float r = 0.75f - x * x;
            r = r - y * y;
            r = r + x * y;
            int v = 1;
            if (r >= 0.0f) {
                volatile float q = 1.1547f * std::sqrt((float)r);
                q = q * (float)nm;
                v = (int)(int8_t)((int)std::floor((float)q) + 1);
                v = v < 1 ? 1 : (v > nm ? nm : v);
            }
            t[(size_t)(a - 1) * nm + (b - 1)] = (uint8_t)(v - 1);
        }
    return t;
}

// LDS plan of the triplet kernel for a.ncfg/a.nm: histogram replicas and
// neighbour capacity within 64 KiB; a histogram too large for LDS goes to
// global atomics instead.
int triplet_wg(double list, bool rsd, bool weighted)
{
    const char* ev = getenv("GS_T3_WG");        // tuning override (unset or empty: automatic)
    if (ev && *ev) {
        const int w = atoi(ev);
        if (w == 64 || w == 128 || w == 256) return w;
    }
    // Measured over uniform catalogues, in ms for 64, 128 and 256 threads.  Lists of 16: mu bins and weights 0.81,
    // 0.73, 1.12, mu bins alone 0.56, 0.69, 1.08, weights alone (32 neighbours) 0.74, 0.76, 1.12.  Lists of 64: 2.32,
    // 1.70, 1.99; 1.33, 1.40, 1.66; 0.88, 0.79, 0.88.  Lists of 128: 2.48, 1.76, 1.74; 1.67, 1.22, 1.29; 0.84, 0.64,
    // 0.63.  Lists of 256: 2.43, 1.58, 1.33 and so on.  (Before the kernel queued its pairs; since, mu bins and weights,
    // lists of 110: 2.21, 1.70, 1.80.)
    if (list < 24.0 && !(rsd && weighted)) return 64;
    return list < 120.0 ? 128 : 256;
}

// With teams of one wave, up to 8 apexes a team between the barriers of a fetch, as long as every work-group gets a
// batch (3,000 points on cells of rmax / 16, 965 stencil rows: batches of 32 0.70 ms, 94 of 750 work-groups; of 4 0.22).
int triplet_batch(int64_t n, int nblocks, int teams)
{
    const int64_t nb = std::max(nblocks, 1);
    const int least = teams > 1 ? teams * (int)std::max<int64_t>(1, std::min<int64_t>(8, n / (teams * nb))) : 1;
    const char* ev = getenv("GS_APEX_BATCH");   // tuning override (unset or empty: automatic)
    if (ev && *ev) return std::max(least, std::min(64, atoi(ev)));
    return std::max(least, (int)std::min<int64_t>(16, n / (128 * nb)));
}

int plan_triplet_lds(TripArgs& a, int nb, bool fp64, bool weighted)
{
    const size_t nh = (size_t)a.ncfg * a.nm * 4;
    const size_t budget = 64 * 1024;
    // (without the queues, and with bin tables at their largest: what fits does not depend on either)
    const size_t tables = (size_t)(2 * (kMaxBins - nb)) * 8;
    auto lds = [&]() {
        return triplet3_lds_bytes(a, nb, fp64, weighted) - triplet3_queue_bytes(a, weighted) + tables;
    };
    a.lds_hist = 1;
    a.reps = 1;
    // replicas up to 4 KiB: the LDS is better spent on work-groups (100k + 200k points, 5 bins, 6 mu bins, 128
    // threads: 16 KiB of replicas 1.75 ms, 4 KiB 1.59; weights, 4 mu bins, 90k points: 4 KiB 1.71, 12 KiB 1.69, 24 KiB
    // 2.13, and weights, equal sides, 117k points: 1.14, 1.47, 1.46)
    while (a.reps < 32 && nh * a.reps * 2 * (weighted ? 16 : 4) <= 4 * 1024) a.reps *= 2;
    a.kmax = 4096;
    while (a.kmax > 512 && lds() > budget) a.kmax -= 256;
    while (a.reps > 1 && lds() > budget) a.reps /= 2;
    if (lds() > budget) {
        a.lds_hist = 0;
        a.reps = 1;
        a.kmax = 4096;
        while (a.kmax > 256 && lds() > budget) a.kmax -= 256;
    }
    if (lds() > budget) return fail(GS_ELIMIT, "3PCF tables do not fit in LDS");
    return GS_OK;
}

// Long lists (more than 256 entries) leave few work-groups a compute unit: more replicas of a weighted histogram, as
// far as the same number of work-groups stays (4 bins, 3 mu bins, ms: 10,000 points with 1,000 neighbours 7.5 -> 6.7;
// 20,000 with 300 1.46 -> 1.30; not below: with 100 0.286 -> 0.297, nor without weights: 1.07 -> 1.15 with 300).
void triplet_replicas(TripArgs& a, int nb, bool fp64, int occ)
{
    if (!a.lds_hist || a.kmax <= 256) return;
    while (a.reps < 32) {
        a.reps *= 2;
        if (triplet3_lds_bytes(a, nb, fp64, true) * std::max(occ, 1) <= 160 * 1024) continue;
        a.reps /= 2;
        break;
    }
}

std::vector<uint32_t> cfg_bins3(int nb)
{
    std::vector<uint32_t> t;
    for (int i = 0; i < nb; ++i)
        for (int j = i; j < nb; ++j)
            for (int k = j; k < nb; ++k) t.push_back((uint32_t)(i | j << 8 | k << 16));
    return t;
}

bool plan_triplet_matrix(TripArgs& a, int nb, bool buf)
{
    a.buf = buf ? 1 : 0;
    a.reps = 2;
    const size_t hist = (size_t)nb * nb * (nb + 2) * 4 * (buf ? 3 : 1) * 4;
    if (hist > 32 * 1024) return false;     // beyond: the general kernel, whose histogram holds configurations
    // replicas up to 12 KiB: more of them leave the LDS room for fewer work-groups (200k + 400k points, 5 bins: 2, 4,
    // 8 replicas 11.1, 11.0, 13.4 ms; 16 regions, 4 bins, buffer points: 2 replicas 3.2, 4 4.8 ms)
    while (a.reps < 16 && hist * a.reps * 2 <= 12 * 1024) a.reps *= 2;
    a.kmax = 4096;
    while (a.kmax > 64 && triplet_matrix_lds(a, nb, 1) > 150 * 1024) a.kmax -= 64;
    return triplet_matrix_lds(a, nb, 1) <= 150 * 1024;
}

// One wave per apex while four lists leave the LDS room for several work-groups, up to 256 entries (16 regions of 60k
// points, lists of 128: 3.6 ms, with work-groups of 256 6.4); a work-group beyond (lists of 512: 11.5 against 20.6 ms).
bool triplet_matrix_team(TripArgs& a, int nb, int kmax1, int wg)
{
    a.kmax = kmax1;
    const char* ev = getenv("GS_T3_WG");        // tuning override (unset or empty: automatic)
    if (ev && *ev && (atoi(ev) == 64 || atoi(ev) == 128 || atoi(ev) == 256)) wg = atoi(ev);
    const bool wave = (wg > 0 ? wg == 64 : kmax1 <= 256) && triplet_matrix_lds(a, nb, kWG / kWave) <= 150 * 1024;
    a.wg = wave ? kWG : (wg > 0 ? wg : (triplet_matrix_lds(a, nb, 1) > 40 * 1024 ? 512 : kWG));
    return wave;
}

// The last pass of the 3PCF: apexes whose neighbours outnumber every LDS list were queued
// (d_list); they run here with their
// neighbour lists in device memory, one list per work-group, and the histogram in global
// memory.  h is the count (positive) and the largest neighbour count.
// `base` carries the pass's tables and outputs; d_queue is an ItemQueue's counters, which it clears.
int triplet_glist_pass(const TripArgs& base, int nb, bool fp64, bool weighted, const int32_t* d_list, const int32_t h[2],
                       int32_t* d_queue, DevBuf<unsigned char>& scratch, int n_cu, hipStream_t st)
{
    hipError_t e;
    TripArgs a = base;
    a.items = d_list;
    a.n_items = h[0];
    a.n_items_dev = nullptr;
    a.ovf = nullptr;
    a.ovf_n = nullptr;
    a.ovf_kmax = nullptr;
    a.kmax = (std::max(h[1], 2) + 3) / 4 * 4;       // every list holds its apex's neighbours
    a.wg = kWG;
    a.batch = 1;
    a.queue = d_queue;
    const size_t stride = (a.kmax * triplet3_glist_entry_bytes(a, fp64, weighted) + 255) / 256 * 256;
    a.glist = (void*)d_list;        // selects the device-memory variant (LDS sizes and occupancy query)
    // the LDS holds no list here: the histogram stays in LDS (replicated) where it fits
    a.lds_hist = 1;
    a.reps = 1;
    const size_t nh = (size_t)a.ncfg * (a.nm > 1 ? a.nm : 1) * 4;
    while (a.reps < 32 && nh * a.reps * 2 * 4 <= 16 * 1024) a.reps *= 2;
    while (a.reps > 1 && triplet3_lds_bytes(a, nb, fp64, weighted) > 64 * 1024) a.reps /= 2;
    if (triplet3_lds_bytes(a, nb, fp64, weighted) > 64 * 1024) a.lds_hist = 0;
    const int occ = triplet3_occupancy(a, nb, fp64, weighted);
    const size_t budget = (size_t)1 << 30;           // device memory for the lists of concurrent apexes
    const int nblk = (int)std::max<size_t>(1, std::min<size_t>({(size_t)h[0], (size_t)n_cu * occ, budget / stride}));
    int rc = scratch.reserve((size_t)nblk * stride);
    if (rc) return rc;
    a.glist = scratch.ptr;
    a.glist_stride = (int64_t)stride;
    e = launch_fill_u32(d_queue, 64 * kQueuePad, 0u, st);
    if (e == hipSuccess) e = launch_triplet3(a, nb, fp64, weighted, nblk, st);
    if (e != hipSuccess) return hip_fail(e, "3PCF device-memory pass");
    return GS_OK;
}

// N2/N3 of the 3PCF from the class sums S[q][4] (q = configuration x mu bin):
// N2 = sum over classes of (-1)^r S_r / (Wd^(3-r) Wr^r) (gramsci.F90:501, :507, :431, :437);
// N3 = S_3 / Wr^3 (:498, :505, :434) unless with_n3 is false (the equilateral RSD
// branch accumulates no N3, :429-431)
void combine3(const long double* S, int nq, long double Wd, long double Wr, bool with_n3, double* n2, double* n3)
{
    for (int q = 0; q < nq; ++q) {
        long double v2 = 0, v3 = 0;
        for (int r = 0; r <= 3; ++r) {
            const long double sv = S[q * 4 + r];
            if (sv == 0) continue;
            long double den = 1;
            for (int t = 0; t < 3 - r; ++t) den *= Wd;
            for (int t = 0; t < r; ++t) den *= Wr;
            v2 += ((r & 1) ? -sv : sv) / den;
        }
        if (with_n3 && Wr > 0) v3 = S[q * 4 + 3] / (Wr * Wr * Wr);
        if (n2) n2[q] = (double)v2;
        if (n3) n3[q] = (double)v3;
    }
}

// The kept-neighbour counts of nsample apexes (none: of buffer points) spread over n, in d_out (2 nsample).  *gather: the
// apexes have so many candidates that finding the neighbours is the work, as where a few outlying points widen the
// cells (a box of 20 with one point at 5,000, 30,000 points, 150 neighbours: matrix kernel 1.75 ms, general kernel 1.35;
// 4,000 points, 40 neighbours: 0.051 and 0.073).
static int sample_neighbours(const TripArgs& a, int n, int nsample, int after_only, int32_t* d_out, hipStream_t st,
                             std::vector<int32_t>& ks, bool* gather)
{
    if (nsample <= 0) return GS_OK;
    std::vector<int32_t> h(2 * (size_t)nsample);
    hipError_t e = launch_nbr_count(a, n / nsample, nsample, after_only, d_out, st);
    if (e == hipSuccess) e = hipMemcpyAsync(h.data(), d_out, h.size() * sizeof(int32_t), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_fail(e, "neighbour sample");
    double cand = 0.0;
    for (int t = 0; t < nsample; ++t)
        if (h[t] >= 0) {
            ks.push_back(h[t]);
            cand += h[nsample + t];
        }
    *gather = cand > 8192.0 * (double)ks.size();
    return GS_OK;
}

// Shared body of gs_count_3pcf (all configurations) and gs_count_3pcf_equi.
static int count3(gs_ctx* c, const gs_params* p, bool equi, uint64_t* cnt, double* wsum, double* n2, double* n3,
                  gs_stats* st)
{
    if (!c) return fail(GS_EINVAL, "NULL context");
    int rc = check_params(p, 3);
    if (rc) return rc;
    if ((rc = ctx_set_device(c))) return rc;
    const int nb = p->nbins, nm = p->nmu;
    const int ncfg = equi ? nb : nb * (nb + 1) * (nb + 2) / 6;
    const int nh = ncfg * nm * 4;
    const bool fp64 = p->precision == GS_FP64;
    CtxView v = view(c);
    const bool weighted = v.has_w;
    const int m = p->cell_div > 0 ? p->cell_div : 2;
    const int sx = apex_cell_sx();

    (void)hipEventRecord(v.ev[0], v.stream);
    double h;
    if ((rc = ctx_build_grid(c, p->rmax, m, sx, &h))) return rc;
    (void)hipEventRecord(v.ev[1], v.stream);
    v = view(c);
    const int mst = (int)std::ceil(p->rmax / h - 1e-12);
    std::vector<Row> rows = full_stencil(h, h / sx, p->rmax, mst);
    BinDesc B;
    double t64[kMaxBins + 2];
    if ((rc = ctx_thresholds(c, *p, t64)) || (rc = fill_bins(*p, t64, 1.5 * p->rmax, ctx_xmax(c), v.wmax_d, v.wmax_r, B))) return rc;
    std::vector<uint16_t> tab = equi ? std::vector<uint16_t>() : table3_hist(nb);
    if (!equi && tab.empty()) return fail(GS_ELIMIT, "3PCF with %d bins: configuration table too large", nb);
    std::vector<uint8_t> ntab = nm > 1 ? normal_table(nm) : std::vector<uint8_t>();

    TripArgs a{};
    a.ncfg = ncfg;
    a.nm = nm;
    a.log_bins = p->log_bins != 0;
    a.equi = equi ? 1 : 0;
    a.nrows = (int)rows.size();      // the LDS plan holds the stencil rows' table
    if ((rc = plan_triplet_lds(a, nb, fp64, weighted))) return rc;
    // FP32 counts of unit weights without mu bins: third sides from the matrix cores (am); its passes are the
    // general kernel's, which also takes the apexes whose lists fit no LDS
    TripArgs am = a;
    bool mat = !equi && nm == 1 && !fp64 && !weighted && plan_triplet_matrix(am, nb, v.has_buf);
    const std::vector<uint32_t> cfgb = mat ? cfg_bins3(nb) : std::vector<uint32_t>();

    // Parameters in one copy from pinned memory.  One region to clear: the work counters of two passes, the error
    // flag, the counts of queued apexes, and the outputs' copies; their sum goes to pinned memory.
    GsExtra& X = *v.extra;
    HostBuf& H = ctx_host(c);
    const size_t tab_off = (sizeof(BinDesc) + 15) / 16 * 16;
    const size_t ntab_off = tab_off + (tab.size() * 2 + 15) / 16 * 16;
    const size_t mat_off = ntab_off + (ntab.size() + 15) / 16 * 16;
    const size_t cfgb_off = mat_off + (mat ? (sizeof(TripMatrix) + 15) / 16 * 16 : 0);
    const size_t rows_off = cfgb_off + (cfgb.size() * 4 + 15) / 16 * 16;
    const size_t blob = rows_off + rows.size() * sizeof(Row), res_off = (blob + 255) / 256 * 256;
    const int64_t words = triplet_copy_words(nh);
    const int copies = output_copies(words);
    constexpr size_t kQueueInts = 64 * kQueuePad, kHeadInts = 2 * kQueueInts + 64;
    const size_t clear = kHeadInts * 4 + (size_t)copies * words * 8;
    if ((rc = X.params.reserve(blob)) || (rc = X.big_zero.reserve(clear)) || (rc = H.reserve(res_off + words * 8 + 16)))
        return rc;
    *(BinDesc*)H.ptr = B;
    std::copy(tab.begin(), tab.end(), (uint16_t*)(H.ptr + tab_off));
    std::copy(ntab.begin(), ntab.end(), H.ptr + ntab_off);
    std::copy(rows.begin(), rows.end(), (Row*)(H.ptr + rows_off));
    if (mat) fill_triplet_matrix(*p, t64, v.g.h, v.g.hx, *(TripMatrix*)(H.ptr + mat_off));
    std::copy(cfgb.begin(), cfgb.end(), (uint32_t*)(H.ptr + cfgb_off));
    hipError_t e = hipMemcpyAsync(X.params.ptr, H.ptr, blob, hipMemcpyHostToDevice, v.stream);
    if (e == hipSuccess) e = launch_fill_u32(X.big_zero.ptr, (int64_t)clear / 4, 0u, v.stream);
    if (e != hipSuccess) return hip_fail(e, "3PCF parameter upload");
    int32_t* const head = (int32_t*)X.big_zero.ptr;
    int32_t* const d_cnt2 = head + 2 * kQueueInts + 16;     // second-pass apexes
    int32_t* const d_cnt3 = head + 2 * kQueueInts + 32;     // last-pass apexes, their largest neighbour count, the error flag
    unsigned long long* const out = (unsigned long long*)(head + kHeadInts);

    a.pw = v.pw;
    a.flags = v.flags;
    a.orig = v.orig;
    a.cell_start = v.cell_start;
    a.rows = (const Row*)(X.params.ptr + rows_off);
    a.bins = (const BinDesc*)X.params.ptr;
    a.cfg_tab = tab.empty() ? nullptr : (const uint16_t*)(X.params.ptr + tab_off);
    a.ntab = ntab.empty() ? nullptr : (const uint8_t*)(X.params.ptr + ntab_off);
    a.queue = head;
    a.err = d_cnt3 + 2;
    a.out_cnt = out;
    a.out_w = out + nh;
    a.out_stats = out + 3 * nh;
    a.copies = copies;
    a.copy_stride = words;
    a.g = v.g;
    a.g.m = mst;
    a.nrows = (int)rows.size();
    const int n = (int)(v.n_data + v.n_rand);
    a.n_items = n;
    a.matrix = (const TripMatrix*)(X.params.ptr + mat_off);
    a.cfg_bins = (const uint32_t*)(X.params.ptr + cfgb_off);
    if (mat) {
        const int reps = am.reps, kmax = am.kmax, buf = am.buf;
        am = a;
        am.reps = reps;
        am.kmax = kmax;
        am.buf = buf;
    }

    // Two passes.  The neighbour list in LDS bounds the work-groups a CU can hold, so the
    // first pass sizes it for the 99.5th percentile of the neighbour counts of ~2048
    // sampled apexes (+5%) and hands every apex with more neighbours to a second pass over
    // just those apexes, with the largest list that fits.  An apex is counted in exactly
    // one pass, so the sums are those of one pass.
    // An apex whose neighbours outnumber even the second pass's list is queued once more, for a
    // last pass with its list in device memory (triplet_glist_pass): no neighbour count is refused.
    // Without a matrix kernel where the gather is the work: its lists leave fewer waves than the general kernel's.
    const int nsample = std::min(n, 2048);
    // i32: second-pass apexes, last-pass apexes, the sample
    if ((rc = X.i32.reserve(2 * (size_t)n + 2 * nsample))) return rc;
    int32_t* d_list2 = X.i32.ptr;
    int32_t* d_list3 = X.i32.ptr + n;
    std::vector<int32_t> ks;
    bool gather = false;
    if ((rc = sample_neighbours(a, n, nsample, nm > 1 ? 0 : 1, X.i32.ptr + 2 * (size_t)n, v.stream, ks, &gather))) return rc;
    if (gather) mat = false;
    const int kmax_full = mat ? am.kmax : a.kmax;
    int kmax1 = kmax_full;
    if (nsample > 0) {
        double ksum = 0.0;
        for (int32_t k : ks) ksum += k;
        if (!ks.empty()) {
            a.wg = triplet_wg(ksum / (double)ks.size(), nm > 1, weighted);
            const size_t q = std::min(ks.size() - 1, (size_t)std::ceil(0.995 * (ks.size() - 1)));
            std::nth_element(ks.begin(), ks.begin() + q, ks.end());
            const int k995 = ks[q];
            kmax1 = std::min(kmax_full, std::max(128, (int)std::ceil(1.05 * k995 / 64.0) * 64));
        }
    }
    {
        const char* ev = getenv("GS_T3_KMAX");      // tuning override (unset or empty: automatic)
        if (ev && *ev) kmax1 = std::max(64, std::min(kmax_full, atoi(ev)));
    }
    {
        const char* ev = getenv("GS_T3_KMAX_LDS");  // test override: a shorter second-pass list
        if (ev && *ev) {
            a.kmax = std::max(64, std::min(a.kmax, atoi(ev)));
            am.kmax = std::max(64, std::min(am.kmax, atoi(ev) / 64 * 64));
            kmax1 = std::min(kmax1, mat ? am.kmax : a.kmax);
        }
    }
    if (mat) kmax1 = std::max(64, kmax1 / 64 * 64);
    const bool two_pass = kmax1 < (mat ? am.kmax : a.kmax);
    (void)hipEventRecord(v.ev[2], v.stream);
    if (n > 0) {
        auto launch = [&](TripArgs& t, bool wave, int most) {
            const int occ = mat ? triplet_matrix_occupancy(t, nb, wave) : triplet3_occupancy(t, nb, fp64, weighted);
            const int teams = wave ? t.wg / kWave : 1;
            const int nblk = std::max(1, std::min(v.n_cu * std::max(occ, 1), (most + teams - 1) / teams));
            if (!mat && weighted) triplet_replicas(t, nb, fp64, occ);
            if (t.batch == 0) t.batch = triplet_batch(n, nblk, teams);
            return mat ? launch_triplet_matrix(t, nb, wave, nblk, v.stream)
                       : launch_triplet3(t, nb, fp64, weighted, nblk, v.stream);
        };
        TripArgs a1 = mat ? am : a;
        bool wave = false;
        a1.ovf_kmax = d_cnt3 + 1;
        a1.ovf = two_pass ? d_list2 : d_list3;
        a1.ovf_n = two_pass ? d_cnt2 : d_cnt3;
        if (two_pass) a1.kmax = kmax1;
        if (mat) wave = triplet_matrix_team(a1, nb, a1.kmax, 0);
        e = launch(a1, wave, n);
        if (e != hipSuccess) return hip_fail(e, "3PCF kernel launch");
        if (two_pass) {
            // the second pass, over the apexes with the most neighbours, reads their number on the device
            TripArgs a2 = mat ? am : a;
            a2.items = d_list2;
            a2.n_items_dev = d_cnt2;
            a2.wg = mat ? 2 * kWG : kWG;
            a2.batch = 1;
            a2.queue = head + kQueueInts;
            a2.ovf = d_list3;
            a2.ovf_n = d_cnt3;
            a2.ovf_kmax = d_cnt3 + 1;
            e = launch(a2, false, n);
            if (e != hipSuccess) return hip_fail(e, "3PCF second pass");
        }
    }
    // The sums of the copies and the counters to pinned memory; once more after a last pass.  Written there word by word
    // also where they are large (20 bins, 40 mu bins, 6 MB: 2.5 ms a call; one copy fetched into pageable memory 3.5).
    unsigned long long* const h_out = (unsigned long long*)(H.ptr + res_off);
    int32_t* const h_cnt = (int32_t*)(h_out + words);
    int32_t err = 0;
    for (int pass = 0;; ++pass) {
        (void)hipEventRecord(v.ev[3], v.stream);
        e = launch_sum_copies(out, copies, words, nh, nh, 8, h_out, v.stream);
        if (e == hipSuccess) e = hipMemcpyAsync(h_cnt, d_cnt3, 3 * sizeof(int32_t), hipMemcpyDeviceToHost, v.stream);
        if (e == hipSuccess) e = hipStreamSynchronize(v.stream);
        if (e != hipSuccess) return hip_fail(e, "3PCF kernel");
        err = h_cnt[2];
        if (pass > 0 || h_cnt[0] <= 0) break;
        if ((rc = triplet_glist_pass(a, nb, fp64, weighted, d_list3, h_cnt, head, X.big, v.n_cu, v.stream))) return rc;
    }
    if (err) return fail(GS_EHIP, "3PCF: an apex's neighbour list overflowed with no later pass (internal error)");

    std::vector<long double> S(nh);
    for (int k = 0; k < nh; ++k) {
        if (cnt) cnt[k] = h_out[k];
        S[k] = weighted ? fx_value(h_out[nh + 2 * k], h_out[nh + 2 * k + 1], B.fx_shift3) : (long double)h_out[k];
        if (wsum) wsum[k] = (double)S[k];
    }
    combine3(S.data(), ncfg * nm, v.wsum_d, v.wsum_r, !(equi && nm > 1), n2, n3);
    fill_stats(st, v.ev, h_out + 3 * nh, mst);
    if (st) {
        st->n_evaluated = h_out[3 * nh + 4];
        st->n_binned = 0;           // the binned triplets are the counts' total
        for (int k = 0; k < nh; ++k) st->n_binned += h_out[k];
    }
    return GS_OK;
}

}  // namespace gs

extern "C" int gs_count_3pcf(gs_ctx* c, const gs_params* p, uint64_t* cnt, double* wsum, double* n2, double* n3,
                             gs_stats* st)
{
    return count3(c, p, false, cnt, wsum, n2, n3, st);
}

extern "C" int gs_count_3pcf_equi(gs_ctx* c, const gs_params* p, uint64_t* cnt, double* wsum, double* n2,
                                  double* n3, gs_stats* st)
{
    return count3(c, p, true, cnt, wsum, n2, n3, st);
}

// ====================================================================== 4PCF

namespace gs {

// Shared body of gs_count_4pcf (perimeter configurations) and gs_count_4pcf_tetra.
static int count4(gs_ctx* c, const gs_params* p, bool tetra, uint64_t* cnt, double* n2, double* n3, double* disc_n,
                  double* disc_r, gs_stats* st)
{
    if (!c) return fail(GS_EINVAL, "NULL context");
    int rc = check_params(p, 4);
    if (rc) return rc;
    if ((rc = ctx_set_device(c))) return rc;
    const int nb = p->nbins;
    if (!tetra && nb > 16) return fail(GS_ELIMIT, "4PCF supports nbins <= 16 (got %d)", nb);
    const int ncfg = tetra ? nb : nb * (nb + 1) * (nb + 2) * (nb + 3) / 24;
    const int ncell = tetra ? nb : ncfg * nb * nb;
    CtxView v = view(c);
    const bool weighted = v.has_w;
    const int m = p->cell_div > 0 ? p->cell_div : 2;
    const int sx = apex_cell_sx();

    (void)hipEventRecord(v.ev[0], v.stream);
    double h;
    if ((rc = ctx_build_grid(c, p->rmax, m, sx, &h))) return rc;
    (void)hipEventRecord(v.ev[1], v.stream);
    v = view(c);
    const int mst = (int)std::ceil(p->rmax / h - 1e-12);
    std::vector<Row> rows = full_stencil(h, h / sx, p->rmax, mst);
    BinDesc B;
    double t64[kMaxBins + 2];
    if ((rc = ctx_thresholds(c, *p, t64)) || (rc = fill_bins(*p, t64, 1.5 * p->rmax, ctx_xmax(c), v.wmax_d, v.wmax_r, B))) return rc;
    std::vector<uint16_t> tab = tetra ? std::vector<uint16_t>() : table4(nb);

    // LDS plan of the last LDS pass: the longest list (64, 128 or 256, with its K x K matrix of links and the fewest
    // masks) that fits gfx950's 160 KiB of LDS per work-group beside the tables and, where it fits in 16 KiB, the count
    // histogram: 256 up to 14 bins (tetrahedra: always), 128 above.  Apexes with more neighbours go to a last pass with
    // device-memory lists, so no neighbour count is refused.
    const size_t budget = 160 * 1024 - 256;     // less the kernel's static part
    QuadArgs a{};
    a.tetra = tetra ? 1 : 0;
    a.ncell = ncell;
    a.nrows = (int)rows.size();
    a.lds_hist = (size_t)ncell * 64 <= 16 * 1024;
    auto fits = [&]() { return quad4_lds_bytes(a, nb, weighted, false) <= budget; };
    for (int pass = 0; pass < 2; ++pass) {
        a.kmax = 256;
        while (a.kmax > 64 && !fits()) a.kmax /= 2;
        if (fits()) break;
        a.lds_hist = 0;
    }
    if (!fits()) return fail(GS_ELIMIT, "4PCF tables do not fit in LDS");
    {
        const char* ev = getenv("GS_T4_KMAX_LDS");  // test override: a shorter second-pass list
        if (ev && *ev)
            while (a.kmax > 64 && a.kmax > atoi(ev)) a.kmax /= 2;
    }
    const int kmax = a.kmax;

    // As for the 3PCF: parameters in one copy, one region to clear (the work counters of the passes, the error flag
    // and counts of queued apexes, the outputs' copies: up to 16 MiB of them, since weighted sums that do not fit
    // LDS go there pair by pair).
    GsExtra& X = *v.extra;
    HostBuf& H = ctx_host(c);
    const size_t tab_off = (sizeof(BinDesc) + 15) / 16 * 16;
    const size_t rows_off = tab_off + (tab.size() * 2 + 15) / 16 * 16;
    const size_t blob = rows_off + rows.size() * sizeof(Row), res_off = (blob + 255) / 256 * 256;
    const size_t ncnt = (size_t)ncell * 16;
    const size_t nw = weighted ? (size_t)ncell * 16 + (size_t)6 * ncell * 4 : 0;
    const int64_t words = (int64_t)(ncnt + 8 + nw);
    int copies = 1;
    while (copies < 64 && 2 * copies * words <= (int64_t)2 << 20) copies *= 2;
    constexpr int kPasses = 3;
    constexpr size_t kQueueInts = 64 * kQueuePad, kHeadInts = kPasses * kQueueInts + 64;
    const size_t clear = kHeadInts * 4 + (size_t)copies * words * 8;
    if ((rc = X.params.reserve(blob)) || (rc = X.big_zero.reserve(clear)) || (copies > 1 && (rc = X.out.reserve(words))) ||
        (rc = H.reserve(res_off + 64)))
        return rc;
    *(BinDesc*)H.ptr = B;
    std::copy(tab.begin(), tab.end(), (uint16_t*)(H.ptr + tab_off));
    std::copy(rows.begin(), rows.end(), (Row*)(H.ptr + rows_off));
    hipError_t e = hipMemcpyAsync(X.params.ptr, H.ptr, blob, hipMemcpyHostToDevice, v.stream);
    if (e == hipSuccess) e = launch_fill_u32(X.big_zero.ptr, (int64_t)clear / 4, 0u, v.stream);
    if (e != hipSuccess) return hip_fail(e, "4PCF parameter upload");
    int32_t* const head = (int32_t*)X.big_zero.ptr;
    int32_t* const d_cnt = head + kPasses * kQueueInts;     // per pass 4: apexes queued for the next, their largest count
    unsigned long long* const out = (unsigned long long*)(head + kHeadInts);

    a.pw = v.pw;
    a.flags = v.flags;
    a.orig = v.orig;
    a.cell_start = v.cell_start;
    a.rows = (const Row*)(X.params.ptr + rows_off);
    a.bins = (const BinDesc*)X.params.ptr;
    a.cfg_tab = tab.empty() ? nullptr : (const uint16_t*)(X.params.ptr + tab_off);
    a.err = d_cnt + 4 * kPasses;
    a.out_cnt = out;
    a.out_stats = out + ncnt;
    a.out_w = (double*)(out + ncnt + 8);
    a.copies = copies;
    a.copy_stride = words;
    a.g = v.g;
    a.g.m = mst;
    a.n_items = (int)(v.n_data + v.n_rand);
    // Passes, each over the apexes whose neighbours outnumbered the list of the one before: one wave per apex (64
    // neighbours), work-groups with a list for the 99.5th percentile of ~2048 sampled neighbour counts (+5%, a power
    // of two), work-groups with the longest LDS list, and last work-groups with device-memory lists.  The waves take
    // unit weights where at least a quarter of the sample fits them: kernels of 0.97 against 1.84 ms (50k + 100k
    // points), 0.42 against 0.63 (27k + 54k, 4 bins); with weights the FP64 atomics of the quads
    // bound both, and work-groups are as fast or faster (0.69 against 0.71, 0.39 against 0.49 ms).
    const int n = a.n_items;
    int kmax1 = kmax;
    double short_lists = 0.0;
    bool long_lists = false;        // a last pass is to be expected
    const int nsample = std::min(n, 2048);
    bool gather = false;
    // i32: the lists of queued apexes, then the sample
    if ((rc = X.i32.reserve(kPasses * (size_t)n + 2 * nsample))) return rc;
    if (nsample > 0) {
        TripArgs ts{};
        ts.pw = a.pw;
        ts.flags = a.flags;
        ts.cell_start = a.cell_start;
        ts.rows = a.rows;
        ts.bins = a.bins;
        ts.g = a.g;
        ts.nrows = a.nrows;
        std::vector<int32_t> ks;
        if ((rc = sample_neighbours(ts, n, nsample, 0, X.i32.ptr + kPasses * (size_t)n, v.stream, ks, &gather))) return rc;
        if (!ks.empty()) {
            short_lists = (double)std::count_if(ks.begin(), ks.end(), [](int32_t k) { return k <= 64; }) / ks.size();
            const size_t q = std::min(ks.size() - 1, (size_t)std::ceil(0.995 * (ks.size() - 1)));
            std::nth_element(ks.begin(), ks.begin() + q, ks.end());
            const double want = 1.05 * ks[q];
            long_lists = ks[q] > kmax;
            kmax1 = 64;
            while (kmax1 < kmax && kmax1 < want) kmax1 *= 2;
        }
    }
    {
        const char* ev = getenv("GS_T4_KMAX");      // tuning override (unset or empty: automatic)
        if (ev && *ev) {
            kmax1 = 64;
            while (kmax1 < kmax && kmax1 < atoi(ev)) kmax1 *= 2;
        }
    }
    // weighted sums in LDS where that leaves room for two work-groups, and the gather (30,000 candidates an apex: 2.3 ms,
    // with sums in global memory 1.3) is not the work
    auto with_sums = [&](int km, bool wv) {
        QuadArgs t = a;
        t.kmax = km;
        // a mask per bin where that fits the same list (6,000 points with 180 neighbours: 8 bins 3.7 ms, with one mask
        // 5.3; 4 bins 4.3, 6.5); else one mask (10 bins 5.0 ms; lists of 128, and longer ones in device memory, 41)
        t.bin_masks = tetra ? 0 : 1;
        if (quad4_lds_bytes(t, nb, weighted, wv) > budget) t.bin_masks = 0;
        t.lds_w = weighted && !gather ? 1 : 0;
        if (quad4_lds_bytes(t, nb, weighted, wv) > 80 * 1024) t.lds_w = 0;
        return t;
    };
    bool wave = !weighted && short_lists >= 0.25;
    {
        const char* ev = getenv("GS_T4_WAVE");      // tuning override (unset or empty: automatic)
        if (ev && *ev) wave = !weighted && *ev != '0';
    }
    wave = wave && quad4_lds_bytes(with_sums(64, true), nb, weighted, true) <= budget;
    (void)hipEventRecord(v.ev[2], v.stream);
    struct Pass { bool wave; int kmax; };
    std::vector<Pass> passes;
    if (wave) passes.push_back({true, 64});
    if (kmax1 < kmax && !(wave && kmax1 == 64)) passes.push_back({false, kmax1});
    passes.push_back({false, kmax});
    const int np = (int)passes.size();
    for (int k = 0; k < np && n > 0; ++k) {
        const bool wv = passes[k].wave;
        QuadArgs t = with_sums(passes[k].kmax, wv);
        t.queue = head + k * kQueueInts;
        t.ovf = X.i32.ptr + (size_t)k * n;
        t.ovf_n = d_cnt + 4 * k;
        t.ovf_kmax = t.ovf_n + 1;
        if (k > 0) {
            // the number of apexes is read on the device
            t.items = X.i32.ptr + (size_t)(k - 1) * n;
            t.n_items_dev = d_cnt + 4 * (k - 1);
        }
        const int teams = wv ? kWG / kWave : 1;
        const int occ = quad4_occupancy(t, nb, weighted, wv);
        const int nblk = std::max(1, std::min(v.n_cu * occ, (n + teams - 1) / teams));
        t.batch = k > 0 ? 1 : std::max(triplet_batch(n, nblk, 1), wv ? 4 * teams : 1);
        e = launch_quad4(t, nb, weighted, wv, nblk, v.stream);
        if (e != hipSuccess) return hip_fail(e, "4PCF kernel launch");
    }
    (void)hipEventRecord(v.ev[3], v.stream);
    // the host makes its buffer (16 bins: 127 MB, 20 ms) beside the last kernels to run
    std::vector<unsigned long long> h_out;
    if (!long_lists) h_out.resize(words);
    int32_t* const h_cnt = (int32_t*)(H.ptr + res_off);
    int32_t* const last = d_cnt + 4 * (np - 1);
    auto counters = [&]() {         // apexes left to a last pass, their largest neighbour count, the error flag
        hipError_t r = hipMemcpyAsync(h_cnt, last, 2 * sizeof(int32_t), hipMemcpyDeviceToHost, v.stream);
        if (r == hipSuccess) r = hipMemcpyAsync(h_cnt + 2, a.err, sizeof(int32_t), hipMemcpyDeviceToHost, v.stream);
        return r;
    };
    auto results = [&]() {          // the copies' sum
        h_out.resize(words);
        hipError_t r = hipSuccess;
        if (copies > 1) {
            r = launch_sum_copies(out, copies, words, (int64_t)ncnt, 0, 8, X.out.ptr, v.stream);
            if (r == hipSuccess)
                r = launch_sum_copies_f64(a.out_w, copies, words, (int64_t)nw, (double*)(X.out.ptr + ncnt + 8), v.stream);
        }
        if (r == hipSuccess)
            r = hipMemcpyAsync(h_out.data(), copies > 1 ? X.out.ptr : out, (size_t)words * 8, hipMemcpyDeviceToHost, v.stream);
        return r;
    };
    // one wait for both where there are copies; a large result (16 bins: 30 ms) is fetched once, when it is complete
    e = counters();
    if (e == hipSuccess && copies > 1) e = results();
    if (e == hipSuccess) e = hipStreamSynchronize(v.stream);
    if (e != hipSuccess) return hip_fail(e, "4PCF kernel");
    const bool big = h_cnt[0] > 0;
    if (big) {
        // a last pass, over the apexes whose neighbours outnumber every LDS list, with their lists in device memory
        // (one per work-group; no link matrix)
        QuadArgs a3 = a;
        a3.items = X.i32.ptr + (size_t)(np - 1) * n;
        a3.n_items = h_cnt[0];
        a3.batch = 1;
        a3.kmax = 64;
        while (a3.kmax < h_cnt[1]) a3.kmax *= 2;        // a power of two for the bitonic sort
        const size_t gstride = (a3.kmax * kQuadGlistEntryBytes + 255) / 256 * 256;
        a3.glist = (void*)a3.items;             // selects the device-memory variant for the occupancy query
        const int occ3 = quad4_occupancy(a3, nb, weighted, false);
        const size_t gbudget = (size_t)1 << 30;
        const int nblk3 = (int)std::max<size_t>(1, std::min<size_t>({(size_t)h_cnt[0], (size_t)v.n_cu * occ3,
                                                                  gbudget / gstride}));
        if ((rc = X.big.reserve((size_t)nblk3 * gstride))) return rc;
        a3.glist = X.big.ptr;
        a3.glist_stride = (int64_t)gstride;
        a3.queue = head;
        e = launch_fill_u32(head, kQueueInts, 0u, v.stream);
        if (e == hipSuccess) e = launch_quad4(a3, nb, weighted, false, nblk3, v.stream);
        if (e != hipSuccess) return hip_fail(e, "4PCF device-memory pass");
        (void)hipEventRecord(v.ev[3], v.stream);
        e = counters();
    }
    if (e == hipSuccess && (big || copies == 1)) e = results();
    if (e == hipSuccess) e = hipStreamSynchronize(v.stream);
    if (e != hipSuccess) return hip_fail(e, "4PCF kernel");
    if (h_cnt[2]) return fail(GS_EHIP, "4PCF: an apex's neighbour list overflowed with no later pass (internal error)");
    const double* const h_w = (const double*)(h_out.data() + ncnt + 8);

    if (cnt) memcpy(cnt, h_out.data(), ncnt * sizeof(uint64_t));
    // normalised weight of one point: +w/Wd (data) or -w/Wr (random) (gramsci.F90:1390-1391)
    const long double Wd = v.wsum_d, Wr = v.wsum_r;
    auto norm = [&](int r) -> long double { return r ? -1.0L / Wr : 1.0L / Wd; };
    for (int q = 0; q < ncell; ++q) {
        long double v2 = 0, v3 = 0;
        for (int pat = 0; pat < 16; ++pat) {
            const long double s = weighted ? (long double)h_w[(size_t)q * 16 + pat] : (long double)h_out[(size_t)q * 16 + pat];
            if (s == 0) continue;
            const long double f = norm(pat & 1) * norm((pat >> 1) & 1) * norm((pat >> 2) & 1) * norm((pat >> 3) & 1);
            v2 += s * f;
            if (pat == 15) v3 += s * f;
        }
        if (n2) n2[q] = (double)v2;
        if (n3) n3[q] = (double)v3;
    }
    // disc terms: t -> (points a, b of the pair product; point c that must be random)
    //   t0: (i,k1 | k3)  t1: (i,k2 | k3)  t2: (i,k3 | k1)  t3: (k1,k2 | i)  t4: (k3,k2 | i)  t5: (k3,k1 | i)
    // the tetrahedron's terms are triple products that also carry c's normalised
    // weight, -w_c/Wr (gramsci.F90:590-631)
    static const int ta[6] = {0, 0, 0, 1, 3, 3}, tb[6] = {1, 2, 3, 2, 2, 1}, tc[6] = {3, 3, 1, 0, 0, 0};
    const long double fc = tetra ? norm(1) : 1.0L;
    for (int t = 0; t < 6; ++t)
        for (int q = 0; q < ncell; ++q) {
            long double dn = 0, dr = 0;
            for (int ab = 0; ab < 4; ++ab) {
                const int ra = ab & 1, rb = (ab >> 1) & 1;
                long double s;
                if (weighted) {
                    s = h_w[(size_t)ncell * 16 + ((size_t)t * ncell + q) * 4 + ab];
                } else {
                    s = 0;
                    for (int pat = 0; pat < 16; ++pat)
                        if (((pat >> tc[t]) & 1) && ((pat >> ta[t]) & 1) == ra && ((pat >> tb[t]) & 1) == rb)
                            s += (long double)h_out[(size_t)q * 16 + pat];
                }
                if (s == 0) continue;
                const long double term = s * norm(ra) * norm(rb) * fc;
                dn += term;
                if (ra && rb) dr += term;
            }
            if (disc_n) disc_n[(size_t)t * ncell + q] = (double)dn;
            if (disc_r) disc_r[(size_t)t * ncell + q] = (double)dr;
        }
    std::vector<unsigned long long> sts(5, 0);
    for (int k = 0; k < 5; ++k) sts[k] = h_out[ncnt + k];
    fill_stats(st, v.ev, sts.data(), mst);
    return GS_OK;
}

}  // namespace gs

extern "C" int gs_count_4pcf(gs_ctx* c, const gs_params* p, uint64_t* cnt, double* n2, double* n3, double* disc_n,
                             double* disc_r, gs_stats* st)
{
    return count4(c, p, false, cnt, n2, n3, disc_n, disc_r, st);
}

extern "C" int gs_count_4pcf_tetra(gs_ctx* c, const gs_params* p, uint64_t* cnt, double* n2, double* n3,
                                   double* disc_n, double* disc_r, gs_stats* st)
{
    return count4(c, p, true, cnt, n2, n3, disc_n, disc_r, st);
}
