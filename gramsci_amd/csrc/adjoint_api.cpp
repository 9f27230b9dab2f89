// adjoint_api.cpp -- C ABI of the 2PCF adjoint (gs_adjoint_2pcf, gs_adjoint_2pcf_device).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "gs_api_internal.h"
#include "gs_kernels.h"

using namespace gs;

static int adjoint_impl(gs_ctx* c, const gs_params* p, const double* gN2, const double* gN3, double* out_host,
                        double* out_dev, gs_stats* st)
{
    if (!c) return fail(GS_EINVAL, "NULL context");
    int rc = check_params(p, 2);
    if (rc) return rc;
    if (!gN2 || !gN3) return fail(GS_EINVAL, "dL/dN2 and dL/dN3 are required");
    if ((rc = ctx_set_device(c))) return rc;
    const int nb = p->nbins, nm = p->nmu;
    if (nb * nm > 2048) return fail(GS_ELIMIT, "adjoint supports nbins*nmu <= 2048");
    const bool rsd = nm >= 2, fp64 = p->precision == GS_FP64;
    CtxView v = view(c);
    const int64_t n = v.n_data + v.n_rand;
    if (!(v.wsum_d > 0) && v.n_data > 0) return fail(GS_EINVAL, "data weights sum to zero");
    if (!(v.wsum_r > 0) && v.n_rand > 0) return fail(GS_EINVAL, "random weights sum to zero");
    const double inv_wd = v.n_data > 0 ? (double)(1.0L / v.wsum_d) : 0.0;
    const double inv_wr = v.n_rand > 0 ? (double)(1.0L / v.wsum_r) : 0.0;
    // FP32: the half-stencil kernel with exact fixed-point sums at the scale 2^F, chosen so that no pair
    // term c * wn exceeds 2^50 (|c| <= 2 gmax, |wn| <= wmax / min(Wd, Wr)); split into a scale of the
    // dL/dN tables (2^Fa, bringing gmax to [1, 2)) and one of the weights (2^Fb).  Non-finite dL/dN
    // (or scales out of range) take the full-stencil kernel, which sums in FP64.
    bool half = !fp64;
    int F = 0, Fa = 0, Fb = 0;
    {
        double gmax = 0.0;
        for (int k = 0; k < nb * nm; ++k) {
            const double a2 = gN2[k], a23 = gN2[k] + gN3[k];
            if (!std::isfinite(a2) || !std::isfinite(a23)) half = false;
            else gmax = std::max(gmax, std::max(std::fabs(a2), std::fabs(a23)));
        }
        const double wn_max = v.wmax * std::max(inv_wd, inv_wr);
        if (half && gmax > 0.0 && wn_max > 0.0) {
            const double T = 2.0 * gmax * wn_max;
            F = 50 - (int)std::ceil(std::log2(T));
            Fa = -std::ilogb(gmax);
            Fb = F - Fa;
            if (!std::isfinite(T) || T <= 0.0 || std::abs(Fa) > 1000 || std::abs(Fb) > 1000 || std::abs(F) > 1000)
                half = false;
        }
    }
    // The half-stencil kernel walks the pair kernel's grid, the full-stencil one its own.  Parameters (bins,
    // dL/dN tables, stencil rows) go to the device in one copy from pinned memory; the counters come back
    // through it, written by a kernel.
    GsExtra& X = *v.extra;
    HostBuf& H = ctx_host(c);
    const size_t ng = (size_t)nb * nm, g_off = (sizeof(BinDesc) + 15) / 16 * 16, rows_off = g_off + (ng * 16 + 15) / 16 * 16;
    const size_t stats_off = rows_off + kMaxRows * sizeof(Row);
    double t64[kMaxBins + 2];
    if ((rc = ctx_thresholds(c, *p, t64)) || (rc = H.reserve(stats_off + 16)) || (rc = X.params.reserve(stats_off)))
        return rc;
    BinDesc& B = *(BinDesc*)H.ptr;
    PairGrid q;
    if (half) {
        q = ctx_pair_grid(c, *p);
        if ((rc = fill_pair_bins(*p, t64, q, ctx_xmax(c), v.wmax_d, v.wmax_r, B))) return rc;
        half = !B.wide;     // beyond the FP32 geometry's range
    }
    const int nblk_red = 256;
    const size_t n1 = (size_t)std::max<int64_t>(n, 1), queue_bytes = 64 * kQueuePad * sizeof(int32_t);
    std::vector<Row> rows;
    int mst;
    unsigned char* z = nullptr;     // cleared: work counters, {candidates, rechecks, ticket}, fixed-point sums
    (void)hipEventRecord(v.ev[0], v.stream);
    if (half) {
        mst = q.mst;
        rows = half_stencil(q.h, q.h / q.sx, p->rmax, mst);
        if ((rc = ctx_build_pair_grid(c, q, (queue_bytes + 256 + n1 * 16 + 255) / 256 * 256, &z))) return rc;
    } else {
        double h;
        const int m = p->cell_div > 0 ? p->cell_div : default_cell_div(c, p->rmax, 2), sx = pair_cell_sx();
        if ((rc = ctx_build_grid(c, p->rmax, m, sx, &h)) || (rc = ctx_row_chunks(c))) return rc;
        mst = (int)std::ceil(p->rmax / h - 1e-12);
        if ((rc = fill_bins(*p, t64, (mst + 1) * h, ctx_xmax(c), v.wmax_d, v.wmax_r, B))) return rc;
        rows = full_stencil(h, h / sx, p->rmax, mst);
        if ((rc = X.queue.reserve((queue_bytes + 256) / 4))) return rc;
        z = (unsigned char*)X.queue.ptr;
    }
    if ((int)rows.size() > kMaxRows) return fail(GS_ELIMIT, "stencil too large");
    if ((rc = X.dbl.reserve(2 * n1 + 2 * nblk_red + 8))) return rc;
    v = view(c);
    double* G = X.dbl.ptr;
    double* outd = out_dev ? out_dev : X.dbl.ptr + n;
    double* part = X.dbl.ptr + 2 * n1;
    int32_t* queue = (int32_t*)z;
    unsigned long long* stats = (unsigned long long*)(z + queue_bytes);
    unsigned long long* Glo = (unsigned long long*)(z + queue_bytes + 256);     // half: [n1] each
    long long* Ghi = (long long*)Glo + n1;
    std::copy(gN2, gN2 + ng, (double*)(H.ptr + g_off));
    std::copy(gN3, gN3 + ng, (double*)(H.ptr + g_off) + ng);
    std::copy(rows.begin(), rows.end(), (Row*)(H.ptr + rows_off));
    unsigned long long* const h_stats = (unsigned long long*)(H.ptr + stats_off);
    hipError_t e = hipMemcpyAsync(X.params.ptr, H.ptr, rows_off + rows.size() * sizeof(Row), hipMemcpyHostToDevice,
                                  v.stream);
    if (e == hipSuccess && !half) e = launch_fill_u32(z, (int64_t)(queue_bytes + 256) / 4, 0u, v.stream);
    if (e == hipSuccess && !half) e = launch_fill_u32(G, (int64_t)n1 * 2, 0u, v.stream);
    if (e != hipSuccess) return hip_fail(e, "adjoint parameter upload");

    const double *g2 = (const double*)(X.params.ptr + g_off), *g3 = g2 + nb * nm;
    (void)hipEventRecord(v.ev[2], v.stream);
    if (half && n > 0) {
        AdjHalfArgs a{};
        a.pw = v.pw;
        a.cell = v.cell;
        a.flags = v.flags;
        a.cell_start = v.cell_start;
        a.rows = (const Row*)(X.params.ptr + rows_off);
        a.bins = (const BinDesc*)X.params.ptr;
        a.queue = queue;
        a.g = v.g;
        a.g.m = mst;
        a.nrows = (int)rows.size();
        a.g2 = g2;
        a.g3 = g3;
        a.Glo = Glo;
        a.Ghi = Ghi;
        a.out_stats = stats;
        a.inv_wd = inv_wd;
        a.inv_wr = inv_wr;
        a.g_scale = std::ldexp(1.0, Fa);
        a.w_scale = std::ldexp(1.0, Fb);
        const bool logb = p->log_bins != 0;
        const int waves = adjoint2h_occupancy(nb, nm, logb, v.has_buf) * (kWG / kWave);
        e = launch_adjoint2h(a, nb, nm, logb, v.has_buf, walk_shape(a, q, n, kWG, waves, v.n_cu), v.stream);
        if (e != hipSuccess) return hip_fail(e, "adjoint kernel launch");
        if ((e = launch_adj_fx(Glo, Ghi, v.orig, n, F, G, v.stream)) != hipSuccess)
            return hip_fail(e, "adjoint fixed-point conversion");
    } else if (n > 0 && v.n_chunks > 0) {
        AdjArgs a{};
        a.pw = v.pw;
        a.cell = v.cell;
        a.flags = v.flags;
        a.orig = v.orig;
        a.cell_start = v.cell_start;
        a.row_chunk = v.row_chunk;
        a.rows = (const Row*)(X.params.ptr + rows_off);
        a.bins = (const BinDesc*)X.params.ptr;
        a.g2 = g2;
        a.g3 = g3;
        a.queue = queue;
        a.G = G;
        a.out_stats = stats;
        a.g = v.g;
        a.g.m = mst;
        a.nrows = (int)rows.size();
        a.n_chunks = v.n_chunks;
        a.inv_wd = inv_wd;
        a.inv_wr = inv_wr;
        const int nblocks = std::min(v.n_cu * adjoint2_occupancy(nb, nm, fp64, rsd), v.n_chunks);
        e = launch_adjoint2(a, nb, nm, fp64, rsd, nblocks, v.stream);
        if (e != hipSuccess) return hip_fail(e, "adjoint kernel launch");
    }
    (void)hipEventRecord(v.ev[3], v.stream);
    e = launch_adj_partials(G, v.w, n, v.n_data, inv_wd, inv_wr, part, nblk_red, stats, h_stats, v.stream);
    if (e == hipSuccess) e = launch_adj_finish(G, n, v.n_data, part + 2 * nblk_red, inv_wd, inv_wr, outd, v.stream);
    if (e == hipSuccess && out_host) e = hipMemcpyAsync(out_host, outd, (size_t)n * 8, hipMemcpyDeviceToHost, v.stream);
    if (e == hipSuccess) e = hipStreamSynchronize(v.stream);
    if (e != hipSuccess) return hip_fail(e, "adjoint kernel");
    if (st) {
        memset(st, 0, sizeof(*st));
        float ms_grid = 0, ms_count = 0;
        (void)hipEventElapsedTime(&ms_grid, v.ev[0], v.ev[2]);
        (void)hipEventElapsedTime(&ms_count, v.ev[2], v.ev[3]);
        st->ms_grid = ms_grid;
        st->ms_count = ms_count;
        st->ms_kernel_avg = ms_count;
        st->n_candidates = h_stats[0];
        st->n_evaluated = h_stats[0];
        st->n_recheck = h_stats[1];
        st->cell_div = mst;
    }
    return GS_OK;
}

extern "C" int gs_adjoint_2pcf(gs_ctx* c, const gs_params* p, const double* dl_dn2, const double* dl_dn3,
                               double* dl_dw, gs_stats* st)
{
    if (!dl_dw) return fail(GS_EINVAL, "dl_dw is NULL");
    return adjoint_impl(c, p, dl_dn2, dl_dn3, dl_dw, nullptr, st);
}

extern "C" int gs_adjoint_2pcf_device(gs_ctx* c, const gs_params* p, const double* dl_dn2, const double* dl_dn3,
                                      double* d_dl_dw, gs_stats* st)
{
    if (!d_dl_dw) return fail(GS_EINVAL, "d_dl_dw is NULL");
    return adjoint_impl(c, p, dl_dn2, dl_dn3, nullptr, d_dl_dw, st);
}
