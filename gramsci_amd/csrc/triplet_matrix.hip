// triplet_matrix.hip -- the isotropic 3PCF of unit weights with FP32 geometry: every configuration of triangles,
// third sides from the matrix cores.
//
// What triplet3.hip's kernel does for this case (the reference's create_graph + query_graph_3pcf_all,
// gramsci.F90:288-348, :463-545, each triangle visited once, from the first of its vertices in the order
// "points that are not buffer points, by index, then buffer points"), with another inner loop.  For an apex
// with K kept neighbours after it, the K (K - 1) / 2 third sides are all the kernel's work beyond some hundreds
// of neighbours, and per pair the vector ALU is what bounds it (three subtractions, three products, bin, guard,
// histogram, and the decoding of both neighbours' bins and classes: about 40 instructions a pair).  So:
//
//  * The squared third side |u - v|^2 = |u|^2 + |v|^2 - 2 u.v comes from one v_mfma_f32_16x16x4_f32 per 16 x 16
//    block of neighbour pairs: rows v as (-2x, -2y, -2z, 1), columns u as (x, y, z, |u|^2), accumulators |v|^2.
//    A lane then holds four pairs of one u, and the vector ALU only bins them.  The blocks are those of the
//    upper triangle, so less than 16 / K of the pairs are computed in vain.
//  * A neighbour's bin, class (random or not) and buffer flag are one tag, its part of the histogram's byte
//    offset: the histogram is [buffer vertices][class][bin of u][bin of v][third side], folded to configurations
//    only when it is added to the outputs, so a pair's slot is one addition and one shift-add.  Third sides below
//    and above the bins are slots too, certain or not like a bin, so that one comparison tells the pairs that FP64
//    has to decide; those below are counted (nobody reads them), those above left out.
//
// Error of the squared side, in units where rmax is in [1, 2) (coordinates are scaled by a power of two), with
// u = 2^-24 and |x| <= rmax for every neighbour: rounding the coordinates moves it by at most 8 u rmax^2, |u|^2
// and |v|^2 by 2 u rmax^2, the products and sums of the matrix instruction by at most 5 roundings of partial
// sums below 4 rmax^2, doubled for an accumulation that does not round to nearest: 50 u rmax^2 in all, bounded by
// 64 u rmax^2 (fill_triplet_matrix's `err`).  A pair within that of a bin edge is decided in FP64 from the catalogue's
// coordinates, as everywhere else, so the counts are those of the FP64 kernel.
//
// A team, one wave (short lists) or a whole work-group, takes one apex at a time: it numbers the candidates of
// the stencil rows consecutively, keeps the neighbours' indices by ballots, then bins the kept ones with all
// lanes busy, then walks its blocks.  With one wave per apex no barrier is needed between these phases.
//
// Measured against the general kernel: 200k + 400k points, rmax 30 of box 500, 5 bins (19.3e9 third sides) 20.2 ->
// 11.0 ms; 16 regions of 60k points, 4 bins, buffer points 6.4 -> 3.2 ms.  63 vector instructions per block, the
// neighbours' gather included, for four pairs a lane (before: 44 per pair), still bound it: 0.81 a CU-cycle, the
// LDS busy half of the time.  Counting the sides above the bins too (their slots are hot) cost 2 ms.
#include "gs_device.h"
#include "gs_kernels.h"

namespace gs {

using namespace dev;

namespace {

typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kMatrixMaxWG = 512;
constexpr int kControlBytes = 64;       // work item, list counters, statistics
constexpr int kListWords = 6;           // per list entry: x, y, z, |.|^2, its two tags (16 bits each), sorted index

// LDS by byte address.  The kernel's LDS is all dynamic, so the array starts at address 0 (the launch refuses a kernel
// with static LDS, which a helper could bring with it); through the array's name the compiler adds that zero to every
// address it forms.
template <class T>
using lds_ptr = __attribute__((address_space(3))) T*;

__host__ __device__ inline size_t team_bytes(int kmax, int nrows)
{
    return (size_t)kListWords * 4 * (kmax + 16) + ((size_t)nrows * 12 + 15) / 16 * 16;
}

__device__ __forceinline__ void lds_count(uint32_t at)
{
    __hip_atomic_fetch_add((lds_ptr<uint32_t>)at, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

}  // namespace

size_t triplet_matrix_lds(const TripArgs& a, int nb, int teams)
{
    size_t b = ((size_t)(nb + 2) * a.reps * 4 + 15) / 16 * 16 + kControlBytes;              // certain intervals
    b += ((size_t)nb * nb * (nb + 2) * 4 * (a.buf ? 3 : 1) * a.reps * 4 + 15) / 16 * 16;    // histogram
    b += ((size_t)(nb + 2) * 8 + 15) / 16 * 16;                                             // t64
    return b + teams * team_bytes(a.kmax, a.nrows);
}

template <bool LOGB, bool WAVE, bool BATCH>
__global__ __launch_bounds__(kMatrixMaxWG) void k_triplet_matrix(TripArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const TripMatrix& M = *a.matrix;
    // slots of a pair of bins: sides below, in, above the nb bins
    const int nb = B.nb, ns = nb + 2, nb3 = nb * nb * ns, nf = a.buf ? 3 : 1;
    const int reps = a.reps, rsh = 31 - __clz(reps);
    const int kmax = a.kmax, stride = kmax + 16;    // 16 mod 64: the four rows of an operand fall on all banks
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, nw = nt >> 6;
    const int wv = scalar(tid >> 6);
    const int tl = WAVE ? lane : tid, tn = WAVE ? kWave : nt;       // thread of the team, threads in it

    // The certain intervals lie at the start, as far apart as the histogram's slots (4 reps bytes, reps >= 2): one
    // shift of a bin gives both its interval's and its slot's offset.
    const unsigned sh = (unsigned)rsh + 2;
    const uint32_t hist_off = (uint32_t)(((size_t)ns * reps * 4 + 15) / 16 * 16) + kControlBytes;
    int* const ctl = (int*)(smem + hist_off - kControlBytes);      // no static LDS: the intervals are at address 0
    int &s_item = ctl[0], &s_k = ctl[1], &s_kall = ctl[2], &s_ncand = ctl[3];
    unsigned long long* const s_stat = (unsigned long long*)(ctl + 4);
    uint32_t* hc = (uint32_t*)(smem + hist_off);
    unsigned char* p = smem + hist_off + ((size_t)nb3 * 4 * nf * reps * 4 + 15) / 16 * 16;
    double* t64 = (double*)p;
    p += ((size_t)(nb + 2) * 8 + 15) / 16 * 16;
    if (WAVE) p += (size_t)wv * team_bytes(kmax, a.nrows);
    float* xs = (float*)p;                          // [4][stride]: x, y, z, |.|^2
    uint32_t* tags = (uint32_t*)(xs + 4 * stride);  // tag as u | tag as v << 16
    int32_t* jl = (int32_t*)(tags + stride);
    int32_t* rw_js = jl + stride;                   // stencil rows: first point, length, number of the first point
    int32_t* rw_len = rw_js + a.nrows;
    int32_t* rw_off = rw_len + a.nrows;

    auto sync = [&]() {
        if constexpr (WAVE) wave_sync();
        else __syncthreads();
    };

    for (int k = tid; k < nb3 * 4 * nf * reps; k += nt) hc[k] = 0;
    for (int k = tid; k < ns; k += nt) *(float2*)(smem + ((uint32_t)k << sh)) = M.ok[k];
    for (int k = tid; k < nb + 2; k += nt) t64[k] = B.t64[k];
    if (tid == 0) { s_k = 0; s_kall = 0; }
    __syncthreads();

    const size_t copy = (size_t)(blockIdx.x & (unsigned)(a.copies - 1)) * (size_t)a.copy_stride;
    // adds the histogram to region r's output and clears it: one output entry per thread t, t + step, ...  Its
    // slots are those of the permutations of its three bins (repeated ones read zero the second time).
    auto drain = [&](int r, int t, int step) {
        for (int o = opaque(t); o < a.ncfg * 4; o += step) {
            const uint32_t ijk = a.cfg_bins[o >> 2];
            const int i = ijk & 255, j = (ijk >> 8) & 255, k = ijk >> 16;
            const int at[6] = {(i * nb + j) * ns + k + 1, (i * nb + k) * ns + j + 1, (j * nb + i) * ns + k + 1,
                               (j * nb + k) * ns + i + 1, (k * nb + i) * ns + j + 1, (k * nb + j) * ns + i + 1};
            unsigned long long sum = 0;
            for (int f = 0; f < nf; ++f)
                for (int q = 0; q < 6; ++q) {
                    uint32_t* h = hc + ((size_t)(at[q] + nb3 * ((o & 3) + 4 * f)) << rsh);
                    unsigned long long s = 0;
                    for (int e = 0; e < reps; ++e) s += atomicExch(&h[e], 0u);
                    // counted at every vertex that is not a buffer point
                    sum += s * (unsigned)(3 - f);
                }
            if (sum) atomicAdd(&a.out_cnt[copy + (size_t)r * a.ncfg * 4 + o], sum);
        }
    };

    const float ua = M.ua, above = M.ok[nb + 1].x, topf = (float)(nb + 1);
    float ubv = M.ub;               // in a VGPR: an FMA reads at most one scalar operand
    asm volatile("" : "+v"(ubv));
    const double t_lo = scalar(B.t64[0]), t_hi = scalar(B.t64[nb + 1]), t_top = scalar(M.t_top);
    const double inv_h = scalar(M.inv_h), inv_hx = scalar(M.inv_hx), scale = scalar(M.scale);
    unsigned long long units = 0, evals = 0, cand = 0;      // of the team, kept by its waves alike
    unsigned rechk = 0, over = 0;                           // of the lane
    unsigned long long bound = 0;   // increments this wave or work-group may have issued since it last drained
    int cur_r = BATCH ? -1 : 0;
    int nx = a.g.dim[0], ny = a.g.dim[1], nz = a.g.dim[2], cb = 0;
    double lx = a.g.lo[0], ly = a.g.lo[1], lz = a.g.lo[2];

    const int n_items = scalar(a.n_items_dev ? *a.n_items_dev : a.n_items);
    const int bsz = max(a.batch, 1);
    ItemQueue items(a.queue, (n_items + bsz - 1) / bsz, 1);

    auto visit_apex = [&](const int item) {
        const int apex = scalar(a.items ? a.items[item] : item);
        const uint32_t fa = (uint32_t)scalar((int)a.flags[apex]);
        if (fa & 2u) return;                        // buffer point: never an apex (gramsci.F90:476)
        double4 Pa = a.pw[apex];
        Pa.x = scalar(Pa.x); Pa.y = scalar(Pa.y); Pa.z = scalar(Pa.z);
        const int cx = min(max((int)floor((Pa.x - lx) * inv_hx), 0), nx - 1);
        const int cy = min(max((int)floor((Pa.y - ly) * inv_h), 0), ny - 1);
        const int cz = min(max((int)floor((Pa.z - lz) * inv_h), 0), nz - 1);
        // ---- the stencil rows' point ranges, numbered consecutively
        for (int r = tl; r < a.nrows; r += tn) {
            const Row rw = a.rows[r];
            const int by = cy + rw.dy, bz = cz + rw.dz;
            const int bx0 = max(cx + rw.x0, 0), bx1 = min(cx + rw.x1, nx - 1);
            int js = 0, len = 0;
            if (by >= 0 && by < ny && bz >= 0 && bz < nz && bx0 <= bx1) {
                const int rb = cb + (bz * ny + by) * nx;
                js = a.cell_start[rb + bx0];
                len = a.cell_start[rb + bx1 + 1] - js;
            }
            rw_js[r] = js;
            rw_len[r] = len;
        }
        sync();
        int ncand = 0;
        if (WAVE || tid < kWave) {
            for (int b0 = 0; b0 < a.nrows; b0 += kWave) {
                const int x = b0 + lane < a.nrows ? rw_len[b0 + lane] : 0;
                int inc = x;
                for (int off = 1; off < kWave; off <<= 1) {
                    const int y = __shfl_up(inc, off, 64);
                    if (lane >= off) inc += y;
                }
                if (b0 + lane < a.nrows) rw_off[b0 + lane] = ncand + inc - x;
                ncand += __shfl(inc, 63, 64);
            }
            if (!WAVE && tid == 0) s_ncand = ncand;
        }
        sync();
        if (!WAVE) ncand = s_ncand;
        ncand = scalar(ncand);
        // ---- the kept neighbours: all are counted, those after the apex enter the list
        int K = 0, kall = 0;
        unsigned n_over = 0;
        {
            int row = 0, row_end = a.nrows > 0 ? rw_len[0] : 0, j0 = a.nrows > 0 ? rw_js[0] : 0;
            for (int base = 0; base < ncand; base += tn) {
                const int next = base + tl;
                bool kept = false, after = false;
                int j = 0;
                if (next < ncand) {
                    while (next >= row_end) {       // the row holding candidate number next
                        ++row;
                        const int beg = rw_off[row];
                        row_end = beg + rw_len[row];
                        j0 = rw_js[row] - beg;
                    }
                    j = j0 + next;
                    const double4 Pj = a.pw[j];
                    const double s = exact_s(Pa.x, Pa.y, Pa.z, Pj.x, Pj.y, Pj.z);
                    kept = s > t_lo && s < t_top;
                    if (s >= t_top && s < t_hi && s > t_lo) ++n_over;
                    if (kept) after = j > apex || (a.buf && (a.flags[j] & 2u));
                }
                const unsigned long long ma = __ballot(after);
                kall += (int)__popcll(__ballot(kept));
                int pos = K;
                if constexpr (!WAVE) {
                    int at = 0;
                    if (lane == 0 && ma) at = atomicAdd(&s_k, (int)__popcll(ma));
                    pos = scalar(at);
                }
                pos += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ma >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ma, 0u));
                if (after && pos < kmax) jl[pos] = j;
                K += (int)__popcll(ma);
            }
            if (!WAVE && lane == 0 && kall) atomicAdd(&s_kall, kall);
        }
        sync();
        if constexpr (!WAVE) {
            K = scalar(s_k);
            kall = scalar(s_kall);
        }
        if (K > kmax) {
            // left to a later pass with room for all its neighbours, which also counts its candidates
            if (tl == 0) {
                a.ovf[atomicAdd(a.ovf_n, 1)] = apex;
                if (a.ovf_kmax) atomicMax(a.ovf_kmax, K);
            }
            if constexpr (!WAVE) {
                __syncthreads();
                if (tid == 0) { s_k = 0; s_kall = 0; }
                __syncthreads();
            }
            return;
        }
        over += n_over;
        // ---- their records and tags, padded to whole blocks with points beyond every range
        const int Kp = (K + 15) & ~15;
        for (int k = tl; k < Kp; k += tn) {
            float x = 0.0f, y = 0.0f, z = 0.0f, n2 = 1e30f;
            uint32_t tag = 0;
            if (k < K) {
                const int j = jl[k];
                const double4 Pj = a.pw[j];
                const uint32_t fj = a.flags[j];
                const double s = exact_s(Pa.x, Pa.y, Pa.z, Pj.x, Pj.y, Pj.z);
                int b = (int)__builtin_amdgcn_fmed3f(bin_estimate((float)(s * scale * scale), LOGB, ua, ubv), 1.0f, topf - 1.0f) - 1;
                while (b > 0 && s < t64[b]) --b;
                while (b < nb - 1 && s >= t64[b + 1]) ++b;
                x = (float)((Pj.x - Pa.x) * scale);
                y = (float)((Pj.y - Pa.y) * scale);
                z = (float)((Pj.z - Pa.z) * scale);
                n2 = (float)((double)x * x + (double)y * y + (double)z * z);
                const int cls = nb3 * ((int)(fj & 1u) + (a.buf ? (int)(fj & 2u) * 2 : 0));
                tag = ((uint32_t)(b * nb * ns + cls) << sh) | ((uint32_t)(b * ns + cls) << sh << 16);
            }
            xs[k] = x;
            xs[stride + k] = y;
            xs[2 * stride + k] = z;
            xs[3 * stride + k] = n2;
            tags[k] = tag;
        }
        sync();
        if (!WAVE && tid == 0) { s_k = 0; s_kall = 0; }
        const unsigned long long P = (unsigned long long)K * (unsigned)max(K - 1, 0) / 2;
        cand += (unsigned)ncand;
        units += (unsigned long long)kall * (unsigned)max(kall - 1, 0) / 2;     // the reference's candidates
        evals += P;
        // ---- third sides: blocks (tu, tv), tu <= tv, of the triangle; a wave takes a range of them
        const int nt16 = Kp >> 4, nblk = nt16 * (nt16 + 1) / 2;
        const int w0 = WAVE ? 0 : wv, wn = WAVE ? 1 : nw;
        int blk = scalar((int)((long long)nblk * w0 / wn));
        const int bend = scalar((int)((long long)nblk * (w0 + 1) / wn));
        if (blk < bend) {
            const int q = lane >> 4, c = lane & 15;
            int vt = (int)((sqrtf(8.0f * (float)blk + 1.0f) - 1.0f) * 0.5f);
            while ((vt + 1) * (vt + 2) / 2 <= blk) ++vt;
            while (vt * (vt + 1) / 2 > blk) --vt;
            vt = scalar(vt);
            int ut = scalar(blk - vt * (vt + 1) / 2);
            // the histogram, the class of the apex and the lane's replica, added to v's tags
            const uint32_t base = hist_off + ((uint32_t)(nb3 * (int)(fa & 1u)) << sh) + ((uint32_t)(lane & (reps - 1)) << 2);
            const float* us = xs + q * stride + c;
            while (true) {
                const int v0 = vt * 16, vi = v0 + 4 * q;
                const float av = q < 3 ? -2.0f * us[v0] : 1.0f;
                const float4v nv = *(const float4v*)(xs + 3 * stride + vi);
                uint32_t tg[4];
                for (int i = 0; i < 4; ++i) tg[i] = (tags[vi + i] >> 16) + base;
                const int uend = min(vt + 1, ut + (bend - blk));
                blk += uend - ut;
                float bu = us[ut * 16];
                uint32_t tc = tags[ut * 16 + c];
                for (; ut < uend; ++ut) {
                    float4v d = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bu, nv, 0, 0, 0);
                    const uint32_t tcur = tc & 0xffffu;
                    const int un = min(ut + 1, vt) * 16;        // the next block's u (or this one's again)
                    bu = us[un];
                    tc = tags[un + c];
                    if (ut == vt) {         // each pair once
                        asm volatile("");   // a branch, not eight selects on every block
                        for (int i = 0; i < 4; ++i) d[i] = c < 4 * q + i ? d[i] : 1e30f;
                    }
                    uint32_t off[4];
                    float2v ok[4];
                    for (int i = 0; i < 4; ++i)
                        off[i] = (uint32_t)(int)__builtin_amdgcn_fmed3f(bin_estimate(d[i], LOGB, ua, ubv), 0.0f, topf) << sh;
                    for (int i = 0; i < 4; ++i) ok[i] = *(lds_ptr<float2v>)off[i];
                    unsigned long long unc[4];      // lanes to decide in FP64
                    for (int i = 0; i < 4; ++i) {
                        // as unsigned: negative differences are above every bound
                        const bool sure = __float_as_uint(d[i] - ok[i].x) < __float_as_uint(ok[i].y);
                        unc[i] = ~__builtin_amdgcn_ballot_w64(sure);
                        if (sure && d[i] < above) lds_count(off[i] + tg[i] + tcur);
                    }
                    if (unc[0] | unc[1] | unc[2] | unc[3]) {
                        const int l = opaque(lane), uj = ut * 16 + (l & 15), vj = vt * 16 + 4 * (l >> 4);
                        for (int i = 0; i < 4; ++i)
                            if (unc[i] >> l & 1) {
                                ++rechk;
                                const double4 Pu = a.pw[jl[uj]], Pv = a.pw[jl[vj + i]];
                                const double se = exact_s(Pu.x, Pu.y, Pu.z, Pv.x, Pv.y, Pv.z);
                                if (se > B.t64[0] && se < B.t64[opaque(nb) + 1]) {
                                    const int be = exact_bin(se, t64, nb);
                                    if (be == nb) ++over;
                                    else lds_count(((uint32_t)(be + 1) << sh) + tg[i] + tcur);
                                }
                            }
                    }
                }
                if (blk >= bend) break;
                ++vt;
                ut = 0;
            }
        }
        // a u32 count takes at most one increment per pair; the teams of a work-group share the histogram
        bound += P;
        if (bound > (WAVE ? 1ull << 28 : 1ull << 31)) {
            if (!WAVE) __syncthreads();
            drain(cur_r, tl, tn);
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
        int lo = b * bsz;
        const int hi = min(n_items, lo + bsz);
        while (lo < hi) {
            int sub = hi;
            if constexpr (BATCH) {
                // apexes of one region: the histogram holds one region's counts
                const int apex = scalar(a.items ? a.items[lo] : lo);
                int r = 0, rh = a.nreg - 1;         // last region with pt_base <= apex
                while (r < rh) {
                    const int mid = (r + rh + 1) >> 1;
                    if (scalar(a.regions[mid].pt_base) <= apex) r = mid; else rh = mid - 1;
                }
                if (r != cur_r) {
                    __syncthreads();
                    if (cur_r >= 0) drain(cur_r, tid, nt);
                    bound = 0;
                    __syncthreads();
                    cur_r = r;
                    const RegionDesc& rd = a.regions[r];
                    nx = scalar(rd.dim[0]); ny = scalar(rd.dim[1]); nz = scalar(rd.dim[2]);
                    cb = scalar(rd.cell_base);
                    lx = scalar(rd.lo[0]); ly = scalar(rd.lo[1]); lz = scalar(rd.lo[2]);
                }
                if (a.items) sub = lo + 1;
                else if (r + 1 < a.nreg) sub = min(hi, scalar(a.regions[r + 1].pt_base));
            }
            for (int it = lo + (WAVE ? wv : 0); it < sub; it += WAVE ? nw : 1) visit_apex(it);
            lo = sub;
        }
        __syncthreads();
    }
    __syncthreads();
    if (cur_r >= 0) drain(cur_r, tid, nt);
    if (tid < 5) s_stat[tid] = 0;
    __syncthreads();
    for (int off = 32; off > 0; off >>= 1) {
        rechk += __shfl_down(rechk, off, 64);
        over += __shfl_down(over, off, 64);
    }
    if (lane == 0) {
        atomicAdd(&s_stat[1], (unsigned long long)rechk);
        atomicAdd(&s_stat[2], (unsigned long long)over);
        if (WAVE || wv == 0) {
            atomicAdd(&s_stat[0], cand);
            atomicAdd(&s_stat[3], units);
            atomicAdd(&s_stat[4], evals);
        }
    }
    __syncthreads();
    if (tid < 5 && s_stat[tid]) atomicAdd(&a.out_stats[copy + tid], s_stat[tid]);
}

template <bool... Done, class F>
static auto with_matrix(bool logb, bool wave, bool batch, F&& f)
{
    if constexpr (sizeof...(Done) == 3) {
        return f(k_triplet_matrix<Done...>);
    } else {
        const bool next = sizeof...(Done) == 0 ? logb : (sizeof...(Done) == 1 ? wave : batch);
        return next ? with_matrix<Done..., true>(logb, wave, batch, f) : with_matrix<Done..., false>(logb, wave, batch, f);
    }
}

hipError_t launch_triplet_matrix(const TripArgs& a, int nb, bool wave, int nblocks, hipStream_t st)
{
    const size_t lds = triplet_matrix_lds(a, nb, wave ? a.wg / kWave : 1);
    return with_matrix(a.log_bins != 0, wave, a.nreg > 0, [&](auto kern) {
        hipFuncAttributes at;
        hipError_t e = hipFuncGetAttributes(&at, (const void*)kern);
        if (e != hipSuccess) return e;
        if (at.sharedSizeBytes != 0) return hipErrorInvalidDeviceFunction;
        if (lds > 64 * 1024) {
            e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kern, dim3(nblocks), dim3(a.wg), lds, st, a);
        return hipGetLastError();
    });
}

int triplet_matrix_occupancy(const TripArgs& a, int nb, bool wave)
{
    const size_t lds = triplet_matrix_lds(a, nb, wave ? a.wg / kWave : 1);
    return with_matrix(a.log_bins != 0, wave, a.nreg > 0, [&](auto kern) {
        int n = 0;
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, a.wg, lds);
        return e == hipSuccess ? n : 0;
    });
}

}  // namespace gs
