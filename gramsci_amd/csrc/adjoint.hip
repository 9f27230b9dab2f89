// adjoint.hip -- adjoint of the weighted 2PCF (r, mu) counts with respect to
// the per-point weights.
//
// Forward (gramsci.F90:352-380): N2[b,m] = sum over kept ordered pairs i->j of
// wn_i wn_j, N3[b,m] the same over random-random pairs, with the normalised
// weights wn = w/Wd (data) and -w/Wr (randoms) of gramsci.F90:1390-1391.
// Given g2 = dL/dN2 and g3 = dL/dN3 this computes, per point k,
//     G_k = dL/dwn_k = sum_j wn_j [c_k (g2 + [k,j random] g3)(b, m_kj)
//                                 + c_j (g2 + [k,j random] g3)(b, m_jk)]
// (c = 1 if the point may be an apex), and then the raw-weight gradient
//     dL/dw_k = (G_k - S_D)/Wd (data),   -(G_k + S_R)/Wr (randoms),
// S_D = sum_{data} wn G, S_R = sum_{randoms} wn G.
//
// Two kernels: k_adjoint2 takes 64 points of one x-row per wave over the FULL
// stencil (FP32 geometry with guard band and FP64 recheck, or plain FP64), so
// that every ordered pair is seen from its apex's lane and G_k accumulates in
// an FP64 register without atomics (FP64 precision, and non-finite dL/dN);
// k_adjoint2h (FP32) walks the pair kernel's tiles over the half stencil, each
// unordered pair once, with exact fixed-point sums.
#include "gs_pair_tiles.h"
#include "gs_kernels.h"

namespace gs {

using namespace dev;

size_t adjoint2_lds_bytes(int nb, int nm, bool fp64)
{
    size_t b = 0;
    b += (size_t)nb * nm * 8 * 2;                              // g2, g2 + g3
    b += ((size_t)(kMaxBins + 1) * 8);                          // ok_lo/ok_hi
    b += ((size_t)(kMaxBins + 2) * 8 + 15) / 16 * 16;           // t64
    const int waves = kWG / kWave;
    b += (size_t)waves * kWave * (fp64 ? 40 : 32);              // tiles
    return b;
}

template <bool FP64, bool RSD>
__global__ __launch_bounds__(kWG) void k_adjoint2(AdjArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const int nb = B.nb;
    const int nm = RSD ? B.nm : 1;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = tid / kWave;

    unsigned char* p = smem;
    double* g2 = (double*)p;                // dL/dN2 per (bin, mu)
    double* g23 = g2 + nb * nm;             // dL/dN2 + dL/dN3 (a random-random pair feeds both)
    p += (size_t)nb * nm * 16;
    float2* okb = (float2*)p;
    p += (size_t)(kMaxBins + 1) * 8;
    double* t64 = (double*)p;
    p += ((size_t)(kMaxBins + 2) * 8 + 15) / 16 * 16;
    constexpr int kTileBytes = FP64 ? kWave * 40 : kWave * 32;
    unsigned char* tb = p + (size_t)wv * kTileBytes;
    double* tx = (double*)tb;
    double* ty = tx + kWave;
    double* tz = ty + kWave;
    float4* tl = (float4*)tb;
    double* tw = FP64 ? (tz + kWave) : (double*)(tl + kWave);
    uint32_t* tf = (uint32_t*)(tw + kWave);

    for (int k = tid; k < nb * nm; k += kWG) { g2[k] = a.g2[k]; g23[k] = a.g2[k] + a.g3[k]; }
    for (int k = tid; k < nb; k += kWG) okb[k] = make_float2(B.ok_lo[k], B.ok_hi[k]);
    for (int k = tid; k < nb + 2; k += kWG) t64[k] = B.t64[k];
    __syncthreads();

    const float rej_lo = B.rej_lo, rej_hi = B.rej_hi, ua = B.ua, ub = B.ub;
    const bool logb = B.log_bins != 0;
    const double t_lo = B.t64[0], t_hi = B.t64[nb + 1];
    const double ms = B.mu_scale;
    const float ms32 = B.ms32;
    const float dt_ew = ms32 * B.mu_ew, dt_em = ms32 * B.mu_em, dt_c = ms32 * B.mu_c;   // mu error bound
    const float nbm1f = (float)(nb - 1), nmm1f = (float)(nm - 1);
    // mu edges are the integers 1..nm-1 of t; with nm = 127 also 0 and 127, where the reference's
    // int8 store of floor(t)+1 wraps (gramsci.F90:326-328), so pairs there get the FP64 recheck
    const float e_lo = nm == 127 ? 0.0f : 1.0f, e_hi = nm == 127 ? 127.0f : nmm1f;
    const int nx = a.g.dim[0], ny = a.g.dim[1], nz = a.g.dim[2];
    const int nrow = ny * nz;
    const float h32 = a.g.h32, hx32 = a.g.hx32;    // cell edges in y/z and in x
    const double inv_wd = a.inv_wd, inv_wr = a.inv_wr;

    unsigned long long cand = 0, rechk = 0;
    const int xcd = blockIdx.x & 7;
    int tried = 0;

    while (true) {
        int item = -1;
        if (lane == 0) item = next_item(a.queue, a.n_chunks, xcd, tried);
        item = __builtin_amdgcn_readfirstlane(item);
        if (item < 0) break;

        const int row = upper_index(a.row_chunk, nrow, item);
        const int q = item - a.row_chunk[row];
        const int cy = row % ny, cz = row / ny;
        const int rs = a.cell_start[row * nx], re = a.cell_start[(row + 1) * nx];
        const int i0 = rs + q * kChunk;
        const int n_i = min(kChunk, re - i0);
        const int i = i0 + lane;
        const bool vi = lane < n_i;
        const int cx_first = a.cell[i0].x;
        const int cx_last = a.cell[i0 + n_i - 1].x;

        // FP32: cell-local coordinates, and the x cell
        auto local = [&](const double4& P, int cx, int ly, int lz) {
            return make_float4((float)(P.x - (a.g.lo[0] + cx * a.g.hx)), (float)(P.y - (a.g.lo[1] + ly * a.g.h)),
                               (float)(P.z - (a.g.lo[2] + lz * a.g.h)), (float)cx);
        };
        double4 Pi = make_double4(0, 0, 0, 0);
        float4 Li = make_float4(0, 0, 0, 0);
        uint32_t fi = 2u;
        if (vi) {
            Pi = a.pw[i];
            if constexpr (!FP64) Li = local(Pi, a.cell[i].x, cy, cz);
            fi = a.flags[i];
        }
        const int ri = fi & 1, ci = (fi & 2) ? 0 : 1;
        const float ax32 = (float)Pi.x, ay32 = (float)Pi.y, az32 = (float)Pi.z;
        double G = 0.0;

        for (int r = 0; r < a.nrows; ++r) {
            const Row rw = a.rows[r];
            const int by = cy + rw.dy, bz = cz + rw.dz;
            if (by < 0 || by >= ny || bz < 0 || bz >= nz) continue;
            const int bx0 = max(cx_first + rw.x0, 0), bx1 = min(cx_last + rw.x1, nx - 1);
            if (bx0 > bx1) continue;
            const int rb = (bz * ny + by) * nx;
            const int js = a.cell_start[rb + bx0], je = a.cell_start[rb + bx1 + 1];
            const float yi_r = Li.y - (float)rw.dy * h32;
            const float zi_r = Li.z - (float)rw.dz * h32;
            for (int jt = js; jt < je; jt += kWave) {
                const int nt = min(kWave, je - jt);
                wave_sync();
                if (lane < nt) {
                    const int j = jt + lane;
                    const double4 Pj = a.pw[j];
                    const uint32_t fj = a.flags[j];
                    if constexpr (FP64) {
                        tx[lane] = Pj.x; ty[lane] = Pj.y; tz[lane] = Pj.z;
                    } else {
                        tl[lane] = local(Pj, a.cell[j].x, by, bz);
                    }
                    tw[lane] = (fj & 1u) ? -Pj.w * inv_wr : Pj.w * inv_wd;   // normalised weight
                    tf[lane] = fj;
                }
                wave_sync();
                const int kend = vi ? nt : 0;
                cand += (unsigned long long)kend;
                for (int k = 0; k < kend; ++k) {
                    int b, m = 0, mr = 0;
                    const uint32_t fj = tf[k];
                    if constexpr (FP64) {
                        const double jx = tx[k], jy = ty[k], jz = tz[k];
                        const double s = exact_s(Pi.x, Pi.y, Pi.z, jx, jy, jz);
                        if (!(s > t_lo && s < t_hi)) continue;
                        b = adjust_bin(s, bin_estimate((float)s, logb, ua, ub), t64, nb);
                        if (b == nb) continue;
                        if constexpr (RSD) exact_mu(Pi.x, Pi.y, Pi.z, jx, jy, jz, ms, nm, m, mr);
                    } else {
                        const float4 tj = tl[k];
                        const float dx = fmaf(tj.w - Li.w, hx32, tj.x - Li.x);
                        const float dy = tj.y - yi_r, dz = tj.z - zi_r;
                        const float s = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                        if (!(s > rej_lo && s < rej_hi)) continue;
                        b = (int)__builtin_amdgcn_fmed3f(bin_estimate(s, logb, ua, ub), 0.0f, nbm1f);
                        const float2 ok = okb[b];
                        bool safe = (s >= ok.x) && (s < ok.y);
                        if constexpr (RSD) {
                            const float mx = fmaf(0.5f, dx, ax32), my = fmaf(0.5f, dy, ay32), mz = fmaf(0.5f, dz, az32);
                            const float D = -fmaf(mz, dz, fmaf(my, dy, mx * dx));
                            const float M2 = fmaf(mz, mz, fmaf(my, my, mx * mx));
                            const float rm = __builtin_amdgcn_rsqf(M2), rsq = __builtin_amdgcn_rsqf(s);
                            const float t = fmaf(D * rm * rsq, ms32, ms32);       // (theta + 1) * mu_scale
                            const float dt = fmaf(dt_ew, rsq, fmaf(dt_em, rm, dt_c));
                            // certain when the nearest mu edge (an integer 1..nm-1 of t) is farther than dt
                            const float edge = __builtin_amdgcn_fmed3f(rintf(t), e_lo, e_hi);
                            safe = safe && (dt < 0.5f) && (fabsf(t - edge) >= dt);
                            m = min((int)t, nm - 1);       // t >= 0 up to rounding; truncation = floor there
                            mr = nm - 1 - m;
                        }
                        if (!safe) {
                            ++rechk;
                            const double4 Pj = a.pw[jt + k];
                            const double se = exact_s(Pi.x, Pi.y, Pi.z, Pj.x, Pj.y, Pj.z);
                            if (!(se > t_lo && se < t_hi)) continue;
                            b = exact_bin(se, t64, nb);
                            if (b == nb) continue;
                            if constexpr (RSD) exact_mu(Pi.x, Pi.y, Pi.z, Pj.x, Pj.y, Pj.z, ms, nm, m, mr);
                        }
                    }
                    const int cj = (fj & 2) ? 0 : 1;
                    const bool rr = ri && (fj & 1);
                    const int o = b * nm;
                    const double* gt = rr ? g23 : g2;
                    double c = 0.0;
                    if (ci) c += gt[o + m];
                    if (cj) c += gt[o + mr];
                    G = fma(c, tw[k], G);
                }
            }
        }
        if (vi) a.G[a.orig[i]] = G;
    }
    for (int off = 32; off > 0; off >>= 1) {
        cand += __shfl_down(cand, off, 64);
        rechk += __shfl_down(rechk, off, 64);
    }
    if (lane == 0) {
        if (cand) atomicAdd(&a.out_stats[0], cand);
        if (rechk) atomicAdd(&a.out_stats[1], rechk);
    }
}

// Half-stencil FP32 adjoint.  The pair (i, j) contributes the same coefficient
//     c = c_i g(b, m_ij) + c_j g(b, m_ji)     (g = dL/dN2, plus dL/dN3 for a random-random pair)
// to both ends: G_i += c wn_j and G_j += c wn_i.  Every unordered pair is evaluated once, by the pair
// kernel's walk (pair2.hip) with its FP32 geometry, guard band and FP64 recheck.  The j-side sum rides along
// with the tile's entries as one more rotated register pair and is added to the neighbour's slot when
// the tile ends.  Terms are rounded to integers at the scale 2^F (|term| * 2^F <= 2^50) and summed exactly:
// at most 64 per tile and 4096 per apex and flush in 64-bit registers, and in device memory in two 64-bit
// words per point, one for the low 32 bits of the register sums and one for the rest (atomics that return
// nothing, no carries).  The result does not depend on the order of the additions and is reproducible
// bit for bit.
//
// Bound by VALU issue like the pair kernel.  Measured, before (one 64-point chunk and a whole stencil per
// item, 128-bit atomics with a returned carry) and after: 2M points, 1.9e10 binned pairs, nmu = 10: 42.6 ->
// 25.3 ms; 60k points, log bins, nmu = 4: 1.24 -> 0.19 ms.
namespace {

constexpr int kFlushTiles = 64;        // tiles between flushes of the apexes' sums

template <bool RSD, bool BUF>
struct AdjSink {
    const AdjHalfArgs& a;
    const double* g;            // LDS: coefficients c of a pair with two apexes, [class][nb * nm] (class 1: a
                                // random-random pair); BUF: then those of one direction, the same way
    int lane, nm, nbm, tiles = 0;
    double wsd, wsr;            // normalised weights times w_scale: w / Wd for data, -w / Wr for randoms
    double w[2];
    int rr[2];                  // offset of the class with a random neighbour
    bool ca[2];
    long long acc[2] = {0, 0};  // sums of the lane's apexes
    double ew = 0.0;
    int ec = 0;                 // entry: all ones for a random (BUF: bit 0 the buffer flag)
    long long eacc = 0;         // sum of the lane's entry

    __device__ __forceinline__ void region(int) {}
    __device__ __forceinline__ double wn(const double4& P, uint32_t f) const { return P.w * ((f & 1u) ? wsr : wsd); }
    __device__ __forceinline__ void apex(int which, const double4& P, uint32_t f)
    {
        w[which] = wn(P, f);
        rr[which] = (f & 1u) ? nbm : 0;
        ca[which] = !(f & 2u);
    }
    __device__ __forceinline__ void entry(const double4& P, uint32_t f)
    {
        ew = wn(P, f);
        ec = BUF ? ((f & 1u) ? ~1 : 0) | (int)((f >> 1) & 1u) : ((f & 1u) ? ~0 : 0);
        eacc = 0;
    }
    __device__ __forceinline__ void entry_of_apex()
    {
        ew = w[0];
        ec = BUF ? (rr[0] ? ~1 : 0) | (ca[0] ? 0 : 1) : (rr[0] ? ~0 : 0);
        eacc = 0;
    }
    __device__ __forceinline__ bool nothing(int which) const { return !ca[which] && (ec & 1); }
    __device__ __forceinline__ void overflow(int) {}
    __device__ __forceinline__ void add(int which, int b, int m)
    {
        int k = (int)__umul24(b, nm) + m;
        if constexpr (BUF) {
            // both ends apexes: the sum of both directions; one: its direction
            const bool ci = ca[which], cj = !(ec & 1);
            k += rr[which] & (ec >> 1);
            if (!(ci && cj)) k += 2 * nbm + (ci ? 0 : nm - 1 - 2 * m);
        } else {
            k += rr[which] & ec;
        }
        const double c = g[k];
        acc[which] += quantise_rn_signed(c * ew);
        eacc += quantise_rn_signed(c * w[which]);
    }
    __device__ __forceinline__ void to_point(int i, long long v)
    {
        atomicAdd(&a.Glo[i], (unsigned long long)v & 0xffffffffull);
        atomicAdd((unsigned long long*)&a.Ghi[i], (unsigned long long)(v >> 32));
    }
    __device__ __forceinline__ void exact_overflow(int, int) {}
    __device__ __forceinline__ void exact(int i, int j, int b, int m, int mr)
    {
        const uint32_t fi = a.flags[i], fj = a.flags[j];
        const double* g1 = a.g2;
        double c = 0.0;
        const int o = b * nm;
        auto coef = [&](int k) { return ((fi & fj & 1u) ? g1[k] + a.g3[k] : g1[k]) * a.g_scale; };
        if (!(fi & 2u)) c = coef(o + m);
        if (!(fj & 2u)) c += coef(o + mr);
        to_point(i, quantise_rn_signed(c * wn(a.pw[j], fj)));
        to_point(j, quantise_rn_signed(c * wn(a.pw[i], fi)));
    }
    __device__ __forceinline__ void rotate()
    {
        ew = rot_lane(ew);
        ec = rot_lane(ec);
        eacc = rot_lane(eacc);
    }
    __device__ __forceinline__ void tile(int, const int* jlist, int rotations, int ib, int n_i)
    {
        // this lane holds entry lane + rotations (a lane's copy of it: the copies' sums add up)
        if (eacc != 0) to_point(jlist[(lane + rotations) & (kWave - 1)], eacc);
        if (++tiles >= kFlushTiles) flush(ib, n_i);
    }
    // adds the apexes' sums to their points: lane L's second apex is lane L ^ (group / 2)'s first, and the lanes
    // L, L + group, ... hold the same apexes.  At most 2 * 64 / group lanes times kFlushTiles * group / 2
    // terms below 2^50 each: no more than 2^62.
    __device__ __forceinline__ void flush(int ib, int n_i)
    {
        long long v = acc[0] + __shfl_xor(acc[1], a.group >> 1, kWave);
        for (int off = a.group; off < kWave; off <<= 1) v += __shfl_xor(v, off, kWave);
        if (lane < n_i && v != 0) to_point(ib + lane, v);
        acc[0] = acc[1] = 0;
        tiles = 0;
    }
    __device__ __forceinline__ void piece(int ib, int n_i) { flush(ib, n_i); }
};

}  // namespace

size_t adjoint2h_lds_bytes(int nb, int nm, bool buf)
{
    return kOkBytes + (size_t)nb * nm * 8 * (buf ? 4 : 2) + (size_t)(kWG / kWave) * kListBytes;
}

template <bool RSD, bool LOGB, bool BUF>
__global__ __launch_bounds__(kWG) void k_adjoint2h(AdjHalfArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const int nb = B.nb, nm = RSD ? B.nm : 1, nbm = nb * nm;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    double* const g = (double*)(smem + kOkBytes);
    unsigned char* const lists = (unsigned char*)(g + (size_t)nbm * (BUF ? 4 : 2)) + wv * kListBytes;
    for (int k = tid; k < nbm; k += kWG) {
        const int km = k - k % nm + (nm - 1 - k % nm);      // the other direction's mu bin
        const double c2 = a.g2[k] * a.g_scale, c2m = a.g2[km] * a.g_scale;
        const double c23 = (a.g2[k] + a.g3[k]) * a.g_scale, c23m = (a.g2[km] + a.g3[km]) * a.g_scale;
        g[k] = c2 + c2m;
        g[nbm + k] = c23 + c23m;
        if constexpr (BUF) {
            g[2 * nbm + k] = c2;
            g[3 * nbm + k] = c23;
        }
    }
    fill_bin_table<false>(smem, B, tid, kWG);
    __syncthreads();

    AdjSink<RSD, BUF> sink{a};
    sink.g = g;
    sink.lane = lane;
    sink.nm = nm;
    sink.nbm = nbm;
    sink.wsd = a.inv_wd * a.w_scale;
    sink.wsr = -a.inv_wr * a.w_scale;
    WalkStats st;
    walk<false, RSD, LOGB, BUF>(a, sink, B, smem, lists, lane, wv, kWG / kWave, st);

    __shared__ unsigned long long s_stat[2];
    if (tid < 2) s_stat[tid] = 0;
    __syncthreads();
    if (lane == 0) {
        if (st.cand) atomicAdd(&s_stat[0], st.cand);
        if (st.rechk) atomicAdd(&s_stat[1], st.rechk);
    }
    __syncthreads();
    if (tid < 2 && s_stat[tid]) atomicAdd(&a.out_stats[tid], s_stat[tid]);
}

// G[orig[k]] = (Ghi * 2^32 + Glo) * 2^-F for sorted point k, converted through the magnitude of the 128-bit
// sum (both words non-negative, so no cancellation)
__global__ __launch_bounds__(256) void k_adj_fx(const unsigned long long* __restrict__ Glo,
                                                const long long* __restrict__ Ghi, const int32_t* __restrict__ orig,
                                                int64_t n, int F, double* __restrict__ G)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        unsigned long long lo = (unsigned long long)Ghi[k] << 32, hi = (unsigned long long)(Ghi[k] >> 32);
        add128(lo, hi, Glo[k], 0ull);
        const bool neg = (long long)hi < 0;
        if (neg) {
            lo = ~lo + 1ull;
            hi = ~hi + (lo == 0ull ? 1ull : 0ull);
        }
        const double v = fma((double)hi, 0x1p64, (double)lo);
        G[orig[k]] = ldexp(neg ? -v : v, -F);
    }
}

// Per-block partial sums of wn*G over data (slot 0) and randoms (slot 1); the last block to finish adds them
// up in double-double (more than the long double the host used) into part[2 gridDim.x ..] and hands the pair
// kernel's counters to the host.  stats[2] is the blocks' ticket.
__global__ __launch_bounds__(256) void k_adj_partials(const double* __restrict__ G, const double* __restrict__ w,
                                                      int64_t n, int64_t n_data, double inv_wd, double inv_wr,
                                                      double* part, unsigned long long* stats,
                                                      unsigned long long* host_stats)
{
    __shared__ double sd[256], sr[256];
    double a = 0.0, b = 0.0;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const double wk = w ? w[k] : 1.0;
        if (k < n_data) a += wk * inv_wd * G[k];
        else b += -wk * inv_wr * G[k];
    }
    sd[threadIdx.x] = a;
    sr[threadIdx.x] = b;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            sd[threadIdx.x] += sd[threadIdx.x + s];
            sr[threadIdx.x] += sr[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sd[0];
        part[2 * blockIdx.x + 1] = sr[0];
    }
    if (!last_block((unsigned*)&stats[2])) return;
    // thread t < 64: partials t, t + 64, ... of both sums, then a tree; (hi, lo) stays exact to ~2^-104
    double hi[2] = {0.0, 0.0}, lo[2] = {0.0, 0.0};
    auto add = [&](int q, double h, double l) {
        const double s = hi[q] + h, bb = s - hi[q];
        const double err = (hi[q] - (s - bb)) + (h - bb);
        hi[q] = s;
        lo[q] += err + l;
    };
    if (threadIdx.x < 64) {
        for (int k = threadIdx.x; k < (int)gridDim.x; k += 64)
            for (int q = 0; q < 2; ++q) add(q, load_agent(&part[2 * k + q]), 0.0);
        for (int off = 32; off > 0; off >>= 1)
            for (int q = 0; q < 2; ++q) {
                const double h = __shfl_down(hi[q], off, 64), l = __shfl_down(lo[q], off, 64);
                add(q, h, l);
            }
        if (threadIdx.x == 0) {
            // a non-finite sum has a NaN in lo: its hi alone is the result
            for (int q = 0; q < 2; ++q) part[2 * gridDim.x + q] = isfinite(hi[q]) ? hi[q] + lo[q] : hi[q];
            for (int q = 0; q < 2; ++q) host_stats[q] = load_agent(&stats[q]);
        }
    }
}

// sums: of wn*G over data and randoms
__global__ __launch_bounds__(256) void k_adj_finish(const double* __restrict__ G, int64_t n, int64_t n_data,
                                                    const double* __restrict__ sums, double inv_wd, double inv_wr,
                                                    double* __restrict__ out)
{
    const double s_d = sums[0], s_r = sums[1];
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
        out[k] = k < n_data ? (G[k] - s_d) * inv_wd : -(G[k] + s_r) * inv_wr;
}

// f(kernel) for the half-stencil kernel's variant
template <bool... Done, class F>
static auto with_half(bool rsd, bool logb, bool buf, F&& f)
{
    if constexpr (sizeof...(Done) == 3) {
        return f(k_adjoint2h<Done...>);
    } else {
        constexpr int k = sizeof...(Done);
        const bool b = k == 0 ? rsd : k == 1 ? logb : buf;
        return b ? with_half<Done..., true>(rsd, logb, buf, f) : with_half<Done..., false>(rsd, logb, buf, f);
    }
}

hipError_t launch_adjoint2h(const AdjHalfArgs& a, int nb, int nm, bool logb, bool buf, int nblocks, hipStream_t st)
{
    const size_t lds = adjoint2h_lds_bytes(nb, nm, buf);
    return with_half(nm >= 2, logb, buf, [&](auto kern) {
        if (lds > 64 * 1024) {
            hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kern, dim3(nblocks), dim3(kWG), lds, st, a);
        return hipGetLastError();
    });
}

int adjoint2h_occupancy(int nb, int nm, bool logb, bool buf)
{
    const size_t lds = adjoint2h_lds_bytes(nb, nm, buf);
    return with_half(nm >= 2, logb, buf, [&](auto kern) {
        int n = 0;
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return 1;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, kWG, lds);
        return e == hipSuccess && n > 0 ? n : 1;
    });
}

hipError_t launch_adj_fx(const unsigned long long* Glo, const long long* Ghi, const int32_t* orig, int64_t n, int F,
                         double* G, hipStream_t st)
{
    int nblk = (int)std::min<int64_t>((n + 255) / 256, 65535);
    if (nblk < 1) nblk = 1;
    hipLaunchKernelGGL(k_adj_fx, dim3(nblk), dim3(256), 0, st, Glo, Ghi, orig, n, F, G);
    return hipGetLastError();
}

template <bool FP64, bool RSD>
static hipError_t launch_a(const AdjArgs& a, size_t lds, int nblocks, hipStream_t st)
{
    auto kern = k_adjoint2<FP64, RSD>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(kWG), lds, st, a);
    return hipGetLastError();
}

hipError_t launch_adjoint2(const AdjArgs& a, int nb, int nm, bool fp64, bool rsd, int nblocks, hipStream_t st)
{
    const size_t lds = adjoint2_lds_bytes(nb, rsd ? nm : 1, fp64);
    if (fp64) return rsd ? launch_a<true, true>(a, lds, nblocks, st) : launch_a<true, false>(a, lds, nblocks, st);
    return rsd ? launch_a<false, true>(a, lds, nblocks, st) : launch_a<false, false>(a, lds, nblocks, st);
}

int adjoint2_occupancy(int nb, int nm, bool fp64, bool rsd)
{
    const size_t lds = adjoint2_lds_bytes(nb, rsd ? nm : 1, fp64);
    int n = 0;
    hipError_t e;
    if (fp64) e = rsd ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_adjoint2<true, true>, kWG, lds)
                      : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_adjoint2<true, false>, kWG, lds);
    else e = rsd ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_adjoint2<false, true>, kWG, lds)
                 : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_adjoint2<false, false>, kWG, lds);
    return (e == hipSuccess && n > 0) ? n : 1;
}

hipError_t launch_adj_partials(const double* G, const double* w, int64_t n, int64_t n_data, double inv_wd,
                               double inv_wr, double* part, int nblk, unsigned long long* stats,
                               unsigned long long* host_stats, hipStream_t st)
{
    hipLaunchKernelGGL(k_adj_partials, dim3(nblk), dim3(256), 0, st, G, w, n, n_data, inv_wd, inv_wr, part, stats,
                       host_stats);
    return hipGetLastError();
}

hipError_t launch_adj_finish(const double* G, int64_t n, int64_t n_data, const double* sums, double inv_wd,
                             double inv_wr, double* out, hipStream_t st)
{
    int nblk = (int)std::min<int64_t>((n + 255) / 256, 65535);
    if (nblk < 1) nblk = 1;
    hipLaunchKernelGGL(k_adj_finish, dim3(nblk), dim3(256), 0, st, G, n, n_data, sums, inv_wd, inv_wr, out);
    return hipGetLastError();
}

}  // namespace gs
