// pair2.hip -- persistent 2PCF pair kernel (binned (r, mu) DD/DR/RR counts).
//
// Replaces create_graph (gramsci.F90:288-348) + query_graph_2pcf (:352-399):
// no neighbour graph is materialised.  Each unordered pair {i, j} is visited
// once; it contributes the reference's two ordered pairs i->j and j->i (each
// only if its apex is not a buffer point, :363), with mu bins m and nmu-1-m
// (theta(j->i) = -theta(i->j) exactly).
//
// Work decomposition.  Points are sorted by cell with x fastest, so an x-row
// of cells (fixed cy, cz) is one contiguous range.  A chunk is up to `group`
// (16, 32 or 64) consecutive points of one x-row; a work item is one of
// `parts` equal shares of a chunk's candidates.  The wave reads the point
// ranges of 64 stencil rows at once (one row per lane), numbers their points
// by a prefix sum, and takes them in tiles of 64 that run across rows, so no
// tile but the last is partial.  Every lane holds two apexes and one tile
// entry; the entries rotate through the wave one lane per step (DPP), and
// group / 2 steps bring every entry to every apex: lane L holds apexes
// a = L mod group and a ^ (group / 2) and meets entries L .. L + group/2 - 1;
// the other lanes that hold apex a cover the remaining entries.  The pairs
// inside the chunk are a tile of their own (steps 1 .. group/2, half the lanes
// in the last), and the own row's candidates start after the chunk, so no pair
// needs an index test; missing apexes and entries are points far away.
// Waves are persistent and independent (no work-group barriers in the main
// loop); they pull items from 64 queues, 8 per XCD, each covering a
// contiguous z-slab of the grid so that an XCD's L2 sees one slab, and steal
// from the other queues when their own is empty.
//
// What bounds it: VALU issue.  The vector ALUs issue adds, multiplies, moves
// and 32-bit logic at about 1.55 wave-instructions per CU-cycle and everything
// else (FMA, compares, DPP moves, conversions, 3-operand integer operations) at
// about 0.95, transcendentals at 0.49 (measured), so the pair loop is written
// for few operations of the second kind.
//
// Measured (kernel time; before: one apex-tile pair of 64 points per item, a tile per stencil row, mu
// from the midpoint with two reciprocal square roots, a u32 and two u64 atomics per update):
//   4M points, 1.90e11 binned pairs, (r, mu), weighted:  FP32 252 -> 183 ms
//   800k points, same bins, FP64 geometry:               142 -> 46 ms
//   60k points, 10 linear bins, unweighted:              0.51 -> 0.08 ms
//   9k points, (r, mu), weighted:                        0.38 -> 0.04 ms
// The small ones were bound by the few items (150 chunks of 64 points, each walking the whole stencil) and
// by device-wide atomics on shared lines: the queue's end, the drains and the statistics.
//
// Precision variants (identical counts):
//   FP64        s = |xj-xi|^2 in FP64 exactly as the reference, bins from the
//               exact thresholds; the mu bin from a FP64 estimate that is
//               taken only when it is farther from a mu edge than its error
//               bound, else with the reference's IEEE sqrt and division.
//   FP32 guard  coordinates relative to a point of the chunk, rounded to FP32.
//               A pair is binned directly only when s32 lies in the bin's
//               certain interval [ok_lo, ok_hi) and its mu is farther than a
//               rigorous error bound from a mu edge; otherwise it is
//               queued in LDS and re-evaluated in FP64, 64 at a time.
//
// mu from squared radii: with D = 2(|xi|^2 - |xj|^2) and
// S = |xi + xj|^2 = 2|xi|^2 + 2|xj|^2 - s, theta = mid.sep / (|mid| |sep|)
// = (D/2) rsq(S s): one transcendental and no midpoint.  The squared radii are
// taken relative to the chunk's reference point p (formed in FP64 as
// (x - p).(x + p)), so that D keeps its precision far from the origin.  The
// error bound of t = (theta + 1) mu_scale is k0 + k1 q + k2 q^2 with
// q = rsq(S s) = 1 / (2 |mid| |sep|); see fill_bins.
//
// Histograms live in LDS, shared by the work-group's waves and replicated
// `reps` times (replica = lane % reps).  Unweighted: u32 counts.  Weighted:
// per bin two u64 planes, lo += q mod 2^32 and hi += (q >> 32) + 2^42, where
// q < 2^52 is the weight product in fixed point: the sum is lo + 2^32 (hi mod
// 2^42) and the count hi >> 42 -- two LDS atomics per update, no carries and
// no returning atomics.  A bin overflows after 2^22 increments: a wave that may
// have issued 2^20 / (waves of the work-group) increments since it last looked
// scans the histogram and drains the bins that hold 2^20 or more.
//
// Without buffer points every pair counts in both directions, so one update at
// mu bin m stands for both ordered pairs; k_pair_reduce adds entry m to m and
// nm-1-m (plane 0 of the outputs).  Pairs exactly on a mu edge, where the two
// directions are not mirror images, are added explicitly (plane 1).  With
// buffer points a pair with one apex goes to plane 1 in the apex's direction.
#include <type_traits>

#include "gs_device.h"
#include "gs_kernels.h"

namespace gs {

namespace {

using namespace dev;

constexpr int kOkBytes = (kMaxBins + 1) * 8;    // certain intervals, at the start of the LDS
constexpr int kListBytes = kWave * 12;          // per wave: queue of pairs to re-evaluate, tile index list
constexpr uint32_t kCountOne = 1u << 10;        // one count in the high word of the hi plane (bit 42)
constexpr unsigned kRunMax = 256;               // increments after which a run ends with its tile

template <class R> struct Real4;                // point in the kernel's geometry precision
template <> struct Real4<float> { static constexpr float far = 1e18f; };
template <> struct Real4<double> { static constexpr double far = 1e150; };

// one apex of a lane
template <class R>
struct Apex {
    R x, y, z;      // FP32: relative to the chunk's reference point; FP64: absolute
    R d;            // 2 (|x|^2 - |p|^2), p the reference point
    R c;            // 2 (|x|^2 + |p|^2)
    double w;       // weight scaled by its class's 2^F
    int cb;         // LDS offset of the pair's class with a data neighbour, with the lane's replica
};

// a lane's run of histogram increments to one bin, merged in registers
struct Run {
    int k;                  // LDS offset of the bin
    uint32_t lo, hi, cn;    // sum of q (split at bit 32), count * kCountOne
};

__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsq(double x) { return __builtin_amdgcn_rsq(x); }
__device__ __forceinline__ float fract(float x) { return __builtin_amdgcn_fractf(x); }
__device__ __forceinline__ double fract(double x) { return __builtin_amdgcn_fract(x); }

// v truncated to an unsigned integer, 0 for a negative v (the conversion saturates)
__device__ __forceinline__ int cvt_sat(float v)
{
    int r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

__device__ __forceinline__ int lane_int(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double lane_double(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = lane_int((int)(b & 0xffffffffll), l), hi = lane_int((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (long long)(uint32_t)lo);
}

}  // namespace

// LDS of one histogram: bins (with a plane per direction where `planes` is 2) times replicas
static size_t hist_bytes(size_t nbt, int planes, int reps, bool weighted)
{
    return ((size_t)planes * nbt * reps * (weighted ? 16 : 4) + 15) / 16 * 16;
}

size_t pair2_lds_bytes(int nb, int nm, int planes, int reps, bool weighted, bool batched, int wg)
{
    const size_t nbt = (size_t)3 * nb * nm;
    const size_t waves = (size_t)(wg / kWave);
    return kOkBytes + hist_bytes(nbt, planes, reps, weighted) * (batched ? waves : 1) + waves * kListBytes;
}

template <bool FP64, bool RSD, bool W, bool LOGB, bool BUF>
__global__ __launch_bounds__(1024) void k_pair2(PairArgs a)
{
    using R = std::conditional_t<FP64, double, float>;
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const int nb = B.nb;
    const int nm = RSD ? B.nm : 1;
    const int nbt = 3 * nb * nm;
    const bool batched = a.nreg > 0;
    const int reps = a.reps;
    const int planes = BUF ? a.planes : 1;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int nthr = blockDim.x;        // a multiple of 64, at most 1024
    const int nwv = nthr / kWave;

    // LDS: certain intervals (FP64: exact thresholds), histogram (one, or one per wave in batched mode),
    // tile index lists
    constexpr int kB = W ? 8 : 4;       // bytes of a histogram word
    const int nent = planes * nbt * reps;                       // words of one plane of the histogram
    const int hsize = (int)((nent * (W ? 16 : 4) + 15) / 16 * 16);
    unsigned char* const hist = smem + kOkBytes + (batched ? wv * hsize : 0);   // this wave's histogram
    const int hi_off = nent * 8;        // W: the hi plane's offset from the lo plane
    unsigned char* const lists = smem + kOkBytes + (size_t)hsize * (batched ? nwv : 1) + wv * kListBytes;
    int2* const queue = (int2*)lists;                   // pairs to re-evaluate
    int* const jlist = (int*)(lists + kWave * 8);       // point of each tile entry
    {
        uint32_t* h0 = (uint32_t*)(smem + kOkBytes);
        const int nw = hsize / 4 * (batched ? nwv : 1);
        for (int k = tid; k < nw; k += nthr) h0[k] = 0;
        if constexpr (FP64) {
            for (int k = tid; k <= nb && k <= kMaxBins; k += nthr) ((double*)smem)[k] = B.t64[k];
        } else {
            // entry nb (an estimate just past the last bin) is never certain
            for (int k = tid; k <= nb; k += nthr)
                ((float2*)smem)[k] = k < nb ? make_float2(B.ok_lo[k], B.ok_hi[k]) : make_float2(INFINITY, -INFINITY);
        }
    }
    __syncthreads();

    const float ua = B.ua, ub = B.ub;
    const R rej_lo = FP64 ? (R)B.t64[0] : (R)B.rej_lo, rej_hi = FP64 ? (R)B.t64[nb + 1] : (R)B.rej_hi;
    const double t_lo = B.t64[0], t_hi = B.t64[nb + 1];
    const double ms = B.mu_scale;
    const R msr = (R)ms, hms = (R)(0.5 * ms);
    // fixed-point scales of data and random weights (batched: the current region's)
    int sd = B.fx_sd, sr = B.fx_sr;
    const int nbm = nb * nm;
    const int n_chunks = *a.n_chunks_dev;
    const int n_items = n_chunks << a.lg_parts;
    const int group = a.group, half = group >> 1;
    const int ai = lane & (group - 1), ai2 = ai ^ half;     // the lane's apexes in the chunk
    const int rep_off = (lane & (reps - 1)) * planes * nbt * kB;
    const float cap = a.cap_cells;
    int nx = a.g.dim[0], ny = a.g.dim[1], nz = a.g.dim[2], cb = 0;
    int cur_r = batched ? -1 : 0;   // region of this wave's histogram

    unsigned long long n_cand = 0;
    unsigned long long n_rechk = 0;
    unsigned int n_over = 0;

    // the work-group's copy of the outputs: [2][nbt] counts and [2][nbt][2] sums of the current region
    const size_t copy = (size_t)(blockIdx.x & (unsigned)(a.copies - 1)) * (size_t)a.copy_stride;
    unsigned long long* out_cnt = a.out_cnt + copy;
    unsigned long long* out_w = a.out_w + copy;

    // adds word k (of this wave's histogram) to the outputs and clears it
    auto drain_word = [&](int k) {
        // with buffer points and a single plane every entry is one direction of a pair: plane 1
        const int o = k % (planes * nbt) + (BUF && planes == 1 ? nbt : 0);
        if constexpr (W) {
            const unsigned long long h = atomicExch((unsigned long long*)(hist + hi_off) + k, 0ull);
            const unsigned long long l = atomicExch((unsigned long long*)hist + k, 0ull);
            if (h | l) {
                const unsigned long long hs = h & ((1ull << 42) - 1);
                const unsigned long long L = (hs << 32) + l;
                const unsigned long long H = (hs >> 32) + (L < l ? 1ull : 0ull);
                atomicAdd(&out_cnt[o], h >> 42);
                glb_add128(&out_w[2 * o], L, H);
            }
        } else {
            const uint32_t c = atomicExch((uint32_t*)hist + k, 0u);
            if (c) atomicAdd(&out_cnt[o], (unsigned long long)c);
        }
    };
    auto drain = [&](int t0, int stride) {
        for (int k = t0; k < nent; k += stride) drain_word(k);
    };

    Run r1{rep_off, 0u, 0u, 0u}, r2{rep_off, 0u, 0u, 0u};
    auto flush = [&](Run& r) {
        atomicAdd((unsigned long long*)(hist + r.k), (unsigned long long)r.lo);
        atomicAdd((unsigned long long*)(hist + r.k + hi_off), ((unsigned long long)r.cn << 32) | r.hi);
        r.lo = 0; r.hi = 0; r.cn = 0;
    };
    // one increment of the bin at LDS offset k: merged with the lane's run of that bin (a lane's
    // consecutive neighbours often share a bin), which is written out when the bin changes.  An empty
    // run adds zeros.
    auto put = [&](Run& r, int k, uint32_t qlo, uint32_t qhi) {
        if (k != r.k) {
            flush(r);
            r.k = k;
        }
        const uint32_t s = r.lo + qlo;
        r.hi += qhi + (s < qlo ? 1u : 0u);
        r.lo = s;
        r.cn += kCountOne;
    };

    // Pairs that are not certain wait in LDS (apex point, neighbour) and are re-evaluated together, with the
    // reference's arithmetic, when 64 are full or the wave changes region or ends: the loop over the
    // pairs keeps few registers, and a recheck fills a wave instead of one lane.
    int nq = 0;
    auto recheck = [&]() {
        wave_sync();
        if (lane < nq) {
            const int2 pr = queue[lane];
            const double4 Pi = a.pw[pr.x], Pj = a.pw[pr.y];
            const uint32_t fi = a.flags[pr.x], fj = a.flags[pr.y];
            const double se = exact_s(Pi.x, Pi.y, Pi.z, Pj.x, Pj.y, Pj.z);
            if (se > t_lo && se < t_hi) {
                const bool ci = !(fi & 2u), cj = !(fj & 2u);
                const int b = adjust_bin(se, bin_estimate((float)se, LOGB, ua, ub), B.t64, nb);
                if (b == nb) {
                    n_over += (unsigned)ci + (unsigned)cj;
                } else {
                    int m = 0, mr = 0;
                    if constexpr (RSD) exact_mu(Pi.x, Pi.y, Pi.z, Pj.x, Pj.y, Pj.z, ms, nm, m, mr);
                    unsigned long long q = 0;
                    if constexpr (W) q = quantise_rn(ldexp(Pi.w, (fi & 1u) ? sr : sd) * ldexp(Pj.w, (fj & 1u) ? sr : sd));
                    const int k0 = (int)((fi & 1u) + (fj & 1u)) * nbm + b * nm;
                    auto add = [&](int k) {
                        if constexpr (W) {
                            unsigned long long* h = (unsigned long long*)(hist + rep_off) + k;
                            atomicAdd(h, q & 0xffffffffull);
                            atomicAdd(h + nent, (q >> 32) + (1ull << 42));
                        } else {
                            atomicAdd((uint32_t*)(hist + rep_off) + k, 1u);
                        }
                    };
                    auto add_global = [&](int k) {
                        atomicAdd(&out_cnt[nbt + k], 1ull);
                        if constexpr (W) glb_add128(&out_w[2 * (nbt + k)], q, 0ull);
                    };
                    if (ci && cj && mr == nm - 1 - m && !(BUF && planes == 1)) {
                        add(k0 + m);
                    } else if (BUF && planes == 2 && ci != cj) {
                        add(k0 + (ci ? m : mr) + nbt);
                    } else {        // exactly on a mu edge (or one plane): the ordered pairs one by one
                        if (ci) add_global(k0 + m);
                        if (cj) add_global(k0 + mr);
                    }
                }
            }
        }
        n_rechk += (unsigned)nq;
        nq = 0;
        wave_sync();
    };

    // increments this wave may have issued since it last looked at its histogram
    unsigned long long bound = 0;
    const unsigned long long look_at = (W ? (1ull << 20) : (1ull << 31)) / (unsigned long long)(batched ? 1 : nwv);
    auto look = [&]() {
        if constexpr (W) {
            flush(r1);
            flush(r2);
            for (int k = lane; k < nent; k += kWave)
                if ((((unsigned long long*)(hist + hi_off))[k] >> 42) >= (1u << 20)) drain_word(k);
        } else {
            drain(lane, kWave);
        }
        bound = 0;
    };

    ItemQueue items(a.queue, n_items, nwv);
    while (true) {
        const int item = items.next(lane, wv);
        if (item < 0) break;
        const int part = item & ((1 << a.lg_parts) - 1);
        const int4 ch = a.chunks[item >> a.lg_parts];
        const int row = __builtin_amdgcn_readfirstlane(ch.z);
        if (batched) {
            const int rg = __builtin_amdgcn_readfirstlane(ch.w);
            if (rg != cur_r) {
                if (nq) recheck();
                if constexpr (W) { flush(r1); flush(r2); }
                if (cur_r >= 0) drain(lane, kWave);
                cur_r = rg;
                const RegionDesc& rd = a.regions[rg];
                nx = rd.dim[0]; ny = rd.dim[1]; nz = rd.dim[2];
                cb = rd.cell_base;
                sd = rd.fx_shift;
                sr = rd.fx_shift_rand;
                out_cnt = a.out_cnt + copy + (size_t)rg * 2 * nbt;
                out_w = a.out_w + copy + (size_t)rg * 4 * nbt;
                bound = 0;
            }
        }
        const int cy = row % ny, cz = row / ny;
        int ib = __builtin_amdgcn_readfirstlane(ch.x);
        const int iend = ib + __builtin_amdgcn_readfirstlane(ch.y);

        // The FP32 error bounds hold for chunks of at most cap + 1 cells in x: a longer one (few points
        // in a long row) is taken in pieces [ib, ib + n_i).
        int n_i;
        for (; ib < iend; ib += n_i) {
            const float cxl = ib + ai < iend ? a.pl[ib + ai].w : INFINITY;
            const int cx_first = (int)__int_as_float(lane_int(__float_as_int(cxl), 0));
            n_i = __popcll(__ballot(lane < group && cxl - (float)cx_first <= cap));
            const int cx_last = (int)__int_as_float(lane_int(__float_as_int(cxl), n_i - 1));

            // ---- the lane's apexes, relative to the chunk's middle point
            double4 P1 = make_double4(0, 0, 0, 0), P2 = P1;
            uint32_t f1 = 2u, f2 = 2u;
            const bool v1 = ai < n_i, v2 = ai2 < n_i;
            if (v1) { P1 = a.pw[ib + ai]; f1 = a.flags[ib + ai]; }
            if (v2) { P2 = a.pw[ib + ai2]; f2 = a.flags[ib + ai2]; }
            const int mid = n_i >> 1;
            const double px = lane_double(P1.x, mid), py = lane_double(P1.y, mid), pz = lane_double(P1.z, mid);
            const double p2 = px * px + py * py + pz * pz;
            // 2 (|x|^2 - |p|^2)
            auto d_of = [&](const double4& P) {
                return 2.0 * ((P.x - px) * (P.x + px) + (P.y - py) * (P.y + py) + (P.z - pz) * (P.z + pz));
            };
            auto apex = [&](const double4& P, uint32_t f, bool v) {
                Apex<R> A;
                if constexpr (FP64) { A.x = P.x; A.y = P.y; A.z = P.z; }
                else { A.x = (float)(P.x - px); A.y = (float)(P.y - py); A.z = (float)(P.z - pz); }
                const double d = d_of(P);
                A.d = (R)d;
                A.c = (R)(d + 4.0 * p2);
                A.w = W ? ldexp(P.w, (f & 1u) ? sr : sd) : 0.0;
                A.cb = rep_off + ((f & 1u) ? nbm * kB : 0);
                if (!v) A.x = Real4<R>::far;
                return A;
            };
            const Apex<R> A1 = apex(P1, f1, v1), A2 = apex(P2, f2, v2);
            const bool c1 = !(f1 & 2u), c2 = !(f2 & 2u);        // may be an apex of the reference
            const bool chunk_buf = BUF && __ballot(c1) == 0;
            // error bound of t for this chunk (wave-uniform): k0 + k1 q + k2 q^2, and the distance from
            // the nearest integer is tested as |fract(t) - 1/2| <= 1/2 - bound
            R l0 = 0, l1 = 0, l2 = 0;
            if constexpr (RSD) {
                const float rho = (float)sqrt(p2) * 1.001f;
                const float sx = 2.0f * rho + B.mu_ab;
                l0 = (R)(0.5f - B.mu_k0);
                l1 = (R)(-(B.mu_k1a * sx + B.mu_k1b * (2.0f * rho + 3.0f * B.mu_ab)));
                l2 = (R)(-(B.mu_k2a + B.mu_k2b * sx * sx));
            }

            // ---- tile entry of the lane
            R ex = 0, ey = 0, ez = 0, ed = 0;
            double ew = 0.0;
            int ec = 0;         // class offset of a random entry; BUF: times 2, plus the buffer flag

            // pair of apex A with the lane's entry: binned, or true if it has to be re-evaluated
            auto visit1 = [&](const Apex<R>& A, const bool ca, Run& run) __attribute__((always_inline)) -> bool {
                R s;
                if constexpr (FP64) {
                    s = exact_s(A.x, A.y, A.z, ex, ey, ez);
                } else {
                    const float dx = ex - A.x, dy = ey - A.y, dz = ez - A.z;
                    s = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                }
                if (!(s > rej_lo && s < rej_hi)) return false;
                if (BUF && !ca && (ec & 1)) return false;     // two buffer points
                int b;
                bool safe;
                if constexpr (FP64) {
                    const float u = bin_estimate((float)s, LOGB, ua, ub);
                    b = min(cvt_sat(u), nb - 1);
                    const double* t = (const double*)smem;
                    if (!(s >= t[b] && s < t[b + 1])) {
                        while (b > 0 && s < t[b]) --b;
                        while (b < nb && s >= t[b + 1]) ++b;
                        if (b == nb) {
                            n_over += (unsigned)ca + (BUF ? 1u - (unsigned)(ec & 1) : 1u);
                            return false;
                        }
                    }
                    safe = true;
                } else {
                    b = cvt_sat(bin_estimate(s, LOGB, ua, ub));
                    const float2 ok = ((const float2*)smem)[b];
                    safe = s >= ok.x && s < ok.y;
                }
                int m = 0;
                if constexpr (RSD) {
                    const R S = (A.c + ed) - s;
                    const R q = rsq(S * s);
                    const R t = fma((A.d - ed) * q, hms, msr);
                    const R lim = fma(fma(l2, q, l1), q, l0);
                    // the negated form also leaves a NaN (mid-point at the origin) to the recheck
                    safe = safe && fabs(fract(t) - (R)0.5) <= lim;
                    m = (int)t;
                }
                if (!safe) return true;
                const int k0 = A.cb + (BUF ? ec >> 1 : ec) + (int)__umul24(b, (unsigned)(nm * kB));
                uint32_t qlo = 0, qhi = 0;
                if constexpr (W) {
                    const unsigned long long q = quantise_rn(A.w * ew);
                    qlo = (uint32_t)q;
                    qhi = (uint32_t)(q >> 32);
                }
                if constexpr (!BUF) {
                    const int kk = k0 + m * kB;
                    if constexpr (W) put(run, kk, qlo, qhi);
                    else atomicAdd((uint32_t*)(hist + kk), 1u);
                } else {
                    // both ends apexes: plane 0; one: plane 1 in its direction
                    const bool cj = !(ec & 1);
                    const int mr = nm - 1 - m;
                    if (planes == 2) {
                        const int kk = k0 + (ca ? m : mr) * kB + (ca && cj ? 0 : nbt * kB);
                        if constexpr (W) put(run, kk, qlo, qhi);
                        else atomicAdd((uint32_t*)(hist + kk), 1u);
                    } else {        // histograms too large for two planes: plane 1 only, each direction added
                        if (ca) {
                            if constexpr (W) put(run, k0 + m * kB, qlo, qhi);
                            else atomicAdd((uint32_t*)(hist + k0 + m * kB), 1u);
                        }
                        if (cj) {
                            if constexpr (W) put(run, k0 + mr * kB, qlo, qhi);
                            else atomicAdd((uint32_t*)(hist + k0 + mr * kB), 1u);
                        }
                    }
                }
                return false;
            };
            // ... and queued if so: entry number (lane + k) & 63 of the tile, apex point ia
            auto visit = [&](const Apex<R>& A, const bool ca, const int ia, const int k, Run& run, const bool on)
                             __attribute__((always_inline)) {
                bool un = false;
                if (on) un = visit1(A, ca, run);
                if constexpr (RSD || !FP64) {
                    const unsigned long long um = __ballot(un);
                    if (um) {
                        const int nu = __popcll(um);
                        if (nq + nu > kWave) recheck();
                        if (un) {
                            const int at = nq + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(um >> 32),
                                                                              __builtin_amdgcn_mbcnt_lo((unsigned)um, 0u));
                            queue[at] = make_int2(ia, jlist[(lane + k) & (kWave - 1)]);
                        }
                        nq += nu;
                    }
                }
            };
            auto rotate = [&]() __attribute__((always_inline)) {
                ex = rot_lane(ex); ey = rot_lane(ey); ez = rot_lane(ez);
                if constexpr (RSD) ed = rot_lane(ed);
                if constexpr (W) ew = rot_lane(ew);
                ec = rot_lane(ec);
            };
            auto entry_class = [&](uint32_t f) {
                const int c = (f & 1u) ? nbm * kB : 0;
                return BUF ? (c << 1) | (int)((f >> 1) & 1u) : c;
            };
            auto tile_done = [&](int nt) {
                bound += (unsigned long long)nt * (BUF && planes == 1 ? 2u : 1u);
                if constexpr (W) {
                    if (r1.cn >= kRunMax * kCountOne) flush(r1);
                    if (r2.cn >= kRunMax * kCountOne) flush(r2);
                }
                if (bound > look_at) look();
            };

            // ---- pairs inside the chunk
            if (part == 0) n_cand += (unsigned long long)(n_i * (n_i - 1) / 2);
            if (part == 0 && !chunk_buf) {
                ex = v1 ? A1.x : -Real4<R>::far; ey = A1.y; ez = A1.z; ed = A1.d; ew = A1.w;
                ec = entry_class(f1);
                wave_sync();
                jlist[lane] = ib + min(ai, n_i - 1);
                wave_sync();
                for (int k = 1; k <= half; ++k) {
                    rotate();
                    visit(A1, c1, ib + ai, k, r1, lane < (k < half ? group : half));
                }
                tile_done(n_i * (n_i - 1) / 2);
            }

            // ---- the other points of the half stencil
            for (int r0 = 0; r0 < a.nrows; r0 += kWave) {
                int js = 0, len = 0;
                if (r0 + lane < a.nrows) {
                    const Row rw = a.rows[r0 + lane];
                    const int by = cy + rw.dy, bz = cz + rw.dz;
                    const int bx0 = max(cx_first + rw.x0, 0), bx1 = min(cx_last + rw.x1, nx - 1);
                    if (by >= 0 && by < ny && bz >= 0 && bz < nz && bx0 <= bx1) {
                        const int rb = cb + (bz * ny + by) * nx;
                        js = a.cell_start[rb + bx0];
                        const int je = a.cell_start[rb + bx1 + 1];
                        if (rw.dy == 0 && rw.dz == 0) js = max(js, ib + n_i);
                        len = max(je - js, 0);
                    }
                }
                int incl = len;
                for (int off = 1; off < kWave; off <<= 1) {
                    const int y = __shfl_up(incl, off, kWave);
                    if (lane >= off) incl += y;
                }
                const int excl = incl - len;
                const int total = lane_int(incl, kWave - 1);
                const int tiles = (total + kWave - 1) / kWave;
                const int t1 = (int)(((long long)tiles * (part + 1)) >> a.lg_parts);
                int t = (int)(((long long)tiles * part) >> a.lg_parts);
                for (; t < t1; ++t) {
                    // the lane's entry: its point, from the row of this tile it falls into
                    const int c0 = t * kWave, my = c0 + lane;
                    const int nt = min(kWave, total - c0);
                    const bool has = lane < nt;
                    int j = ib;
                    unsigned long long rows = __ballot(incl > c0 && excl < c0 + kWave && len > 0);
                    while (rows) {
                        const int r = (int)__builtin_ctzll(rows);
                        rows &= rows - 1;
                        const int e0 = lane_int(excl, r), j0 = lane_int(js, r);
                        if (my >= e0) j = j0 + (my - e0);
                    }
                    if (!has) j = ib;
                    n_cand += (unsigned long long)(n_i * nt);
                    const uint32_t f = a.flags[j];
                    if (chunk_buf && __ballot(has && !(f & 2u)) == 0) continue;
                    const double4 P = a.pw[j];
                    if constexpr (FP64) { ex = P.x; ey = P.y; ez = P.z; }
                    else { ex = (float)(P.x - px); ey = (float)(P.y - py); ez = (float)(P.z - pz); }
                    if constexpr (RSD) ed = (R)d_of(P);
                    if constexpr (W) ew = ldexp(P.w, (f & 1u) ? sr : sd);
                    ec = entry_class(f);
                    if (!has) ex = -Real4<R>::far;
                    wave_sync();
                    jlist[lane] = j;
                    wave_sync();
                    for (int k = 0; k < half; ++k) {
                        visit(A1, c1, ib + ai, k, r1, true);
                        visit(A2, c2, ib + ai2, k, r2, true);
                        rotate();
                    }
                    tile_done(n_i * nt);
                }
            }
        }
    }
    if (nq) recheck();
    if constexpr (W) { flush(r1); flush(r2); }
    if (batched) {
        if (cur_r >= 0) drain(lane, kWave);
    } else {
        __syncthreads();
        drain(tid, nthr);
    }

    // statistics (candidates and rechecks are counted per wave, overflow pairs per lane), one atomic per
    // work-group each
    unsigned long long ov = n_over;
    for (int off = 32; off > 0; off >>= 1) ov += __shfl_down(ov, off, 64);
    __shared__ unsigned long long s_stat[3];
    if (tid < 3) s_stat[tid] = 0;
    __syncthreads();
    if (lane == 0) {
        if (n_cand) atomicAdd(&s_stat[0], n_cand);
        if (n_rechk) atomicAdd(&s_stat[1], n_rechk);
        if (ov) atomicAdd(&s_stat[2], ov);
    }
    __syncthreads();
    if (tid < 3 && s_stat[tid]) atomicAdd(&a.out_stats[copy + tid], s_stat[tid]);
}

// Sums the copies of the outputs and folds their two planes: counts [nreg][nbt] and 128-bit sums
// [nreg][nbt][2] over ordered pairs, and the statistics.  Every work-group drains its histogram with
// device-wide atomics, which run one after another where they meet (about 40 ns each): with one copy
// the drains of a small catalogue's 2048 work-groups into 30 bins took 1.3 ms, longer than its pairs.
// One wave per entry, one lane per copy.
__global__ __launch_bounds__(256) void k_pair_reduce(const unsigned long long* __restrict__ in, int copies,
                                                     int64_t copy_stride, int nreg, int nbt, int nm, int weighted,
                                                     unsigned long long* __restrict__ out)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t e = blockIdx.x * (int64_t)(blockDim.x / kWave) + threadIdx.x / kWave;
    const int64_t ne = (int64_t)nreg * nbt;
    const unsigned long long* c = in + (size_t)lane * (size_t)copy_stride;
    if (e < ne) {
        const int64_t r = e / nbt;
        const int k = (int)(e % nbt);
        const int km = k - k % nm + (nm - 1 - k % nm);
        unsigned long long n = 0, lo = 0, hi = 0;
        if (lane < copies) {
            const unsigned long long* cc = c + r * 2 * nbt;
            n = cc[k] + cc[km] + cc[nbt + k];
            if (weighted) {
                const unsigned long long* cw = c + ne * 2 + r * 4 * nbt;
                add128(lo, hi, cw[2 * k], cw[2 * k + 1]);
                add128(lo, hi, cw[2 * km], cw[2 * km + 1]);
                add128(lo, hi, cw[2 * (nbt + k)], cw[2 * (nbt + k) + 1]);
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            n += __shfl_down(n, off, 64);
            const unsigned long long l = __shfl_down(lo, off, 64), h = __shfl_down(hi, off, 64);
            add128(lo, hi, l, h);
        }
        if (lane == 0) {
            out[e] = n;
            out[ne + 2 * e] = lo;
            out[ne + 2 * e + 1] = hi;
        }
    } else if (e == ne) {
        for (int q = 0; q < 4; ++q) {
            unsigned long long v = lane < copies ? c[6 * ne + q] : 0;
            for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
            if (lane == 0) out[3 * ne + q] = v;
        }
    }
}

hipError_t launch_pair_reduce(const unsigned long long* in, int copies, int nreg, int nbt, int nm, bool weighted,
                              unsigned long long* out, hipStream_t st)
{
    const int64_t ne = (int64_t)nreg * nbt;
    const int64_t nblk = (ne + 1 + kWG / kWave - 1) / (kWG / kWave);
    hipLaunchKernelGGL(k_pair_reduce, dim3((unsigned)nblk), dim3(kWG), 0, st, in, copies, pair_copy_words(nreg, nbt),
                       nreg, nbt, nm, weighted ? 1 : 0, out);
    return hipGetLastError();
}

template <bool FP64, bool RSD, bool W, bool LOGB, bool BUF>
struct Pair2 {
    static hipError_t launch(const PairArgs& a, size_t lds, int nblocks, int wg, hipStream_t st)
    {
        auto kern = k_pair2<FP64, RSD, W, LOGB, BUF>;
        if (lds > 64 * 1024) {
            hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kern, dim3(nblocks), dim3(wg), lds, st, a);
        return hipGetLastError();
    }
    static int occupancy(size_t lds, int wg)
    {
        int nb = 0;
        auto kern = k_pair2<FP64, RSD, W, LOGB, BUF>;
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, wg, lds) != hipSuccess) return 1;
        return nb;
    }
};

// f(Pair2<...>{}) for the variant v
template <bool... Done, class F>
static auto with_variant(const PairVariant& v, F&& f)
{
    if constexpr (sizeof...(Done) == 5) {
        return f(Pair2<Done...>{});
    } else {
        constexpr int k = sizeof...(Done);
        const bool b = k == 0 ? v.fp64 : k == 1 ? v.nm >= 2 : k == 2 ? v.weighted : k == 3 ? v.logb : v.buf;
        return b ? with_variant<Done..., true>(v, f) : with_variant<Done..., false>(v, f);
    }
}

hipError_t launch_pair2(const PairArgs& a, const PairVariant& v, int nblocks, int wg, hipStream_t st)
{
    const size_t lds = pair2_lds_bytes(v.nb, v.nm, v.buf ? a.planes : 1, a.reps, v.weighted, a.nreg > 0, wg);
    return with_variant(v, [&](auto k) { return k.launch(a, lds, nblocks, wg, st); });
}

int pair2_occupancy(const PairVariant& v, int planes, int reps, bool batched, int wg)
{
    const size_t lds = pair2_lds_bytes(v.nb, v.nm, planes, reps, v.weighted, batched, wg);
    if (lds > kPairLdsMax) return 0;
    return with_variant(v, [&](auto k) { return k.occupancy(lds, wg); });
}

// ---------------------------------------------------------------- chunks
// Descriptors of the pair kernels' chunks: {first point, points, x-row in its region, region}.
__global__ __launch_bounds__(256) void k_chunks(const int32_t* __restrict__ row_chunk, int nrow,
                                                const int32_t* __restrict__ cell_start, int nx,
                                                const RegionDesc* __restrict__ regions,
                                                const int32_t* __restrict__ row_base, int nreg, int group,
                                                int4* __restrict__ out)
{
    const int n = row_chunk[nrow];
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
        const int grow = upper_index(row_chunk, nrow, c);
        int row = grow, r = 0, c0, dim = nx;
        if (nreg > 0) {
            r = upper_index(row_base, nreg, grow);
            row = grow - regions[r].row_base;
            dim = regions[r].dim[0];
            c0 = regions[r].cell_base + row * dim;
        } else {
            c0 = row * dim;
        }
        const int i0 = cell_start[c0] + (c - row_chunk[grow]) * group;
        out[c] = make_int4(i0, min(group, cell_start[c0 + dim] - i0), row, r);
    }
}

hipError_t launch_chunks(const int32_t* row_chunk, int nrow, const int32_t* cell_start, int nx,
                         const RegionDesc* regions, const int32_t* row_base, int nreg, int group, int64_t max_chunks,
                         int4* out, hipStream_t st)
{
    int64_t nblk = (max_chunks + 255) / 256;
    if (nblk > 4096) nblk = 4096;
    if (nblk < 1) nblk = 1;
    hipLaunchKernelGGL(k_chunks, dim3((unsigned)nblk), dim3(256), 0, st, row_chunk, nrow, cell_start, nx, regions,
                       row_base, nreg, group, out);
    return hipGetLastError();
}

}  // namespace gs
