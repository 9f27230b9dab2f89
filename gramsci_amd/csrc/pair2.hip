// pair2.hip -- persistent 2PCF pair kernel (binned (r, mu) DD/DR/RR counts).
//
// Replaces create_graph (gramsci.F90:288-348) + query_graph_2pcf (:352-399):
// no neighbour graph is materialised.  Each unordered pair {i, j} is visited
// once; it contributes the reference's two ordered pairs i->j and j->i (each
// only if its apex is not a buffer point, :363), with mu bins m and nmu-1-m
// (theta(j->i) = -theta(i->j) exactly).
//
// Work decomposition.  Points are sorted by cell with x fastest, so an x-row
// of cells (fixed cy, cz) is one contiguous range.  A chunk is `group` (16, 32
// or 64) consecutive points, taken in pieces of one x-row; a work item is one
// of `parts` equal shares of a chunk's candidates.  The wave reads the point
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
//   4M points, 1.90e11 binned pairs, (r, mu), weighted:  FP32 252 -> 171 ms
//   800k points, same bins, FP64 geometry:               142 -> 47 ms
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
#include "gs_pair_tiles.h"

namespace gs {

namespace {

using namespace dev;

constexpr uint32_t kCountOne = 1u << 10;        // one count in the high word of the hi plane (bit 42)
constexpr unsigned kRunMax = 256;               // increments after which a run ends with its tile

// a lane's run of histogram increments to one bin, merged in registers
struct Run {
    int k;                  // LDS offset of the bin
    uint32_t cn;            // count * kCountOne
    unsigned long long q;   // sum of q (at most kRunMax + 64 of them, below 2^61)
};

// What the pair kernel does with a pair: histogram updates.
template <bool RSD, bool W, bool BUF>
struct HistSink {
    static constexpr int kB = W ? 8 : 4;        // bytes of a histogram word
    const PairArgs& a;
    unsigned char* hist;        // this wave's histogram
    int lane, nm, nbt, nbm, planes, nent, hi_off, rep_off;
    bool batched;
    int cur_r;
    int sd, sr;                 // fixed-point scales of data and random weights (batched: the region's)
    // the work-group's copy of the outputs: [2][nbt] counts and [2][nbt][2] sums of the current region
    size_t copy;
    unsigned long long *out_cnt, *out_w;
    unsigned int n_over = 0;
    // increments this wave may have issued since it last looked at its histogram
    unsigned long long bound = 0, look_at;
    // the lane's apexes: scaled weight, LDS offset of the pair's class with a data neighbour (with the
    // lane's replica), whether it may be an apex of the reference; and its run of increments
    double w[2];
    int cb[2];
    bool ca[2];
    Run run[2];
    // the lane's entry: scaled weight, class offset (BUF: times 2, plus the buffer flag)
    double ew = 0.0;
    int ec = 0;

    // adds word k of the histogram to the outputs and clears it
    __device__ __forceinline__ void drain_word(int k)
    {
        // with buffer points and a single plane every entry is one direction of a pair: plane 1
        const int o = k % opaque(planes * nbt) + (BUF && planes == 1 ? nbt : 0);
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
    }
    __device__ __forceinline__ void drain(int t0, int stride)
    {
        for (int k = t0; k < nent; k += stride) drain_word(k);
    }
    __device__ __forceinline__ void write_out(const Run& r)
    {
        atomicAdd((unsigned long long*)(hist + r.k), r.q & 0xffffffffull);
        atomicAdd((unsigned long long*)(hist + r.k + hi_off), ((unsigned long long)r.cn << 32) | (r.q >> 32));
    }
    __device__ __forceinline__ void flush(Run& r)
    {
        write_out(r);
        r.q = 0;
        r.cn = 0;
    }
    __device__ __forceinline__ void flush_runs()
    {
        if constexpr (W) {
            flush(run[0]);
            flush(run[1]);
        }
    }
    // one increment of the bin at LDS offset k: merged with the lane's run of that bin (a lane's
    // consecutive neighbours often share a bin), which is written out when the bin changes.  An empty
    // run adds zeros.
    __device__ __forceinline__ void put(Run& r, int k, unsigned long long q)
    {
        if (k != r.k) {
            write_out(r);
            // cleared in place: written as assignments, the merge of the two paths copies every register
            asm volatile("v_mov_b64 %0, 0\n\tv_mov_b32 %1, 0\n\tv_mov_b32 %2, %3" : "+v"(r.q), "+v"(r.cn), "+v"(r.k) : "v"(k));
        }
        r.q += q;
        r.cn += kCountOne;
    }

    __device__ __forceinline__ void region(int rg)
    {
        flush_runs();
        if (cur_r >= 0) drain(opaque(lane), kWave);
        cur_r = rg;
        sd = a.regions[rg].fx_shift;
        sr = a.regions[rg].fx_shift_rand;
        out_cnt = a.out_cnt + copy + (size_t)rg * 2 * nbt;
        out_w = a.out_w + copy + (size_t)rg * 4 * nbt;
        bound = 0;
    }
    __device__ __forceinline__ void apex(int which, const double4& P, uint32_t f)
    {
        w[which] = W ? ldexp(P.w, (f & 1u) ? sr : sd) : 0.0;
        cb[which] = rep_off + ((f & 1u) ? nbm * kB : 0);
        ca[which] = !(f & 2u);
    }
    __device__ __forceinline__ void entry(const double4& P, uint32_t f)
    {
        if constexpr (W) ew = ldexp(P.w, (f & 1u) ? sr : sd);
        const int c = (f & 1u) ? nbm * kB : 0;
        ec = BUF ? (c << 1) | (int)((f >> 1) & 1u) : c;
    }
    __device__ __forceinline__ void entry_of_apex()
    {
        ew = w[0];
        const int c = cb[0] - rep_off;
        ec = BUF ? (c << 1) | (ca[0] ? 0 : 1) : c;
    }
    __device__ __forceinline__ bool nothing(int which) const { return !ca[which] && (ec & 1); }
    __device__ __forceinline__ void overflow(int which) { n_over += (unsigned)ca[which] + (BUF ? 1u - (unsigned)(ec & 1) : 1u); }
    __device__ __forceinline__ void add_at(int which, int k, unsigned long long q)
    {
        if constexpr (W) put(run[which], k, q);
        else atomicAdd((uint32_t*)(hist + k), 1u);
    }
    __device__ __forceinline__ void add(int which, int b, int m)
    {
        const int k0 = cb[which] + (BUF ? ec >> 1 : ec) + (int)__umul24(b, (unsigned)(nm * kB));
        unsigned long long q = 0;
        if constexpr (W) q = quantise_rn(w[which] * ew);
        if constexpr (!BUF) {
            add_at(which, k0 + m * kB, q);
        } else {
            // both ends apexes: plane 0; one: plane 1 in its direction
            const bool ci = ca[which], cj = !(ec & 1);
            const int mr = nm - 1 - m;
            if (planes == 2) {
                add_at(which, k0 + (ci ? m : mr) * kB + (ci && cj ? 0 : nbt * kB), q);
            } else {            // histograms too large for two planes: plane 1 only, each direction added
                if (ci) add_at(which, k0 + m * kB, q);
                if (cj) add_at(which, k0 + mr * kB, q);
            }
        }
    }
    __device__ __forceinline__ void exact_overflow(int i, int j)
    {
        n_over += (a.flags[i] & 2u ? 0u : 1u) + (a.flags[j] & 2u ? 0u : 1u);
    }
    __device__ __forceinline__ void exact(int i, int j, int b, int m, int mr)
    {
        const uint32_t fi = a.flags[i], fj = a.flags[j];
        const bool ci = !(fi & 2u), cj = !(fj & 2u);
        unsigned long long q = 0;
        if constexpr (W) q = quantise_rn(ldexp(a.pw[i].w, (fi & 1u) ? sr : sd) * ldexp(a.pw[j].w, (fj & 1u) ? sr : sd));
        const int k0 = (int)((fi & 1u) + (fj & 1u)) * nbm + b * nm;
        auto add_lds = [&](int k) {
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
            add_lds(k0 + m);
        } else if (BUF && planes == 2 && ci != cj) {
            add_lds(k0 + (ci ? m : mr) + nbt);
        } else {        // exactly on a mu edge (or one plane): the ordered pairs one by one
            if (ci) add_global(k0 + m);
            if (cj) add_global(k0 + mr);
        }
    }
    __device__ __forceinline__ void rotate()
    {
        if constexpr (W) ew = rot_lane(ew);
        ec = rot_lane(ec);
    }
    __device__ __forceinline__ void tile(int pairs, const int*, int, int, int)
    {
        bound += (unsigned long long)pairs * (BUF && planes == 1 ? 2u : 1u);
        if constexpr (W) {
            if (run[0].cn >= kRunMax * kCountOne) flush(run[0]);
            if (run[1].cn >= kRunMax * kCountOne) flush(run[1]);
        }
        if (bound > look_at) {
            flush_runs();
            if constexpr (W) {
                for (int k = opaque(lane); k < nent; k += kWave)
                    if ((((unsigned long long*)(hist + hi_off))[k] >> 42) >= (1u << 20)) drain_word(k);
            } else {
                drain(opaque(lane), kWave);
            }
            bound = 0;
        }
    }
    __device__ __forceinline__ void piece(int, int) {}
};

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
    // LDS: bin table, histogram (one, or one per wave in batched mode), the waves' lists
    extern __shared__ __align__(16) unsigned char smem[];
    const BinDesc& B = *a.bins;
    const int nb = B.nb, nm = RSD ? B.nm : 1;
    const bool batched = a.nreg > 0;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int nthr = blockDim.x;        // a multiple of 64, at most 1024
    const int nwv = nthr / kWave;

    HistSink<RSD, W, BUF> sink{a};
    sink.lane = lane;
    sink.nm = nm;
    sink.nbm = nb * nm;
    sink.nbt = 3 * nb * nm;
    sink.planes = BUF ? a.planes : 1;
    sink.nent = sink.planes * sink.nbt * a.reps;                // words of one plane of the histogram
    sink.hi_off = sink.nent * 8;
    sink.rep_off = (lane & (a.reps - 1)) * sink.planes * sink.nbt * sink.kB;
    sink.batched = batched;
    sink.cur_r = batched ? -1 : 0;
    sink.sd = B.fx_sd;
    sink.sr = B.fx_sr;
    sink.copy = (size_t)(blockIdx.x & (unsigned)(a.copies - 1)) * (size_t)a.copy_stride;
    sink.out_cnt = a.out_cnt + sink.copy;
    sink.out_w = a.out_w + sink.copy;
    sink.look_at = (W ? (1ull << 20) : (1ull << 31)) / (unsigned long long)(batched ? 1 : nwv);
    sink.run[0] = sink.run[1] = Run{sink.rep_off, 0u, 0ull};
    const int hsize = (int)((sink.nent * (W ? 16 : 4) + 15) / 16 * 16);
    sink.hist = smem + kOkBytes + (batched ? wv * hsize : 0);
    unsigned char* const lists = smem + kOkBytes + (size_t)hsize * (batched ? nwv : 1) + wv * kListBytes;
    {
        uint32_t* h0 = (uint32_t*)(smem + kOkBytes);
        const int nw = hsize / 4 * (batched ? nwv : 1);
        for (int k = tid; k < nw; k += nthr) h0[k] = 0;
        fill_bin_table<FP64>(smem, B, tid, nthr);
    }
    __syncthreads();

    WalkStats st;
    walk<FP64, RSD, LOGB, BUF>(a, sink, B, smem, lists, lane, wv, nwv, st);

    sink.flush_runs();
    if (batched) {
        if (sink.cur_r >= 0) sink.drain(opaque(lane), kWave);
    } else {
        __syncthreads();
        sink.drain(tid, nthr);
    }

    // statistics (candidates and rechecks are counted per wave, overflow pairs per lane), one atomic per
    // work-group each
    unsigned long long ov = sink.n_over;
    for (int off = 32; off > 0; off >>= 1) ov += __shfl_down(ov, off, 64);
    __shared__ unsigned long long s_stat[3];
    if (tid < 3) s_stat[tid] = 0;
    __syncthreads();
    if (lane == 0) {
        if (st.cand) atomicAdd(&s_stat[0], st.cand);
        if (st.rechk) atomicAdd(&s_stat[1], st.rechk);
        if (ov) atomicAdd(&s_stat[2], ov);
    }
    __syncthreads();
    if (tid < 3 && s_stat[tid]) atomicAdd(&a.out_stats[sink.copy + tid], s_stat[tid]);
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

}  // namespace gs
