// gs_pair_kernel.h -- device code of the 2PCF pair kernel (pair2.hip describes it), compiled for given weights in
// pair2.hip and for unit weights in pair2_unit.hip.
#pragma once

#include "gs_pair_tiles.h"

namespace gs {

namespace {

using namespace dev;

constexpr uint32_t kCountOne = 1u << 10;        // one count in the high word of the hi plane (bit 42)
constexpr unsigned kRunMax = 256;               // increments after which a run ends with its tile

// a lane's run of histogram increments to one bin, merged in registers.  LDS atomics are the kernel's second bound:
// two of them for every pair, and no runs, took a weighted (r, mu) survey from 168 to 270 ms.
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

// f(Pair2<...>{}) for the variant v with W weights
template <bool W, bool... Done, class F>
static auto with_variant(const PairVariant& v, F&& f)
{
    if constexpr (sizeof...(Done) == 5) {
        return f(Pair2<Done...>{});
    } else if constexpr (sizeof...(Done) == 2) {
        return with_variant<W, Done..., W>(v, f);
    } else {
        constexpr int k = sizeof...(Done);
        const bool b = k == 0 ? v.fp64 : k == 1 ? v.nm >= 2 : k == 3 ? v.logb : v.buf;
        return b ? with_variant<W, Done..., true>(v, f) : with_variant<W, Done..., false>(v, f);
    }
}

}  // namespace gs
