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
//   4M points, 1.90e11 binned pairs, (r, mu), weighted:  FP32 252 -> 158 ms
//   800k points, same bins, FP64 geometry:               142 -> 47 ms
//   60k points, 10 linear bins, unweighted:              0.51 -> 0.08 ms
//   9k points, (r, mu), weighted:                        0.38 -> 0.04 ms
//   16 regions of 60k points, (r, mu), buffers:          19 -> 13 ms
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
#include "gs_pair_kernel.h"

namespace gs {

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

hipError_t launch_pair2(const PairArgs& a, const PairVariant& v, int nblocks, int wg, hipStream_t st)
{
    const size_t lds = pair2_lds_bytes(v.nb, v.nm, v.buf ? a.planes : 1, a.reps, v.weighted, a.nreg > 0, wg);
    if (!v.weighted) return launch_pair2_unit(a, v, lds, nblocks, wg, st);
    return with_variant<true>(v, [&](auto k) { return k.launch(a, lds, nblocks, wg, st); });
}

int pair2_occupancy(const PairVariant& v, int planes, int reps, bool batched, int wg)
{
    const size_t lds = pair2_lds_bytes(v.nb, v.nm, planes, reps, v.weighted, batched, wg);
    if (lds > kPairLdsMax) return 0;
    if (!v.weighted) return pair2_unit_occupancy(v, lds, wg);
    return with_variant<true>(v, [&](auto k) { return k.occupancy(lds, wg); });
}

}  // namespace gs
