// gs_device.h -- device helpers shared by the counting kernels: the
// reference's FP64 pair arithmetic, exact binning against the thresholds,
// fixed-point splitting and small synchronisation/accumulation utilities.
#pragma once

#include "gs_common.h"

namespace gs {
namespace dev {

__device__ __forceinline__ void glb_add128(unsigned long long* slot, unsigned long long lo, unsigned long long hi)
{
    unsigned long long old = atomicAdd(slot, lo);
    if (old + lo < old) hi += 1ull;
    if (hi) atomicAdd(slot + 1, hi);
}

// (lo, hi) += (l, h) as 128-bit numbers
__device__ __forceinline__ void add128(unsigned long long& lo, unsigned long long& hi, unsigned long long l,
                                       unsigned long long h)
{
    lo += l;
    hi += h + (lo < l ? 1ull : 0ull);
}

// s = (bx-ax)^2 + (by-ay)^2 + (bz-az)^2 in FP64, evaluated left to right with
// no contraction, as the reference forms it (kdtree2.F90:1689, gramsci.F90:1532).
__device__ __forceinline__ double exact_s(double ax, double ay, double az, double bx, double by, double bz)
{
    double dx = __dsub_rn(bx, ax), dy = __dsub_rn(by, ay), dz = __dsub_rn(bz, az);
    return __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
}

// 0-based bin of a kept s: #{k in 1..nb : s >= t[k]}; nb means the reference's
// out-of-range bin nbins+1.
__device__ __forceinline__ int exact_bin(double s, const double* t, int nb)
{
    int lo = 0, hi = nb;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (t[mid] <= s) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// exact 0-based bin, -1 if not kept, nb on overflow
__device__ __forceinline__ int bin_of(double s, const double* t, int nb)
{
    if (!(s > t[0] && s < t[nb + 1])) return -1;
    return exact_bin(s, t, nb);
}

// exact bin of a kept s, starting from the FP32 estimate u and correcting it
// against the FP64 thresholds (0 or 1 steps in practice)
__device__ __forceinline__ int adjust_bin(double s, float u, const double* t, int nb)
{
    int b = (int)u;
    b = b < 0 ? 0 : (b > nb - 1 ? nb - 1 : b);
    while (b > 0 && s < t[b]) --b;
    while (b < nb && s >= t[b + 1]) ++b;
    return b;
}

// mu bin from t = (theta+1)*mu_scale (gramsci.F90:326-328), 0-based.  The
// reference stores floor(t)+1 in an int8 before clamping; that wrap is kept.
__device__ __forceinline__ int mu_from_t(double t, int nm)
{
    int v = (int)floor(t) + 1;
    v = (int)(int8_t)v;
    v = v < 1 ? 1 : (v > nm ? nm : v);
    return v - 1;
}

// mu bins of apex a -> neighbour b and of b -> a (gramsci.F90:320-325),
// in the reference's operation order with IEEE sqrt and division.
__device__ __forceinline__ void exact_mu(double ax, double ay, double az, double bx, double by, double bz, double ms,
                                         int nm, int& m, int& mr)
{
    double m1 = __dmul_rn(0.5, __dadd_rn(ax, bx));
    double m2 = __dmul_rn(0.5, __dadd_rn(ay, by));
    double m3 = __dmul_rn(0.5, __dadd_rn(az, bz));
    double w1 = __dsub_rn(ax, bx), w2 = __dsub_rn(ay, by), w3 = __dsub_rn(az, bz);
    double th = __dadd_rn(__dadd_rn(__dmul_rn(m1, w1), __dmul_rn(m2, w2)), __dmul_rn(m3, w3));
    double mm = __dadd_rn(__dadd_rn(__dmul_rn(m1, m1), __dmul_rn(m2, m2)), __dmul_rn(m3, m3));
    double ww = __dadd_rn(__dadd_rn(__dmul_rn(w1, w1), __dmul_rn(w2, w2)), __dmul_rn(w3, w3));
    double den = __dmul_rn(__dsqrt_rn(mm), __dsqrt_rn(ww));
    th = __ddiv_rn(th, den);
    m = mu_from_t(__dmul_rn(__dadd_rn(th, 1.0), ms), nm);
    mr = mu_from_t(__dmul_rn(__dadd_rn(-th, 1.0), ms), nm);
}

// FP32 estimate of the radial bin coordinate of s (exactness comes from the
// thresholds, not from this estimate)
__device__ __forceinline__ float bin_estimate(float s, bool logb, float ua, float ub)
{
    return logb ? fmaf(__builtin_amdgcn_logf(s), ua, ub) : fmaf(__builtin_amdgcn_sqrtf(s), ua, ub);
}

// floor(x) split at bit 32 for 0 <= x < 2^61: q = hi * 2^32 + lo.
__device__ __forceinline__ void quantise(double x, uint32_t& lo, uint32_t& hi)
{
    const double h = floor(x * 0x1p-32);
    hi = (uint32_t)h;
    lo = (uint32_t)fma(-h, 0x1p32, x);
}

// rint(x) (round to nearest even) as a 64-bit integer, for 0 <= x < 2^52: x + 2^52
// lies in [2^52, 2^53], where the spacing of doubles is 1, so the addition rounds x to an
// integer and the bit pattern of the sum is that of 2^52 plus it (also at 2^53)
__device__ __forceinline__ unsigned long long quantise_rn(double x)
{
    return (unsigned long long)(__double_as_longlong(x + 0x1p52) - 0x4330000000000000ll);
}

// Rotation of a register across the 64 lanes of a wavefront by one lane (DPP
// wave_rol:1); every lane must be active.
// The register itself is passed as the unused "old" operand (a full rotation
// writes every lane), so the move can be done in place: one v_mov_b32_dpp per
// 32-bit register and step, with no zeroed temporary and no copy back.
__device__ __forceinline__ int rot_lane(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x134, 0xf, 0xf, false); }
__device__ __forceinline__ float rot_lane(float v) { return __int_as_float(rot_lane(__float_as_int(v))); }
__device__ __forceinline__ long long rot_lane(long long b)
{
    const int lo = rot_lane((int)(b & 0xffffffffll)), hi = rot_lane((int)(b >> 32));
    return ((long long)hi << 32) | (long long)(uint32_t)lo;
}
__device__ __forceinline__ double rot_lane(double v) { return __longlong_as_double(rot_lane(__double_as_longlong(v))); }

// rint(x) as a signed 64-bit integer, for |x| < 2^51: x + 1.5 * 2^52 lies in
// [2^52, 2^53), where the spacing of doubles is 1, so the addition rounds x to an
// integer and the bit pattern of the sum is that of 1.5 * 2^52 plus it
__device__ __forceinline__ long long quantise_rn_signed(double x)
{
    return __double_as_longlong(x + 0x1.8p52) - 0x4338000000000000ll;
}

// largest r with off[r] <= v over off[0..n-1] (off non-decreasing)
__device__ __forceinline__ int upper_index(const int32_t* off, int n, int v)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= v) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Next work item from 8 queues, one per XCD segment of [0, n): own segment
// first, then the others.  `tried` is per-caller state.  Returns -1 at the end.
__device__ __forceinline__ int next_item(int32_t* queue, int n, int xcd, int& tried)
{
    while (tried < 8) {
        const int sidx = (xcd + tried) & 7;
        const int lo = (int)(((long long)n * sidx) >> 3);
        const int hi = (int)(((long long)n * (sidx + 1)) >> 3);
        const int k = atomicAdd(&queue[sidx], 1);
        if (lo + k < hi) return lo + k;
        ++tried;
    }
    return -1;
}

// v, the same in all lanes, in scalar registers
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float scalar(float v) { return __int_as_float(scalar(__float_as_int(v))); }
__device__ __forceinline__ double scalar(double v)
{
    const long long b = __double_as_longlong(v);
    return __longlong_as_double((long long)(unsigned)scalar((int)b) | ((long long)scalar((int)(b >> 32)) << 32));
}

// v, in a way the compiler cannot see through: keeps what is computed from it inside a rarely run block
// instead of in registers over the loop around it
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Work items [0, n) in 64 segments, 8 per XCD, each with a counter on a cache line of its own (device-wide
// atomics on one line run one after another, about 40 ns each: measured).  A wave's first item is its own
// slot of its home segment, taken without an atomic; later ones come from the segment's counter, and when
// that is used up from the next segment that has items left, found with one load of all counters.
struct ItemQueue {
    int32_t* counters;      // [64], kQueuePad apart, zero before the launch
    int n;                  // items
    int nwv;                // waves per work-group
    int seg;                // the segment this wave takes items from
    bool first;

    __device__ __forceinline__ ItemQueue(int32_t* c, int items, int waves)
        : counters(c), n(items), nwv(waves), seg((int)(((blockIdx.x & 7) << 3) | ((blockIdx.x >> 3) & 7))), first(true)
    {
    }
    __device__ __forceinline__ int lo(int s) const { return (int)(((long long)n * s) >> 6); }
    // waves whose home is segment s: those of the work-groups b with b mod 64 = f
    __device__ __forceinline__ int slots(int s) const
    {
        const int f = (s >> 3) | ((s & 7) << 3), g = (int)gridDim.x;
        return f < g ? (((g - 1 - f) >> 6) + 1) * nwv : 0;
    }
    // the next item of wave wv (uniform), -1 at the end; called by the whole wave
    __device__ __forceinline__ int next(int lane, int wv)
    {
        if (first) {
            first = false;
            const int k = lo(seg) + (int)(blockIdx.x >> 6) * nwv + wv;
            if (k < lo(seg + 1)) return k;
        }
        while (true) {
            if (lo(seg + 1) - lo(seg) > slots(seg)) {
                int k = 0;
                if (lane == 0) k = atomicAdd(&counters[seg * kQueuePad], 1);
                k = lo(seg) + slots(seg) + __builtin_amdgcn_readfirstlane(k);
                if (k < lo(seg + 1)) return k;
            }
            const int s = opaque(lane);
            const int used = __hip_atomic_load(&counters[s * kQueuePad], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long m = __ballot(used < lo(s + 1) - lo(s) - slots(s));
            if (!m) return -1;
            // the first such segment after this one, cyclically: the own XCD's come first
            const int sh = (seg + 1) & 63;
            const unsigned long long rot = sh ? (m >> sh) | (m << (64 - sh)) : m;
            seg = (sh + (int)__builtin_ctzll(rot)) & 63;
        }
    }
};

// true in every thread of the last block to call it; resets the counter.  What the blocks wrote before is visible
// to it through load_agent.  Only thread 0 releases, for the whole block (the barrier orders the others' writes
// before): the release writes the XCD's L2 back, which cost four waves of 500 blocks 60 us.
__device__ __forceinline__ bool last_block(unsigned* ticket)
{
    __shared__ bool s_last;
    __syncthreads();
    if (threadIdx.x == 0) {
        s_last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
        if (s_last) *ticket = 0;
    }
    __syncthreads();
    return s_last;
}

template <class T>
__device__ __forceinline__ T load_agent(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace dev
}  // namespace gs
