// gs_pair_tiles.h -- device code shared by the kernels that walk the half stencil in tiles (pair2.hip,
// adjoint.hip): apexes relative to a chunk's reference point, the candidates of a chunk's stencil rows,
// and the certain (r, mu) bin of a pair.  pair2.hip describes the decomposition.
#pragma once

#include <type_traits>

#include "gs_device.h"
#include "gs_kernels.h"

namespace gs {
namespace dev {

constexpr int kOkBytes = (kMaxBins + 1) * 8;    // bin table at the start of the LDS (fill_bin_table)
// Pairs waiting to be re-evaluated, per wave: a wave less a few, plus one wave (a wave would fit but for the largest
// histograms, which leave 1.2 KB)
constexpr int kQueue = 2 * kWave - 8;
constexpr int kListBytes = kQueue * 8 + kWave * 4;      // per wave: the queue, tile index list

__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsq(double x) { return __builtin_amdgcn_rsq(x); }
__device__ __forceinline__ float fract(float x) { return __builtin_amdgcn_fractf(x); }
__device__ __forceinline__ double fract(double x) { return __builtin_amdgcn_fract(x); }

// v truncated to an unsigned integer, 0 for a negative v or NaN, 2^32 - 1 for one beyond it (the conversion saturates)
__device__ __forceinline__ unsigned cvt_sat(float v)
{
    unsigned r;
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
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
// mask of the lanes where p holds
__device__ __forceinline__ unsigned long long lanes(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// bits of the mask below this lane
__device__ __forceinline__ int below(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// x of missing apexes (entries: negative), farther from every point than any rmax: FP32 geometry runs up to 1e8, FP64
// as long as rmax^2 is finite (an infinite squared distance is rejected like any other)
template <class R> constexpr R far_away() { return std::is_same<R, double>::value ? (R)INFINITY : (R)1e18f; }

// A point in the kernel's geometry: FP32 relative to the chunk's reference point p, FP64 absolute.
template <class R>
struct Pt {
    R x, y, z;
    R d;            // 2 (|x|^2 - |p|^2)
    R c;            // 2 (|x|^2 + |p|^2)
};

// The chunk's reference point (one of its points).
struct Ref {
    double x, y, z, p2;
    __device__ __forceinline__ void set(const double4& P, int l)
    {
        x = lane_double(P.x, l); y = lane_double(P.y, l); z = lane_double(P.z, l);
        p2 = x * x + y * y + z * z;
    }
    __device__ __forceinline__ double d_of(const double4& P) const
    {
        return 2.0 * ((P.x - x) * (P.x + x) + (P.y - y) * (P.y + y) + (P.z - z) * (P.z + z));
    }
    template <class R>
    __device__ __forceinline__ Pt<R> point(const double4& P) const
    {
        Pt<R> q;
        if constexpr (std::is_same<R, double>::value) { q.x = P.x; q.y = P.y; q.z = P.z; }
        else { q.x = (float)(P.x - x); q.y = (float)(P.y - y); q.z = (float)(P.z - z); }
        const double d = d_of(P);
        q.d = (R)d;
        q.c = (R)(d + 4.0 * p2);
        return q;
    }
};

// The point ranges of 64 stencil rows, one per lane, their points numbered by a prefix sum.
struct RowTable {
    int js, len, excl, incl, total;
    // rows r0 .. r0 + 63 for a chunk with x cells cx_first .. cx_last in x-row (cy, cz); the own row's points
    // start at `after`
    __device__ __forceinline__ void load(const Row* rows, int nrows, int r0, int lane, const int32_t* cell_start, int cb,
                                         int nx, int ny, int nz, int cy, int cz, int cx_first, int cx_last, int after)
    {
        js = 0;
        len = 0;
        lane = opaque(lane);
        if (r0 + lane < nrows) {
            const Row rw = rows[r0 + lane];
            const int by = cy + rw.dy, bz = cz + rw.dz;
            const int bx0 = max(cx_first + rw.x0, 0), bx1 = min(cx_last + rw.x1, nx - 1);
            if (by >= 0 && by < ny && bz >= 0 && bz < nz && bx0 <= bx1) {
                const int rb = cb + (bz * ny + by) * nx;
                js = cell_start[rb + bx0];
                const int je = cell_start[rb + bx1 + 1];
                if (rw.dy == 0 && rw.dz == 0) js = max(js, after);
                len = max(je - js, 0);
            }
        }
        incl = len;
        for (int off = 1; off < kWave; off <<= 1) {
            const int y = __shfl_up(incl, off, kWave);
            if (lane >= off) incl += y;
        }
        excl = incl - len;
        total = lane_int(incl, kWave - 1);
    }
    // the point of candidate c0 + lane (called by the whole wave), `none` beyond the last
    __device__ __forceinline__ int point(int c0, int lane, int none) const
    {
        const int my = c0 + lane;
        int j = none;
        unsigned long long m = lanes(incl > c0 && excl < c0 + kWave && len > 0);
        while (m) {             // the rows this tile runs across, in order
            const int r = (int)__builtin_ctzll(m);
            m &= m - 1;
            const int e0 = lane_int(excl, r), j0 = lane_int(js, r);
            if (my >= e0) j = j0 + (my - e0);
        }
        return my < total ? j : none;
    }
};

// LDS bin table: certain intervals (FP32; entry nb, an estimate just past the last bin, is never certain) or
// exact thresholds (FP64)
template <bool FP64>
__device__ __forceinline__ void fill_bin_table(unsigned char* smem, const BinDesc& B, int tid, int nthr)
{
    for (int k = tid; k <= B.nb; k += nthr) {
        if constexpr (FP64) ((double*)smem)[k] = B.t64[k];
        else {
            // start and width; a width of 0 is never certain.  s - lo rounds monotonically, so s >= hi gives a
            // rounded difference of at least the rounded width
            const bool some = k < B.nb && B.ok_hi[k] > B.ok_lo[k];
            ((float2*)smem)[k] = some ? make_float2(B.ok_lo[k], B.ok_hi[k] - B.ok_lo[k]) : make_float2(INFINITY, 0.0f);
        }
    }
}

enum PairKind { kPairNone = 0, kPairBinned, kPairOverflow, kPairUncertain };

// The bin of a pair where it is certain.
template <bool FP64, bool RSD, bool LOGB>
struct Binner {
    using R = std::conditional_t<FP64, double, float>;
    const unsigned char* table;     // fill_bin_table
    int nb;
    float ua, ub;
    R rej_lo, rej_hi, ms, hms;
    uint32_t rej_w;                 // FP32: not rejected if 0 <= s - rej_lo < this (a float's bits)
    R l0, l1, l2;                   // mu: certain where |fract(t) - 1/2| <= l0 + l1 q + l2 q^2 (1/2 - error bound)

    __device__ __forceinline__ Binner(const BinDesc& B, const unsigned char* t)
        : table(t), nb(B.nb), ua(B.ua), ub(B.ub), rej_lo(FP64 ? (R)B.t64[0] : (R)B.rej_lo),
          rej_hi(FP64 ? (R)B.t64[B.nb + 1] : (R)B.rej_hi), ms((R)B.mu_scale), hms((R)(0.5 * B.mu_scale)), l0(0), l1(0),
          l2(0)
    {
        // one unit above the rounded width, so that no s below rej_hi is rejected
        rej_w = FP64 ? 0u : __float_as_uint(B.rej_hi - B.rej_lo) + 1u;
        // in a vector register: an FMA reads one scalar operand at most
        asm volatile("" : "+v"(ub));
    }
    // the error bound for a chunk whose reference point has squared radius p2 (see fill_pair_bins)
    __device__ __forceinline__ void chunk(const BinDesc& B, double p2)
    {
        if constexpr (RSD) {
            const R rho = (R)sqrt(p2) * (R)1.001, ab = (R)B.mu_ab;
            const R sx = (R)2.0 * rho + ab;
            l0 = (R)0.5 - (R)B.mu_k0;
            l1 = -((R)B.mu_k1a * sx + (R)B.mu_k1b * ((R)2.0 * rho + (R)3.0 * ab));
            l2 = -((R)B.mu_k2a + (R)B.mu_k2b * sx * sx);
        }
    }
    __device__ __forceinline__ R separation2(const Pt<R>& A, R ex, R ey, R ez) const
    {
        if constexpr (FP64) {
            return exact_s(A.x, A.y, A.z, ex, ey, ez);
        } else {
            const float dx = ex - A.x, dy = ey - A.y, dz = ez - A.z;
            return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        }
    }
    __device__ __forceinline__ bool rejected(R s) const
    {
        // FP32: one comparison of the difference's bits, in which negative numbers are above all others
        if constexpr (FP64) return !(s > rej_lo && s < rej_hi);
        else return !(__float_as_uint(s - rej_lo) < rej_w);
    }
    // bins of a pair that is not rejected
    __device__ __forceinline__ PairKind bins(const Pt<R>& A, R ed, R s, int& b, int& m) const
    {
        bool safe = true;
        if constexpr (FP64) {
            // as unsigned: s may be beyond a float's range, and its estimate 2^32 - 1
            b = (int)min(cvt_sat(bin_estimate((float)s, LOGB, ua, ub)), (unsigned)(nb - 1));
            const double* t = (const double*)table;
            if (!(s >= t[b] && s < t[b + 1])) {
                while (b > 0 && s < t[b]) --b;
                while (b < nb && s >= t[b + 1]) ++b;
                if (b == nb) return kPairOverflow;
            }
        } else {
            b = (int)cvt_sat(bin_estimate(s, LOGB, ua, ub));
            const float2 ok = ((const float2*)table)[b];
            safe = __float_as_uint(s - ok.x) < __float_as_uint(ok.y);
        }
        m = 0;
        if constexpr (RSD) {
            const R S = (A.c + ed) - s;
            const R q = rsq(S * s);
            const R t = fma((A.d - ed) * q, hms, ms);
            const R lim = fma(fma(l2, q, l1), q, l0);
            // written so that a NaN (mid-point at the origin) is uncertain
            safe = safe && fabs(fract(t) - (R)0.5) <= lim;
            m = (int)t;
        }
        return safe ? kPairBinned : kPairUncertain;
    }
};

// Walks the items of a wave: every unordered pair of the item's chunk with itself and with the candidates of
// its half stencil (see pair2.hip).  The sink holds what its kernel does with a pair:
//   region(r)                   batch: the wave goes on with region r
//   apex(which, P, f, v)        point P with flags f becomes the lane's apex `which` (0, 1); v: there is one
//   entry(P, f, has)            the lane's tile entry, or none
//   entry_of_apex(v)            the lane's first apex as tile entry (pairs inside the chunk)
//   nothing(which)              the apex and the lane's entry are two buffer points
//   add(which, b, m)            the pair of an apex with the lane's entry, in radial bin b, mu bin m
//   overflow(which)             ... beyond the last bin
//   exact(i, j, b, m, mr), exact_overflow(i, j)     a re-evaluated pair of points
//   rotate()                    the lane's entry comes from the next lane
//   tile(pairs, jlist, r, ib, n_i)  a tile is done: at most `pairs` pairs, entry (lane + r) & 63 in this lane
//   piece(ib, n_i)              the chunk's points ib .. ib + n_i - 1 are done
// Pairs that are not certain wait in LDS and are re-evaluated together when more than 64 are waiting: a
// recheck then fills a wave instead of one lane.
struct WalkStats {
    unsigned long long cand = 0, rechk = 0;
};

template <bool FP64, bool RSD, bool LOGB, bool BUF, class Sink>
__device__ __forceinline__ void walk(const WalkArgs& a, Sink& sink, const BinDesc& B, const unsigned char* table,
                                     unsigned char* lists, int lane, int wv, int nwv, WalkStats& st)
{
    using R = std::conditional_t<FP64, double, float>;
    int2* const queue = (int2*)lists;
    int* const jlist = (int*)(lists + kQueue * 8);
    Binner<FP64, RSD, LOGB> binner(B, table);
    const int nb = B.nb;
    const int group = a.group, half = group >> 1;
    const int ai = lane & (group - 1), ai2 = ai ^ half;     // the lane's apexes in the chunk
    const bool batched = a.nreg > 0;
    int nx = a.g.dim[0], ny = a.g.dim[1], nz = a.g.dim[2], cb = 0;
    int row0 = 0, row1 = batched ? 0 : ny * nz;     // x-rows of the current region

    int nq = 0;
    auto recheck = [&]() {
        wave_sync();
        for (int k = opaque(lane); k < nq; k += kWave) {
            const int2 pr = queue[k];
            int b, m = 0, mr = 0;
            {
                const double4 Pi = a.pw[pr.x], Pj = a.pw[pr.y];
                const double s = exact_s(Pi.x, Pi.y, Pi.z, Pj.x, Pj.y, Pj.z);
                if (!(s > B.t64[0] && s < B.t64[nb + 1])) continue;
                b = adjust_bin(s, bin_estimate((float)s, LOGB, B.ua, B.ub), B.t64, nb);
            }
            if (b == nb) {
                sink.exact_overflow(pr.x, pr.y);
                continue;
            }
            if constexpr (RSD) {
                const double4 Pi = a.pw[pr.x], Pj = a.pw[pr.y];
                exact_mu(Pi.x, Pi.y, Pi.z, Pj.x, Pj.y, Pj.z, B.mu_scale, B.nm, m, mr);
            }
            sink.exact(pr.x, pr.y, b, m, mr);
        }
        st.rechk += (unsigned)nq;
        nq = 0;
        wave_sync();
    };

    const int n_chunks = (int)(((long long)a.n + group - 1) / group);
    ItemQueue items(a.queue, n_chunks << a.lg_parts, nwv);
    while (true) {
        const int item = items.next(lane, wv);
        if (item < 0) break;
        const int part = item & ((1 << a.lg_parts) - 1);
        int ib = (item >> a.lg_parts) * group;
        const int iend = (int)min((long long)a.n, (long long)ib + group);

        // A chunk is taken in pieces [ib, ib + n_i) of one x-row and at most cap_cells + 1 cells in x, for which
        // the FP32 error bounds hold.
        int n_i;
        for (; ib < iend; ib += n_i) {
            int2 cl = make_int2(0, -1);
            if (ib + ai < iend) cl = a.cell[ib + ai];
            const int cx_first = lane_int(cl.x, 0), grow = lane_int(cl.y, 0);
            n_i = uniform(__popcll(lanes(lane < group && cl.y == grow && cl.x - cx_first <= a.cap_cells)));
            const int cx_last = lane_int(cl.x, n_i - 1);
            if (batched && (grow < row0 || grow >= row1)) {
                if (nq) recheck();
                const int rg = uniform(upper_index(a.row_base, a.nreg, grow));
                const RegionDesc& rd = a.regions[rg];
                nx = rd.dim[0]; ny = rd.dim[1]; nz = rd.dim[2];
                cb = rd.cell_base;
                row0 = rd.row_base;
                row1 = row0 + ny * nz;
                sink.region(rg);
            }
            const int cy = (grow - row0) % ny, cz = (grow - row0) / ny;

            // ---- the lane's apexes, relative to the chunk's middle point
            const bool v1 = ai < n_i, v2 = ai2 < n_i;
            Pt<R> A1, A2;
            Ref ref;
            bool chunk_buf;
            {
                double4 P1 = make_double4(0, 0, 0, 0), P2 = P1;
                uint32_t f1 = 2u, f2 = 2u;
                if (v1) { P1 = a.pw[ib + ai]; f1 = a.flags[ib + ai]; }
                if (v2) { P2 = a.pw[ib + ai2]; f2 = a.flags[ib + ai2]; }
                ref.set(P1, n_i >> 1);
                A1 = ref.point<R>(P1);
                A2 = ref.point<R>(P2);
                if (!v1) A1.x = far_away<R>();
                if (!v2) A2.x = far_away<R>();
                sink.apex(0, P1, f1);
                sink.apex(1, P2, f2);
                chunk_buf = BUF && lanes(!(f1 & 2u)) == 0;
            }
            binner.chunk(B, ref.p2);

            R ex = 0, ey = 0, ez = 0, ed = 0;       // the lane's tile entry
            // the pair of apex A with the lane's entry; true if it has to be re-evaluated
            auto visit = [&](const Pt<R>& A, const int which) __attribute__((always_inline)) -> bool {
                const R s = binner.separation2(A, ex, ey, ez);
                if (binner.rejected(s)) return false;
                if (BUF && sink.nothing(which)) return false;
                int b, m;
                const PairKind kind = binner.bins(A, ed, s, b, m);
                if (kind == kPairUncertain) return true;
                if (FP64 && kind == kPairOverflow) sink.overflow(which);
                else sink.add(which, b, m);
                return false;
            };
            auto enqueue = [&](const bool un, const int ia, const int k) __attribute__((always_inline)) {
                const unsigned long long um = lanes(un);
                if (un) queue[nq + below(um)] = make_int2(ia, jlist[(lane + k) & (kWave - 1)]);
                nq = uniform(nq + __popcll(um));
            };

            for (int r0 = 0; r0 < a.nrows; r0 += kWave) {
                RowTable rows;
                rows.load(a.rows, a.nrows, r0, lane, a.cell_start, cb, nx, ny, nz, cy, cz, cx_first, cx_last, ib + n_i);
                const int tiles = (rows.total + kWave - 1) / kWave;
                const int t0 = uniform((int)(((long long)tiles * part) >> a.lg_parts));
                const int t1 = uniform((int)(((long long)tiles * (part + 1)) >> a.lg_parts));
                // tile t0 - 1 of the first rows' first part: the chunk with itself, entries ai, steps
                // 1 .. half with the first apexes of one copy of the chunk (half of them in the last step)
                for (int t = r0 == 0 && part == 0 ? t0 - 1 : t0; t < t1; ++t) {
                    const bool self = uniform(t < t0 ? 1 : 0) != 0;
                    const int nt = self ? n_i : min(kWave, rows.total - t * kWave);
                    const int pairs = self ? n_i * (n_i - 1) / 2 : n_i * nt;
                    st.cand += (unsigned)pairs;
                    int j;
                    if (self) {
                        if (chunk_buf) continue;
                        j = ib + min(ai, n_i - 1);
                        ex = v1 ? A1.x : -far_away<R>(); ey = A1.y; ez = A1.z; ed = A1.d;
                        sink.entry_of_apex();
                    } else {
                        const bool has = lane < nt;
                        j = rows.point(t * kWave, lane, ib);
                        const uint32_t f = a.flags[j];
                        if (chunk_buf && lanes(has && !(f & 2u)) == 0) continue;
                        const double4 P = a.pw[j];
                        const Pt<R> E = ref.point<R>(P);
                        ex = has ? E.x : -far_away<R>(); ey = E.y; ez = E.z;
                        if constexpr (RSD) ed = E.d;
                        sink.entry(P, f);
                    }
                    wave_sync();
                    jlist[lane] = j;
                    wave_sync();
                    const int steps = uniform(self ? half + 1 : half);
                    for (int k = 0; k < steps; ++k) {
                        if (k) {
                            ex = rot_lane(ex); ey = rot_lane(ey); ez = rot_lane(ez);
                            if constexpr (RSD) ed = rot_lane(ed);
                            sink.rotate();
                        }
                        bool u1 = false, u2 = false;
                        if (!self || (k && lane < (k < half ? group : half))) u1 = visit(A1, 0);
                        if (!self) u2 = visit(A2, 1);
                        if constexpr (RSD || !FP64) {
                            if (lanes(u1 || u2)) {
                                enqueue(u1, ib + ai, k);
                                if (nq > kQueue - kWave) recheck();
                                enqueue(u2, ib + ai2, k);
                                if (nq > kQueue - kWave) recheck();
                            }
                        }
                    }
                    sink.tile(pairs, jlist, steps - 1, ib, n_i);
                }
            }
            sink.piece(ib, n_i);
        }
    }
    if (nq) recheck();
}

}  // namespace dev
}  // namespace gs
