// api.cpp -- the C ABI (include/gramsci_hip.h): contexts, catalogue upload,
// grid build, exact bin thresholds, kernel launches and the host-side
// combination of exact class sums into the reference's N2 / N3.
#include "../../include/gramsci_hip.h"

#include <algorithm>
#include <array>
#include <map>
#include <mutex>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "gs_kernels.h"
#include "gs_api_internal.h"

using namespace gs;

namespace gs {

thread_local std::string g_err;

int fail(int code, const char* fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

int hip_fail(hipError_t e, const char* what)
{
    return fail(GS_EHIP, "%s: %s", what, hipGetErrorString(e));
}

// ------------------------------------------------------------ device buffers
template <class T>
int DevBuf<T>::reserve(size_t count)
{
    if (count <= cap) return GS_OK;
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    cap = 0;
    size_t c = std::max<size_t>(count, 1);
    hipError_t e = hipMalloc((void**)&ptr, c * sizeof(T));
    if (e != hipSuccess) {
        ptr = nullptr;
        return fail(GS_ENOMEM, "hipMalloc(%zu bytes): %s", c * sizeof(T), hipGetErrorString(e));
    }
    cap = c;
    return GS_OK;
}

template <class T>
void DevBuf<T>::release()
{
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    cap = 0;
}

template struct DevBuf<double>;
template struct DevBuf<int32_t>;
template struct DevBuf<double4>;
template struct DevBuf<unsigned long long>;
template struct DevBuf<unsigned char>;
template struct DevBuf<float>;
template struct DevBuf<int2>;
template struct DevBuf<unsigned>;
template struct DevBuf<CatalogueStats>;
template struct DevBuf<IngestScratch>;

int HostBuf::reserve(size_t bytes)
{
    if (bytes <= cap) return GS_OK;
    release();
    const size_t c = std::max<size_t>(bytes, 4096);
    hipError_t e = hipHostMalloc((void**)&ptr, c, hipHostMallocDefault);
    if (e != hipSuccess) {
        ptr = nullptr;
        return fail(GS_ENOMEM, "hipHostMalloc(%zu bytes): %s", c, hipGetErrorString(e));
    }
    cap = c;
    return GS_OK;
}

void HostBuf::release()
{
    if (ptr) (void)hipHostFree(ptr);
    ptr = nullptr;
    cap = 0;
}

// ------------------------------------------------------------ thresholds
// The reference's radial bin of a squared distance s (gramsci.F90:136-145,
// :334-338), 1-based, evaluated with the host libm exactly as written.
struct RefBin {
    double inv_delta_r, log_rmin, rmin;
    bool log_bins;
    explicit RefBin(const gs_params& p) : log_rmin(0), rmin(p.rmin), log_bins(p.log_bins != 0)
    {
        double delta_r;
        if (p.log_bins) {
            delta_r = (std::log10(p.rmax) - std::log10(p.rmin)) / (double)p.nbins;
            log_rmin = std::log10(p.rmin);
        } else {
            delta_r = (p.rmax - p.rmin) / (double)p.nbins;
        }
        inv_delta_r = 1.0 / delta_r;
    }
    int operator()(double s) const
    {
        const double d = std::sqrt(s);
        if (log_bins) return (int)std::floor((std::log10(d) - log_rmin) * inv_delta_r) + 1;
        return (int)std::floor((d - rmin) * inv_delta_r) + 1;
    }
};

static inline uint64_t dbits(double x)
{
    uint64_t u;
    memcpy(&u, &x, 8);
    return u;
}
static inline double bitsd(uint64_t u)
{
    double x;
    memcpy(&x, &u, 8);
    return x;
}

// smallest non-negative double s in [lo, hi] (bit patterns) with pred(s) true; pred monotone false->true.
template <class F>
static uint64_t first_true(uint64_t lo, uint64_t hi, F pred)
{
    while (lo < hi) {
        uint64_t mid = lo + (hi - lo) / 2;
        if (pred(bitsd(mid))) hi = mid; else lo = mid + 1;
    }
    return lo;
}

int check_params(const gs_params* p, int mode)
{
    if (!p) return fail(GS_EINVAL, "params is NULL");
    if (p->nbins < 1 || p->nbins > kMaxBins) return fail(GS_EINVAL, "nbins must be in 1..127 (got %d)", p->nbins);
    if (p->nmu < 1 || p->nmu > kMaxBins) return fail(GS_EINVAL, "nmu must be in 1..127 (got %d)", p->nmu);
    if (!(p->rmin >= 0.0) || !(p->rmax > p->rmin) || !std::isfinite(p->rmax))
        return fail(GS_EINVAL, "need 0 <= rmin < rmax (got rmin=%g rmax=%g)", p->rmin, p->rmax);
    if (p->log_bins && !(p->rmin > 0.0)) return fail(GS_EINVAL, "log bins need rmin > 0");
    if (p->precision != GS_FP64 && p->precision != GS_FP32_GUARD)
        return fail(GS_EINVAL, "precision must be GS_FP64 or GS_FP32_GUARD");
    if (p->cell_div < 0 || p->cell_div > 16) return fail(GS_EINVAL, "cell_div must be in 0..16");
    if (mode >= 4 && p->nmu != 1) return fail(GS_EINVAL, "the 4PCF has no mu binning: nmu must be 1");
    return GS_OK;
}

}  // namespace gs

extern "C" int gs_bin_thresholds(const gs_params* p, double* t)
{
    int rc = check_params(p, 2);
    if (rc) return rc;
    if (!t) return fail(GS_EINVAL, "t is NULL");
    const gs_params P = *p;
    const int nb = P.nbins;
    const RefBin ref_bin(P);
    const double rmax2 = P.rmax * P.rmax;
    const uint64_t top = dbits(rmax2 * 4.0 + 1.0);
    // t[0]: largest s with sqrt(s) <= rmin
    uint64_t u = first_true(0, top, [&](double s) { return std::sqrt(s) > P.rmin; });
    t[0] = bitsd(u - (u > 0 ? 1 : 0));
    if (std::sqrt(t[0]) > P.rmin) t[0] = 0.0;
    // t[nb+1]: smallest s not kept by the r-ball (s <= rmax^2) and the strict d < rmax
    const uint64_t hi = first_true(dbits(t[0]), top, [&](double s) { return !(s <= rmax2 && std::sqrt(s) < P.rmax); });
    t[nb + 1] = bitsd(hi);
    const uint64_t lo = dbits(t[0]) + 1;
    for (int k = 1; k <= nb; ++k) {
        uint64_t v = first_true(lo, hi, [&](double s) { return ref_bin(s) >= k + 1; });
        t[k] = bitsd(v);
    }
    // the bin must be a non-decreasing step function of s near each edge, with
    // bin >= 1 just above rmin; verify in a window of ulps around every threshold
    const int win = 256;
    if (lo < hi && ref_bin(bitsd(lo)) < 1) return fail(GS_EINVAL, "bin formula gives 0 just above rmin");
    for (int k = 0; k <= nb + 1; ++k) {
        const uint64_t c = dbits(t[k]);
        int prev = -1000000;
        for (int64_t d = -win; d <= win; ++d) {
            const int64_t b = (int64_t)c + d;
            if (b <= (int64_t)lo || b >= (int64_t)hi) continue;
            const int v = ref_bin(bitsd((uint64_t)b));
            if (v < prev) return fail(GS_EINVAL, "bin formula not monotone near threshold %d", k);
            prev = v;
        }
    }
    return GS_OK;
}

namespace gs {

// ------------------------------------------------------------ FP32 guard band
// Upper bound of |s32 - s| for a pair whose cell-relative FP32 coordinates are
// bounded by rrel per component (the squared distance s near t).
static double s_guard(double t, double ew)
{
    const double root = std::sqrt(std::max(t, 0.0));
    return 2.0 * (2.0 * std::sqrt(3.0) * root * ew + 3.0 * ew * ew + std::ldexp(t, -22));
}

static float f_up(double x)
{
    float f = (float)x;
    if ((double)f < x) f = std::nextafter(f, INFINITY);
    return f;
}
static float f_down(double x)
{
    float f = (float)x;
    if ((double)f > x) f = std::nextafter(f, -INFINITY);
    return f;
}

int fill_bins(const gs_params& p, const double* t64, double rrel, double xmax, double wmax_d, double wmax_r, BinDesc& B)
{
    memset(&B, 0, sizeof(B));
    const int nb = p.nbins;
    std::copy(t64, t64 + nb + 2, B.t64);
    B.nb = nb;
    B.nm = p.nmu;
    B.log_bins = p.log_bins;
    B.rsd = p.nmu >= 2;
    B.mu_scale = (double)(0.5f * (float)p.nmu);
    B.ms32 = (float)B.mu_scale;
    // error of one cell-relative coordinate difference (FP64 -> FP32 rounding of both ends + the FP32 subtract)
    const double ew = std::ldexp(2.0 * rrel + p.rmax, -24) * 1.01;
    for (int b = 0; b < nb; ++b) {
        const double lo = b == 0 ? B.t64[0] : B.t64[b];
        const double hi = b == nb - 1 ? std::min(B.t64[nb], B.t64[nb + 1]) : B.t64[b + 1];
        B.ok_lo[b] = f_up(lo + s_guard(lo, ew));
        B.ok_hi[b] = f_down(hi - s_guard(hi, ew));
    }
    B.rej_lo = f_down(B.t64[0] - s_guard(B.t64[0], ew));
    B.rej_hi = f_up(B.t64[nb + 1] + s_guard(B.t64[nb + 1], ew));
    if (p.log_bins) {
        const double delta = (std::log10(p.rmax) - std::log10(p.rmin)) / nb;
        const double inv = 1.0 / delta;
        B.ua = (float)(0.5 * std::log10(2.0) * inv);
        B.ub = (float)(-std::log10(p.rmin) * inv);
    } else {
        const double inv = 1.0 / ((p.rmax - p.rmin) / nb);
        B.ua = (float)inv;
        B.ub = (float)(-p.rmin * inv);
    }
    // mu guard: per-component errors of sep (ew) and of the absolute midpoint (em)
    const double em = std::ldexp(2.0 * xmax + 3.0 * rrel, -24) * 1.01;
    B.mu_ew = (float)(2.0 * std::sqrt(3.0) * ew * 4.0);
    B.mu_em = (float)(2.0 * std::sqrt(3.0) * em * 4.0);
    B.mu_c = (float)std::ldexp(1.0, -18);
    B.fx_sd = fx_shift_point(wmax_d);
    B.fx_sr = fx_shift_point(wmax_r);
    B.fx_shift3 = fx_shift_triples(std::max(wmax_d, wmax_r));
    return GS_OK;
}

// Tables of the triplet kernel on the matrix cores; its header derives the error bound.  ok[k].y bounds differences
// rounded to FP32: rounding is monotonic, so s >= hi implies s - lo >= hi - lo also when rounded.
void fill_triplet_matrix(const gs_params& p, const double* t64, double h, double hx, TripMatrix& M)
{
    memset(&M, 0, sizeof(M));
    const int nb = p.nbins, e = std::ilogb(p.rmax);
    M.t_top = std::min(t64[nb], t64[nb + 1]);
    M.inv_h = 1.0 / h;
    M.inv_hx = 1.0 / hx;
    M.scale = std::ldexp(1.0, -e);
    const double r = std::ldexp(p.rmax, -e), err = std::ldexp(r * r, -18) * 1.01;
    auto t = [&](int b) { return std::ldexp(t64[b], -2 * e); };
    auto interval = [](float lo, float hi) { return make_float2(lo, hi > lo ? hi - lo : 0.0f); };
    // a squared side is below 4 r^2 <= 16 but for its error and the padding (1e30)
    M.ok[0] = interval(-16.0f, f_down(t(0) - err));
    for (int b = 0; b < nb; ++b)
        M.ok[b + 1] = interval(f_up(t(b) + err), f_down((b == nb - 1 ? std::min(t(nb), t(nb + 1)) : t(b + 1)) - err));
    M.ok[nb + 1] = make_float2(f_up(t(nb + 1) + err), INFINITY);
    if (p.log_bins) {
        const double inv = 1.0 / ((std::log10(p.rmax) - std::log10(p.rmin)) / nb);
        M.ua = (float)(0.5 * std::log10(2.0) * inv);
        M.ub = (float)((std::log10(2.0) * e - std::log10(p.rmin)) * inv + 1.0);
    } else {
        const double inv = 1.0 / ((p.rmax - p.rmin) / nb);
        M.ua = (float)std::ldexp(inv, e);
        M.ub = (float)(-p.rmin * inv + 1.0);
    }
}

// fill_bins for the pair kernel.  A chunk's points lie within q.ext of its reference point per axis, so a
// pair within rmax has coordinates (relative to that point) of at most q.ext and q.ext + rmax: rounding
// both to FP32 and subtracting costs at most u (2 ext + 2 rmax) per component, u = 2^-24.
//
// mu guard.  With a = sqrt(3) ext and b = a + rmax bounding the two points' distances from the reference
// point p, rho = |p|, u the rounding unit of the kernel's geometry and g(s) the error of s:
//   D = 2(|xi|^2 - |xj|^2): both terms are rounded, |2(|x|^2 - rho^2)| <= 2 b (|x| + rho), which moves
//     theta = (D/2) q by at most u (a + b)(2 rho + 3 (a + b)) q;
//   S = |xi + xj|^2: relative error <= 5 u + (9 u b^2 + g) / S, and 1/S = s q^2 <= rmax^2 q^2;
//   s: relative error g/s <= 4 sqrt(3) ew / |sep| + 6 ew^2 / s + 2^-21, 1/|sep| = q sqrt(S) <= q Sx with
//     Sx = 2 rho + a + b;
//   the reciprocal square root (half of the relative errors of s and S, plus 2^-22 in FP32 and less than
//   2^-21 in FP64), the products and the FMA round by less than 2^-21 together.
// k0, k1 and k2 q^2 carry factors of 2, 2 and 4 over these, so that a relative error of S s near one,
// where the linearisation fails, gives a bound above 1/2 and hence a recheck.  Outside the range of
// coordinates where S s neither overflows nor loses bits to underflow every pair is rechecked.
int fill_pair_bins(const gs_params& p, const double* t64, const PairGrid& q, double xmax, double wmax_d, double wmax_r, BinDesc& B)
{
    int rc = fill_bins(p, t64, q.ext + 0.5 * p.rmax, xmax, wmax_d, wmax_r, B);
    if (rc) return rc;
    const bool fp64 = p.precision == GS_FP64;
    const double ms = B.mu_scale, r = p.rmax;
    const double u = fp64 ? std::ldexp(1.0, -52) : std::ldexp(1.0, -24);
    // FP64: the coordinates are exact, s is rounded three times
    const double ew = fp64 ? 0.0 : std::ldexp(2.0 * q.ext + 2.0 * r, -24) * 1.01;
    const double g = fp64 ? std::ldexp(r * r, -50) : s_guard(r * r, ew);
    const double a = std::sqrt(3.0) * q.ext * 1.001, b = a + r * 1.001;
    B.mu_ab = (a + b) * 1.001;
    B.mu_k0 = ms * 2.0 * std::ldexp(1.0, -20);
    B.mu_k1a = ms * 2.0 * 2.0 * std::sqrt(3.0) * ew;
    B.mu_k1b = ms * 2.0 * u * (a + b);
    B.mu_k2a = ms * 4.0 * 0.5 * (9.0 * u * b * b + g) * r * r;
    B.mu_k2b = ms * 4.0 * 3.0 * ew * ew;
    const bool in_range = fp64 ? (r > 1e-30 && xmax < 1e30 && q.ext < 1e30)
                               : (r > 1e-5 && r < 1e8 && xmax < 1e8 && q.ext < 1e8);
    if (!in_range) B.mu_k0 = 1.0;
    // The kernel's bin table has one entry past the last bin: the estimate of a pair that is not yet rejected must
    // not go beyond it.  The largest such s, the estimate with the kernel's rounded constants, and its error: the
    // square root or logarithm and the FMA, 2^-21 of each term (in a narrow range of bins the terms are large and
    // nearly cancel: 100 log bins in the last 1e-4 of rmax are estimated 0.23 too high).
    const double top = (double)B.rej_hi + std::ldexp(std::fabs((double)B.rej_hi) + std::fabs((double)B.rej_lo), -22);
    const double fs = p.log_bins ? std::log2(top) : std::sqrt(top), ua = B.ua, ub = B.ub;
    const double err = std::ldexp(std::fabs(ua) * (std::fabs(fs) + (p.log_bins ? 1.0 : 0.0)) + std::fabs(ub), -21);
    B.wide = !(ua * fs + ub + err < p.nbins + 0.9) || r > 1e8 || q.ext > 1e8;
    return GS_OK;
}

// Fixed-point scales 2^F of the weights and products.  Pairs: each weight is scaled by its
// class's 2^F, below 2^26, so the largest pair product of every class stays below 2^52 (the
// pair kernel rounds it to an integer with one FP64 addition of 2^52 and sums a run, of some
// hundreds at most, in one 64-bit register) and each class sum is exact to 2^-52 of its own largest product.
// Triples: the largest triple product stays below 2^61.
int fx_shift_point(double wmax)
{
    const double wm = std::max(wmax, 1e-300);
    return std::min(500, 26 - (int)std::ceil(std::log2(wm * (1.0 + 1e-12))));
}

int fx_shift_triples(double wmax)
{
    const double wm = std::max(wmax, 1e-300);
    return std::min(1000, 61 - (int)std::ceil(std::log2(wm * wm * wm * (1.0 + 1e-12))));
}

// Half stencil of x-rows for cells of edge h in y/z and hx in x, search radius rmax, m = ceil(rmax/h).
// Row (dy, dz) takes x-offsets dx with gap(dy)^2 h^2 + gap(dz)^2 h^2 + gap(dx)^2 hx^2 <= rmax^2 (plus a
// relative margin of 1e-6), gap(d) = max(|d| - 1, 0) being the fewest whole cells between two cells d
// apart: no pair within rmax is left out, and a fine hx cuts each row close to the sphere.
std::vector<Row> half_stencil(double h, double hx, double rmax, int m)
{
    std::vector<Row> rows;
    auto gap = [](int d) { return (double)std::max(std::abs(d) - 1, 0); };
    const double lim = rmax * (1.0 + 1e-6) + 1e-9 * h;
    const double lim2 = lim * lim;
    const int mxmax = (int)std::ceil(lim / hx) + 1;
    for (int dz = 0; dz <= m; ++dz)
        for (int dy = -m; dy <= m; ++dy) {
            if (dz == 0 && dy < 0) continue;
            const double gyz = (gap(dy) * gap(dy) + gap(dz) * gap(dz)) * h * h;
            if (gyz > lim2) continue;
            int mx = 0;
            for (int dx = 1; dx <= mxmax; ++dx)
                if (gyz + gap(dx) * gap(dx) * hx * hx <= lim2) mx = dx;
            Row r;
            r.dy = (int16_t)dy;
            r.dz = (int16_t)dz;
            r.x0 = (int16_t)((dz == 0 && dy == 0) ? 0 : -mx);
            r.x1 = (int16_t)mx;
            rows.push_back(r);
        }
    return rows;
}

// Full stencil (both half spaces) as x-rows, for apex-centred kernels.
std::vector<Row> full_stencil(double h, double hx, double rmax, int m)
{
    std::vector<Row> half = half_stencil(h, hx, rmax, m);
    std::vector<Row> rows;
    for (const Row& r : half) {
        if (r.dy == 0 && r.dz == 0) {
            Row c = r;
            c.x0 = (int16_t)(-r.x1);
            rows.push_back(c);
        } else {
            rows.push_back(r);
            Row n = r;
            n.dy = (int16_t)(-r.dy);
            n.dz = (int16_t)(-r.dz);
            rows.push_back(n);
        }
    }
    return rows;
}

// 128-bit fixed point (lo, hi) scaled by 2^-shift -> long double
long double fx_value(unsigned long long lo, unsigned long long hi, int shift)
{
    long double v = (long double)hi * 18446744073709551616.0L + (long double)lo;
    return std::ldexp(v, -shift);
}

}  // namespace gs

// ====================================================================== context

struct gs_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    int n_cu = 256;
    // catalogue (original order)
    int64_t n_data = 0, n_rand = 0;
    bool has_w = false, has_buf = false;
    long double wsum_d = 0, wsum_r = 0;
    double wmax = 1.0, wmax_d = 1.0, wmax_r = 1.0;
    double bbox[6] = {0, 0, 0, 0, 0, 0};
    DevBuf<double> xyz, w;
    DevBuf<int32_t> buf;
    // grid
    GridDesc g{};
    bool grid_valid = false;
    double grid_h = 0.0;
    int grid_sx = 1;
    DevBuf<int32_t> rank, boff, cell_start, chunk_nc, chunk_off, scan_tmp;
    DevBuf<unsigned> ticket;
    DevBuf<double4> pw;
    DevBuf<int2> cell;
    DevBuf<uint32_t> flags;
    DevBuf<int32_t> orig;
    int32_t n_chunks = 0;
    bool row_chunks_valid = false;
    // launch scratch: one region that a launch clears (work counters, output copies, cell counts), parameters
    DevBuf<unsigned char> zero, params;
    HostBuf host;               // parameters and results in flight
    // catalogue hand-over: statistics, and a ring of pinned pieces for catalogues in host memory
    DevBuf<CatalogueStats> stats;
    DevBuf<IngestScratch> ingest;
    HostBuf stats_host, ring;
    hipEvent_t ring_ev[4] = {nullptr, nullptr, nullptr, nullptr};
    // exact bin thresholds of the last parameter sets
    struct Thresholds {
        double rmin, rmax;
        int32_t nbins, log_bins;
        std::vector<double> t;
    };
    std::vector<Thresholds> thresholds;
    GsExtra extra;
    GsBatch batch;
};

using namespace gs;

static int set_device(gs_ctx* c)
{
    hipError_t e = hipSetDevice(c->device);
    return e == hipSuccess ? GS_OK : hip_fail(e, "hipSetDevice");
}

extern "C" const char* gs_last_error(void) { return gs::g_err.c_str(); }
extern "C" const char* gs_version(void) { return "gramsci_hip 0.1 (gfx950)"; }

extern "C" int gs_create(gs_ctx** out, int device)
{
    if (!out) return fail(GS_EINVAL, "ctx is NULL");
    *out = nullptr;
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev <= device || device < 0) return fail(GS_ENODEV, "no HIP device %d", device);
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, device);
    if (e != hipSuccess) return hip_fail(e, "hipGetDeviceProperties");
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(GS_ENODEV, "device %d is %s; this library is built for gfx950 only", device, prop.gcnArchName);
    gs_ctx* c = new gs_ctx();
    c->device = device;
    c->n_cu = prop.multiProcessorCount;
    if ((e = hipSetDevice(device)) != hipSuccess || (e = hipStreamCreate(&c->stream)) != hipSuccess) {
        delete c;
        return hip_fail(e, "hipStreamCreate");
    }
    for (auto& ev : c->ev)
        if ((e = hipEventCreate(&ev)) != hipSuccess) {
            delete c;
            return hip_fail(e, "hipEventCreate");
        }
    // pinned memory for the parameters and results of any 2PCF count (the histogram is bounded by the LDS), so
    // that no call has to allocate it; catalogue statistics: zero but for the address of the pinned host copy
    int rc;
    if ((rc = c->stats.reserve(1)) || (rc = c->ingest.reserve(kIngestBlocks)) || (rc = c->ticket.reserve(1)) ||
        (rc = c->stats_host.reserve(sizeof(CatalogueStats))) || (rc = c->host.reserve(1 << 20))) {
        (void)gs_destroy(c);
        return rc;
    }
    CatalogueStats s0{};
    s0.host = (CatalogueStats*)c->stats_host.ptr;
    e = hipMemcpy(c->stats.ptr, &s0, sizeof(s0), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(c->ticket.ptr, 0, sizeof(unsigned));
    if (e != hipSuccess) {
        (void)gs_destroy(c);
        return hip_fail(e, "context set-up");
    }
    *out = c;
    return GS_OK;
}

extern "C" int gs_destroy(gs_ctx* c)
{
    if (!c) return GS_OK;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    c->xyz.release(); c->w.release(); c->buf.release();
    c->rank.release(); c->boff.release(); c->cell_start.release(); c->chunk_nc.release(); c->chunk_off.release();
    c->scan_tmp.release(); c->ticket.release(); c->pw.release(); c->cell.release(); c->flags.release();
    c->orig.release(); c->zero.release(); c->params.release(); c->host.release();
    c->stats.release(); c->ingest.release(); c->stats_host.release(); c->ring.release();
    for (auto& ev : c->ring_ev)
        if (ev) (void)hipEventDestroy(ev);
    extra_release(c->extra);
    batch_release(c->batch);
    for (auto& ev : c->ev)
        if (ev) (void)hipEventDestroy(ev);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return GS_OK;
}

long double gs::fixed_sum(const double* w, int64_t n, int k)
{
    unsigned __int128 s = 0;
    for (int64_t i = 0; i < n; ++i) {
        uint64_t lo, hi;
        wsum_fixed(w[i], k, lo, hi);
        s += ((unsigned __int128)hi << 64) | lo;
    }
    return std::ldexp((long double)s, -k);
}

int gs::ctx_catalogue_info(gs_ctx* c, const double* xyz, const double* w, const int32_t* buf, int64_t n, int64_t n_data,
                           double* xyz_out, double* w_out, int32_t* buf_out, IngestScratch* scratch, CatalogueInfo* out)
{
    *out = CatalogueInfo{};
    out->wsum_d = (long double)n_data;
    out->wsum_r = (long double)(n - n_data);
    if (n == 0) return GS_OK;
    hipError_t e = launch_ingest(xyz, w, buf, n, n_data, xyz_out, w_out, buf_out, scratch, c->stats.ptr, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return hip_fail(e, "catalogue copy");
    const CatalogueStats& s = *(const CatalogueStats*)c->stats_host.ptr;
    if (w) {
        if (s.v[8] < 1e308) {
            double v = 0.0;
            (void)hipMemcpy(&v, w + (int64_t)s.v[8], sizeof(double), hipMemcpyDeviceToHost);
            return fail(GS_EINVAL, "weights must be finite and >= 0 (w[%lld]=%g)", (long long)s.v[8], v);
        }
        const int k = wsum_scale(std::max(s.v[6], s.v[7]));
        auto sum = [&](int q) {
            return std::ldexp((long double)(((unsigned __int128)s.s[q + 1] << 64) | s.s[q]), -k);
        };
        out->wsum_d = sum(0);
        out->wsum_r = sum(2);
        if (std::max(s.v[6], s.v[7]) > 0) out->wmax = std::max(s.v[6], s.v[7]);
        if (s.v[6] > 0) out->wmax_d = s.v[6];
        if (s.v[7] > 0) out->wmax_r = s.v[7];
    }
    for (int k = 0; k < 6; ++k) {
        if (!std::isfinite(s.v[k])) return fail(GS_EINVAL, "catalogue has non-finite coordinates");
        out->bbox[k] = s.v[k];
    }
    return GS_OK;
}

// Takes a catalogue in device memory over.  No half-set catalogue stays behind a failure.
static int ingest(gs_ctx* c, const double* d_xyz, const double* d_w, const int32_t* d_buf, int64_t n_data,
                  int64_t n_rand)
{
    CatalogueInfo s;
    int rc = ctx_catalogue_info(c, d_xyz, d_w, d_buf, n_data + n_rand, n_data, c->xyz.ptr, c->w.ptr, c->buf.ptr,
                                c->ingest.ptr, &s);
    if (rc) return rc;
    c->has_w = d_w != nullptr;
    c->has_buf = d_buf != nullptr;
    std::copy(s.bbox, s.bbox + 6, c->bbox);
    c->wsum_d = s.wsum_d;
    c->wsum_r = s.wsum_r;
    c->wmax = s.wmax;
    c->wmax_d = s.wmax_d;
    c->wmax_r = s.wmax_r;
    c->n_data = n_data;
    c->n_rand = n_rand;
    return GS_OK;
}

static int check_catalogue(gs_ctx* c, const double* xyz, int64_t n_data, int64_t n_rand)
{
    if (!c) return fail(GS_EINVAL, "NULL context or coordinates");
    c->n_data = c->n_rand = 0;      // no catalogue stays behind a failure
    c->grid_valid = false;
    if (!xyz && n_data + n_rand > 0) return fail(GS_EINVAL, "NULL context or coordinates");
    if (n_data < 0 || n_rand < 0 || n_data + n_rand > (int64_t)INT32_MAX - 1024)
        return fail(GS_EINVAL, "bad catalogue size (n_data=%lld n_rand=%lld)", (long long)n_data, (long long)n_rand);
    return set_device(c);
}

// Host memory to the device through a ring of four pinned pieces: a piece is filled while the ones before it
// are on their way (a copy from pageable memory is staged by the runtime, one piece at a time).
static int upload(gs_ctx* c, void* dst, const void* src, size_t bytes)
{
    constexpr size_t kPiece = (size_t)1 << 20;
    int rc;
    if ((rc = c->ring.reserve(4 * kPiece))) return rc;
    for (auto& ev : c->ring_ev)
        if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess)
            return fail(GS_EHIP, "hipEventCreate");
    hipError_t e = hipSuccess;
    size_t k = 0;
    for (size_t at = 0; at < bytes && e == hipSuccess; at += kPiece, ++k) {
        const size_t m = std::min(kPiece, bytes - at);
        unsigned char* p = c->ring.ptr + (k & 3) * kPiece;
        e = hipEventSynchronize(c->ring_ev[k & 3]);     // the piece's last copy (also one of an earlier call)
        if (e == hipSuccess) {
            memcpy(p, (const unsigned char*)src + at, m);
            e = hipMemcpyAsync((unsigned char*)dst + at, p, m, hipMemcpyHostToDevice, c->stream);
        }
        if (e == hipSuccess) e = hipEventRecord(c->ring_ev[k & 3], c->stream);
    }
    return e == hipSuccess ? GS_OK : hip_fail(e, "catalogue upload");
}

extern "C" int gs_set_catalogue(gs_ctx* c, const double* xyz, const double* w, const int32_t* buf, int64_t n_data,
                                int64_t n_rand)
{
    int rc = check_catalogue(c, xyz, n_data, n_rand);
    if (rc) return rc;
    const int64_t n = n_data + n_rand;
    if ((rc = c->xyz.reserve(3 * n)) || (w && (rc = c->w.reserve(n))) || (buf && (rc = c->buf.reserve(n)))) return rc;
    if ((rc = upload(c, c->xyz.ptr, xyz, 3 * n * sizeof(double))) || (w && (rc = upload(c, c->w.ptr, w, n * sizeof(double)))) ||
        (buf && (rc = upload(c, c->buf.ptr, buf, n * sizeof(int32_t)))))
        return rc;
    return ingest(c, c->xyz.ptr, w ? c->w.ptr : nullptr, buf ? c->buf.ptr : nullptr, n_data, n_rand);
}

extern "C" int gs_set_catalogue_device(gs_ctx* c, const double* d_xyz, const double* d_w, const int32_t* d_buf,
                                       int64_t n_data, int64_t n_rand)
{
    int rc = check_catalogue(c, d_xyz, n_data, n_rand);
    if (rc) return rc;
    const int64_t n = n_data + n_rand;
    if ((rc = c->xyz.reserve(3 * n)) || (d_w && (rc = c->w.reserve(n))) || (d_buf && (rc = c->buf.reserve(n)))) return rc;
    return ingest(c, d_xyz, d_w, d_buf, n_data, n_rand);
}

namespace gs {

// h rounded up to 11 significant bits: then k*h is exact in FP32 for |k| < 2^13
double round11(double h)
{
    int ex;
    const double fr = std::frexp(h, &ex);
    return std::ldexp(std::ceil(std::ldexp(fr, 11)), ex - 11);
}

// Picks the y/z cell edge for a catalogue with bounding box bbox: rmax / m rounded up to 11 significant
// bits (then k*h is exact in FP32 for |k| < 2^13), widened while the grid, with x cells of edge h / sx,
// would exceed max_cells.
double choose_h_bbox(const double* bbox, double rmax, int m, int64_t max_cells, int sx)
{
    int ex;
    double fr = std::frexp(rmax / m, &ex);
    double h = std::ldexp(std::ceil(std::ldexp(fr, 11)), ex - 11);
    for (;;) {
        int64_t nc = 1;
        for (int k = 0; k < 3; ++k) nc *= (int64_t)std::floor((bbox[3 + k] - bbox[k]) / (k == 0 ? h / sx : h)) + 1;
        if (nc <= max_cells) break;
        h = std::ldexp(std::ceil(std::ldexp(std::frexp(h * 1.25, &ex), 11)), ex - 11);
    }
    return h;
}

static double choose_h(const gs_ctx* c, double rmax, int m, int sx)
{
    return choose_h_bbox(c->bbox, rmax, m, (int64_t)1 << 24, sx);
}

int grid_desc(const double* bbox, double h, int sx, int64_t max_cells, GridDesc* out)
{
    GridDesc g{};
    g.h = h;
    g.hx = h / sx;
    int64_t ncell = 1;
    for (int k = 0; k < 3; ++k) {
        g.lo[k] = bbox[k];
        g.dim[k] = (int32_t)std::floor((bbox[3 + k] - bbox[k]) / (k == 0 ? g.hx : h)) + 1;
        ncell *= g.dim[k];
    }
    if (ncell > max_cells) return fail(GS_ELIMIT, "grid too large (%lld cells)", (long long)ncell);
    g.ncell = (int32_t)ncell;
    g.h32 = (float)h;
    g.hx32 = (float)g.hx;
    *out = g;
    return GS_OK;
}

// The context's grid with cells h and h / sx, and `extra` cleared bytes (a multiple of 256) at zero.ptr for
// the caller, cleared in the same launch as the cell counts behind them.
static int build_grid(gs_ctx* c, double h, int sx, size_t extra)
{
    const bool have = c->grid_valid && c->grid_h == h && c->grid_sx == sx;
    const int64_t n = c->n_data + c->n_rand;
    GridDesc g = c->g;
    int rc;
    if (!have && (rc = grid_desc(c->bbox, h, sx, (int64_t)1 << 26, &g))) return rc;
    const size_t clear = extra + (have ? 0 : (2 * (size_t)g.ncell + 1) * sizeof(int32_t));
    if (clear == 0) return GS_OK;
    if ((rc = c->zero.reserve(clear))) return rc;
    hipError_t e = launch_fill_u32(c->zero.ptr, (int64_t)(clear / 4), 0u, c->stream);
    if (e == hipSuccess && !have) {
        c->grid_valid = false;
        if ((rc = c->rank.reserve(n)) || (rc = c->boff.reserve(cell_scan_blocks(g.ncell))) ||
            (rc = c->cell_start.reserve(g.ncell + 1)) || (rc = c->pw.reserve(n)) || (rc = c->cell.reserve(n)) ||
            (rc = c->flags.reserve(n)) || (rc = c->orig.reserve(n)))
            return rc;
        GridArgs a{};
        a.xyz = c->xyz.ptr;
        a.w = c->has_w ? c->w.ptr : nullptr;
        a.buf = c->has_buf ? c->buf.ptr : nullptr;
        a.n = n;
        a.n_data = c->n_data;
        a.ncell = g.ncell;
        a.g = g;
        a.rank = c->rank.ptr;
        a.count = (int32_t*)(c->zero.ptr + extra);
        a.boff = c->boff.ptr;
        a.ticket = c->ticket.ptr;
        a.pw = c->pw.ptr;
        a.cell = c->cell.ptr;
        a.flags = c->flags.ptr;
        a.orig = c->orig.ptr;
        a.cell_start = c->cell_start.ptr;
        e = launch_cell_sort(a, c->stream);
        if (e == hipSuccess) {
            c->g = g;
            c->grid_h = h;
            c->grid_sx = sx;
            c->row_chunks_valid = false;
            c->grid_valid = true;
        }
    }
    return e == hipSuccess ? GS_OK : hip_fail(e, "grid build");
}

PairGrid ctx_pair_grid(const gs_ctx* c, const gs_params& p)
{
    return pair_grid(c->n_data + c->n_rand, c->bbox, p.rmax, p.cell_div, (int64_t)1 << 24);
}

int ctx_build_pair_grid(gs_ctx* c, const PairGrid& q, size_t extra, unsigned char** cleared)
{
    int rc = build_grid(c, q.h, q.sx, extra);
    if (cleared) *cleared = c->zero.ptr;
    return rc;
}

int ctx_row_chunks(gs_ctx* c)
{
    if (c->row_chunks_valid) return GS_OK;
    const int nrow = c->g.dim[1] * c->g.dim[2];
    int rc;
    if ((rc = c->chunk_nc.reserve(nrow + 1)) || (rc = c->chunk_off.reserve(nrow + 1)) ||
        (rc = c->scan_tmp.reserve(scan_scratch_size(nrow + 1))))
        return rc;
    hipError_t e = launch_row_chunks(c->cell_start.ptr, c->g.dim[0], nrow, kChunk, c->chunk_nc.ptr, c->stream);
    if (e == hipSuccess) e = exclusive_scan(c->chunk_nc.ptr, c->chunk_off.ptr, nrow + 1, c->scan_tmp.ptr, c->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(&c->n_chunks, c->chunk_off.ptr + nrow, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return hip_fail(e, "row chunks");
    c->row_chunks_valid = true;
    return GS_OK;
}

HostBuf& ctx_host(gs_ctx* c) { return c->host; }

int ctx_thresholds(gs_ctx* c, const gs_params& p, double* t)
{
    for (const auto& k : c->thresholds)
        if (k.rmin == p.rmin && k.rmax == p.rmax && k.nbins == p.nbins && (k.log_bins != 0) == (p.log_bins != 0)) {
            std::copy(k.t.begin(), k.t.end(), t);
            return GS_OK;
        }
    int rc = gs_bin_thresholds(&p, t);
    if (rc) return rc;
    if (c->thresholds.size() >= 8) c->thresholds.erase(c->thresholds.begin());
    c->thresholds.push_back({p.rmin, p.rmax, p.nbins, p.log_bins, std::vector<double>(t, t + p.nbins + 2)});
    return GS_OK;
}

// Cells per rmax of the adjoint kernels for n points in bounding box bbox: the finest grid (m <= 8)
// whose cells still hold ~32 points or more.
static int adjoint_cell_div(int64_t n, const double* bbox, double rmax)
{
    double vol = 1.0;
    for (int k = 0; k < 3; ++k) vol *= std::max(bbox[3 + k] - bbox[k], rmax * 1e-3);
    const double dens = n / vol;
    int best = 1;
    for (int m = 1; m <= 8; ++m) {
        const double h = rmax / m;
        if (dens * h * h * h >= 32.0) best = m;
    }
    return best;
}

static int env_int(const char* name)    // a tuning override, 0 if unset or empty
{
    const char* ev = getenv(name);
    return ev && *ev ? atoi(ev) : 0;
}

// Modelled VALU cycles per point of the pair kernel with chunks of `group` points on cells h and h / sx.  A
// chunk spans about group / (dens h^2) in x; its candidates are half the volume within rmax of its box
// (grown by the neighbour rows' cell width), in tiles of 64 that cost group / 2 steps of two pairs.
static double pair_cost(const PairGrid& q, int group, double dens, double len_x, double rmax, double* cap,
                        double* tiles_out)
{
    const double lin = std::max(dens * q.h * q.h, 1e-30);       // points per unit length of a row
    const double row = lin * len_x;
    const double len = std::min(group / lin, len_x);
    *cap = std::min(std::max(2.0 * len, 0.25 * rmax), rmax);    // a chunk's largest extent
    const double pieces = std::max(1.0, len / *cap);
    const double pts = std::max(1.0, row) / std::max(1.0, std::ceil(row / group)) / pieces;     // per chunk
    const double ax = len / pieces + 1.5 * q.h / q.sx, ay = 2.0 * q.h;
    const double vol = ax * ay * ay + 2.0 * (2.0 * ax * ay + ay * ay) * rmax + M_PI * (ax + 2.0 * ay) * rmax * rmax +
                       4.0 / 3.0 * M_PI * rmax * rmax * rmax;
    const double tiles = 0.5 * dens * vol / kWave + 0.5;
    const double rows = 0.5 * M_PI * (q.mst + 1.0) * (q.mst + 1.0);
    *tiles_out = tiles;
    return (tiles * (47.0 * group + 150.0) + 1500.0 + rows * 250.0) / pts;
}

void pair_group(PairGrid& q, double dens, double len_x, double rmax)
{
    const int want = env_int("GS_PAIR_GROUP");
    double cap = rmax, c, tiles;
    q.cost = 1e300;
    for (int group : {64, 32, 16}) {
        if ((want == 16 || want == 32 || want == 64) && want != group) continue;
        const double cost = pair_cost(q, group, dens, len_x, rmax, &c, &tiles);
        if (cost < q.cost) { q.cost = cost; q.group = group; q.tiles = tiles; cap = c; }
    }
    const double hx = q.h / q.sx;
    q.cap_cells = (int)std::min(std::floor(cap / hx), 1e6);
    q.ext = std::max((q.cap_cells + 1) * hx, q.h) * 1.001;
}

PairGrid pair_grid(int64_t n, const double* bbox, double rmax, int cell_div, int64_t max_cells)
{
    double vol = 1.0;
    for (int k = 0; k < 3; ++k) vol *= std::max(bbox[3 + k] - bbox[k], rmax * 1e-3);
    const double dens = (double)n / vol;
    PairGrid best;
    for (int m = cell_div > 0 ? cell_div : 1; m <= (cell_div > 0 ? cell_div : 8); ++m) {
        PairGrid q;
        q.m = m;
        q.sx = pair_cell_sx();
        q.h = choose_h_bbox(bbox, rmax, m, max_cells, q.sx);
        q.mst = (int)std::ceil(rmax / q.h - 1e-12);
        pair_group(q, dens, std::max(bbox[3] - bbox[0], rmax * 1e-3), rmax);
        if (best.h == 0 || q.cost < best.cost) best = q;
    }
    return best;
}

int pair_lg_parts(int64_t n, const PairGrid& q)
{
    const int want = env_int("GS_PAIR_PARTS");
    const double chunks = std::max(1.0, (double)n / q.group);
    int lg = 0;
    if (want) {
        while (lg < 6 && (2 << lg) <= want && chunks * (2 << lg) < 1e9) ++lg;
    } else {
        // two items for every SIMD at least; beyond that, items of no less than 12 tiles' work with the
        // smallest chunks, as long as a wave takes few of them (an item costs some 10 us of dependent loads)
        while (lg < 6 && (chunks * (1 << lg) < 2048.0 ||
                          (chunks * (1 << lg) < 131072.0 && q.tiles * q.group / 16.0 >= 12.0 * (2 << lg))))
            ++lg;
    }
    return lg;
}

// x cells per y/z cell of the pair kernels' grid: finer x cells cut each stencil row to the x-range that
// can reach rmax from the work item's apexes, at the cost of one more entry per cell in the cell index.
static int cell_sx_env(const char* name, int dflt)
{
    const char* ev = getenv(name);                  // tuning override (unset or empty: automatic)
    if (ev && *ev) {
        int v = atoi(ev), sx = 1;
        while (sx < 64 && sx * 2 <= v) sx *= 2;
        return sx;
    }
    return dflt;
}
int pair_cell_sx() { return cell_sx_env("GS_CELL_SX", 8); }

// x cells per y/z cell of the triplet and quad kernels' grid: their gathers scan the apex's stencil, whose
// x-range finer x cells cut close to the sphere.
int apex_cell_sx() { return cell_sx_env("GS_T3_CELL_SX", 4); }

int default_cell_div(const gs_ctx* c, double rmax, int mode)
{
    if (mode != 2) return 1;
    return adjoint_cell_div(c->n_data + c->n_rand, c->bbox, rmax);
}

}  // namespace gs

// ====================================================================== 2PCF

namespace gs {

// Launch shape of the pair kernel: work-group size, LDS histogram replicas (spreading same-bin atomics)
// and, with buffer points, histogram planes.  256-thread work-groups (four waves per shared histogram)
// are kept when they reach 16 resident waves per CU; otherwise larger work-groups share one histogram
// among more waves to raise residency.  Among shapes with the same residency, more replicas win.  A
// histogram that does not fit otherwise runs with one plane and, at last, one wave.  Cached per variant.
int pair2_shape(const PairVariant& v, PairShape* out)
{
    const int ev_reps = env_int("GS_PAIR_REPS"), ev_wg = env_int("GS_PAIR_WG");     // tuning overrides
    char key[96];
    snprintf(key, sizeof(key), "%d/%d/%d%d%d%d/%d/%d", v.nb, v.nm, (int)v.fp64, (int)v.weighted, (int)v.logb,
             (int)v.buf, ev_reps, ev_wg);
    static std::mutex mu;
    static std::map<std::string, PairShape> shapes;
    std::lock_guard<std::mutex> lock(mu);
    auto it = shapes.find(key);
    if (it != shapes.end()) {
        *out = it->second;
        return it->second.waves ? GS_OK : fail(GS_ELIMIT, "histogram of %d bins does not fit in LDS", 3 * v.nb * v.nm);
    }
    PairShape s;
    auto consider = [&](int planes, int r, int w) {
        if (ev_reps && ev_reps != r) return;
        if (ev_wg && ev_wg != w) return;
        if (pair2_lds_bytes(v.nb, v.nm, planes, r, v.weighted, false, w) > kPairLdsMax) return;
        const int waves = pair2_occupancy(v, planes, r, false, w) * (w / kWave);
        if (waves > s.waves || (waves == s.waves && planes == s.planes && r > s.reps))
            s = PairShape{planes, r, w, waves};
    };
    // The most waves, then the most replicas, of work-groups of 256 threads; of 512 where those would have a single
    // replica (1,800 weighted bins, 4M points: 256 threads and 1 replica 164 ms, 512 and 2 158 ms; 360 bins, 150k
    // points: 1 to 8 replicas of either 0.40 ms; 144 bins, 9k points: 256 threads 0.039, 512 0.048 ms).  Sizes that
    // do not fill the four SIMDs evenly only where there is no other (640 threads, 20 waves by the occupancy query,
    // 232 ms).
    for (int planes = v.buf ? 2 : 1; planes >= 1 && s.waves == 0; --planes) {
        for (int w = 256; w <= 512 && (w == 256 || s.reps == 1); w += 256)
            for (int r = 1; r <= 32; r *= 2) consider(planes, r, w);
        if (s.waves < 16)
            for (int r = 1; r <= 32; r *= 2)
                for (int w = 320; w <= 1024; w += 64) consider(planes, r, w);
    }
    for (int w = 192; w >= 64 && s.waves == 0; w -= 64) consider(1, 1, w);
    shapes[key] = s;
    if (s.waves == 0) return fail(GS_ELIMIT, "histogram of %d bins does not fit in LDS", 3 * v.nb * v.nm);
    *out = s;
    return GS_OK;
}

// Work split of a walk over one catalogue's chunks on work-groups of wg threads, `waves` waves per CU; returns
// the number of work-groups.
int walk_shape(WalkArgs& a, const PairGrid& q, int64_t n, int wg, int waves, int n_cu)
{
    a.group = q.group;
    a.cap_cells = q.cap_cells;
    a.lg_parts = pair_lg_parts(n, q);
    a.n = (int32_t)n;
    // no more work-groups than items could fill, a multiple of 8 (the same number on each XCD)
    const int64_t wpg = wg / kWave;
    const int64_t items = ((n + q.group - 1) / q.group) << a.lg_parts;
    const int64_t nblocks = std::min<int64_t>((int64_t)n_cu * waves / wpg, (items + wpg - 1) / wpg);
    return (int)((nblocks + 7) / 8 * 8);
}

// Launch of the pair kernel over one catalogue's chunks (a: the arrays and outputs).
hipError_t pair_launch(PairArgs& a, const PairVariant& var, const PairShape& shape, const PairGrid& q, int64_t n,
                       int n_cu, hipStream_t st)
{
    a.reps = shape.reps;
    a.planes = shape.planes;
    const int nblocks = walk_shape(a, q, n, shape.wg, shape.waves, n_cu);
    return launch_pair2(a, var, nblocks, shape.wg, st);
}

// Pair kernel outputs (counts [3][nb][nm], 128-bit class sums, statistics) -> the C ABI's outputs:
// cnt, the class sums of raw-weight products, N2 = DD/Wd^2 - DR/(Wd Wr) + RR/Wr^2 and N3 = RR/Wr^2
// (gramsci.F90:373-379 over ordered pairs), and the pair statistics of st (times left to the caller).
void combine2(const unsigned long long* h_out, int nb, int nm, const BinDesc& B, bool weighted, long double Wd,
              long double Wr, uint64_t* cnt, double* wsum, double* n2, double* n3, gs_stats* st)
{
    const int nbt = 3 * nb * nm;
    uint64_t total = 0;
    for (int k = 0; k < nbt; ++k) {
        if (cnt) cnt[k] = h_out[k];
        total += h_out[k];
    }
    std::vector<long double> S(nbt);
    for (int k = 0; k < nbt; ++k)
        S[k] = weighted ? fx_value(h_out[nbt + 2 * k], h_out[nbt + 2 * k + 1], fx_pair_class_shift(B, k / (nb * nm)))
                        : (long double)h_out[k];
    if (wsum)
        for (int k = 0; k < nbt; ++k) wsum[k] = (double)S[k];
    for (int b = 0; b < nb * nm; ++b) {
        const long double dd = S[b], dr = S[nb * nm + b], rr = S[2 * nb * nm + b];
        long double v2 = 0, v3 = 0;
        if (Wd > 0) v2 += dd / (Wd * Wd);
        if (Wd > 0 && Wr > 0) v2 -= dr / (Wd * Wr);
        if (Wr > 0) { v2 += rr / (Wr * Wr); v3 = rr / (Wr * Wr); }
        if (n2) n2[b] = (double)v2;
        if (n3) n3[b] = (double)v3;
    }
    if (st) {
        memset(st, 0, sizeof(*st));
        st->n_units = total;
        st->n_binned = total;
        st->n_candidates = h_out[3 * nbt + 0];
        st->n_evaluated = st->n_candidates;
        st->n_recheck = h_out[3 * nbt + 1];
        st->n_overflow = h_out[3 * nbt + 2];
    }
}

}  // namespace gs


extern "C" int gs_count_2pcf(gs_ctx* c, const gs_params* p, uint64_t* cnt, double* wsum, double* n2, double* n3,
                             gs_stats* st)
{
    if (!c) return fail(GS_EINVAL, "NULL context");
    int rc = check_params(p, 2);
    if (rc) return rc;
    if ((rc = set_device(c))) return rc;
    const int nb = p->nbins, nm = p->nmu;
    const int nbt = 3 * nb * nm;
    const bool weighted = c->has_w;
    const int64_t n = c->n_data + c->n_rand;
    const PairGrid q = ctx_pair_grid(c, *p);
    const std::vector<Row> rows = half_stencil(q.h, q.h / q.sx, p->rmax, q.mst);
    if ((int)rows.size() > kMaxRows) return fail(GS_ELIMIT, "stencil too large");
    double t64[kMaxBins + 2], xmax = 0;
    for (int k = 0; k < 6; ++k) xmax = std::max(xmax, std::fabs(c->bbox[k]));
    // Small catalogues are bound by launches, copies and waits, not by their pairs.  So parameters and results are
    // in pinned host memory (bins and stencil rows go to the device in one copy, the results are written back by
    // the last kernel), and hand-over plus count take 8 launches and 2 waits; with a copy per array, a memset per
    // buffer and 19 launches, 3,000 + 6,000 weighted points took 342 us, now 138 (the pair kernel: 41).
    const int copies = pair_copies(1, nbt);
    const size_t nwork = (size_t)copies * pair_copy_words(1, nbt), nout = 3 * (size_t)nbt + 4;
    const size_t rows_off = (sizeof(BinDesc) + 15) / 16 * 16, blob = rows_off + rows.size() * sizeof(Row);
    const size_t out_off = (blob + 255) / 256 * 256;
    if ((rc = ctx_thresholds(c, *p, t64)) || (rc = c->params.reserve(blob)) || (rc = c->host.reserve(out_off + nout * 8)))
        return rc;
    BinDesc& B = *(BinDesc*)c->host.ptr;
    if ((rc = fill_pair_bins(*p, t64, q, xmax, c->wmax_d, c->wmax_r, B))) return rc;
    std::copy(rows.begin(), rows.end(), (Row*)(c->host.ptr + rows_off));
    const PairVariant var{nb, nm, p->precision == GS_FP64 || B.wide, weighted, p->log_bins != 0, c->has_buf};
    PairShape shape;
    if ((rc = pair2_shape(var, &shape))) return rc;
    hipError_t e = hipMemcpyAsync(c->params.ptr, c->host.ptr, blob, hipMemcpyHostToDevice, c->stream);
    if (e != hipSuccess) return hip_fail(e, "parameter upload");

    // one region to clear: work counters, copies of the outputs, and the cell counts of the grid build
    const size_t queue_bytes = 64 * kQueuePad * sizeof(int32_t), clear = (queue_bytes + nwork * 8 + 255) / 256 * 256;
    (void)hipEventRecord(c->ev[0], c->stream);
    unsigned char* z = nullptr;
    if ((rc = ctx_build_pair_grid(c, q, clear, &z))) return rc;
    unsigned long long* work = (unsigned long long*)(z + queue_bytes);

    PairArgs a{};
    a.pw = c->pw.ptr;
    a.cell = c->cell.ptr;
    a.flags = c->flags.ptr;
    a.cell_start = c->cell_start.ptr;
    a.rows = (const Row*)(c->params.ptr + rows_off);
    a.bins = (const BinDesc*)c->params.ptr;
    a.queue = (int32_t*)z;
    a.out_cnt = work;
    a.out_w = work + 2 * nbt;
    a.out_stats = work + 6 * nbt;
    a.copies = copies;
    a.copy_stride = pair_copy_words(1, nbt);
    a.g = c->g;
    a.g.m = q.mst;
    a.nrows = (int)rows.size();
    (void)hipEventRecord(c->ev[2], c->stream);
    if (n > 0) {
        e = pair_launch(a, var, shape, q, n, c->n_cu, c->stream);
        if (e != hipSuccess) return hip_fail(e, "pair kernel launch");
    }
    (void)hipEventRecord(c->ev[3], c->stream);
    unsigned long long* const h_out = (unsigned long long*)(c->host.ptr + out_off);
    e = launch_pair_reduce(work, copies, 1, nbt, nm, weighted, h_out, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return hip_fail(e, "pair kernel");

    combine2(h_out, nb, nm, B, weighted, c->wsum_d, c->wsum_r, cnt, wsum, n2, n3, st);
    if (st) {
        float ms_grid = 0, ms_count = 0;
        (void)hipEventElapsedTime(&ms_grid, c->ev[0], c->ev[2]);
        (void)hipEventElapsedTime(&ms_count, c->ev[2], c->ev[3]);
        st->ms_grid = ms_grid;
        st->ms_count = ms_count;
        st->ms_kernel_avg = ms_count;
        st->cell_div = q.mst;
    }
    return GS_OK;
}

// ====================================================================== one-shot

static gs_ctx* g_ctx = nullptr;

static int oneshot_ctx(gs_ctx** c)
{
    if (!g_ctx) {
        int rc = gs_create(&g_ctx, 0);
        if (rc) return rc;
    }
    *c = g_ctx;
    return GS_OK;
}

extern "C" int gs_pcf2(const double* xyz, const double* w, const int32_t* buf, int64_t n_data, int64_t n_rand,
                       const gs_params* p, uint64_t* cnt, double* n2, double* n3, gs_stats* st)
{
    gs_ctx* c;
    int rc = oneshot_ctx(&c);
    if (rc) return rc;
    if ((rc = gs_set_catalogue(c, xyz, w, buf, n_data, n_rand))) return rc;
    return gs_count_2pcf(c, p, cnt, nullptr, n2, n3, st);
}

extern "C" int gs_pcf3(const double* xyz, const double* w, const int32_t* buf, int64_t n_data, int64_t n_rand,
                       const gs_params* p, uint64_t* cnt, double* n2, double* n3, gs_stats* st)
{
    gs_ctx* c;
    int rc = oneshot_ctx(&c);
    if (rc) return rc;
    if ((rc = gs_set_catalogue(c, xyz, w, buf, n_data, n_rand))) return rc;
    return gs_count_3pcf(c, p, cnt, nullptr, n2, n3, st);
}

extern "C" int gs_pcf4(const double* xyz, const double* w, const int32_t* buf, int64_t n_data, int64_t n_rand,
                       const gs_params* p, uint64_t* cnt, double* n2, double* n3, double* disc_n, double* disc_r,
                       gs_stats* st)
{
    gs_ctx* c;
    int rc = oneshot_ctx(&c);
    if (rc) return rc;
    if ((rc = gs_set_catalogue(c, xyz, w, buf, n_data, n_rand))) return rc;
    return gs_count_4pcf(c, p, cnt, n2, n3, disc_n, disc_r, st);
}

// Internal accessors for the other translation units (3PCF/4PCF/adjoint).
namespace gs {
CtxView view(gs_ctx* c)
{
    CtxView v;
    v.stream = c->stream;
    v.ev = c->ev;
    v.n_cu = c->n_cu;
    v.n_data = c->n_data;
    v.n_rand = c->n_rand;
    v.has_w = c->has_w;
    v.has_buf = c->has_buf;
    v.wsum_d = c->wsum_d;
    v.wsum_r = c->wsum_r;
    v.wmax = c->wmax;
    v.wmax_d = c->wmax_d;
    v.wmax_r = c->wmax_r;
    for (int k = 0; k < 6; ++k) v.bbox[k] = c->bbox[k];
    v.g = c->g;
    v.pw = c->pw.ptr;
    v.flags = c->flags.ptr;
    v.orig = c->orig.ptr;
    v.cell_start = c->cell_start.ptr;
    v.cell = c->cell.ptr;
    v.row_chunk = c->chunk_off.ptr;
    v.w = c->has_w ? c->w.ptr : nullptr;
    v.n_chunks = c->n_chunks;
    v.extra = &c->extra;
    v.batch = &c->batch;
    return v;
}
int ctx_build_grid(gs_ctx* c, double rmax, int m, int sx, double* h_out)
{
    double h = choose_h(c, rmax, m, sx);
    *h_out = h;
    return build_grid(c, h, sx, 0);
}
double ctx_xmax(gs_ctx* c)
{
    double xmax = 0;
    for (int k = 0; k < 6; ++k) xmax = std::max(xmax, std::fabs(c->bbox[k]));
    return xmax;
}
int ctx_set_device(gs_ctx* c) { return set_device(c); }
}  // namespace gs
