"""CPU check of the pair kernel's bin constants (fill_pair_bins): the kernel looks the certain interval of a pair up at
its estimated bin, and the table has one entry past the last bin, so the estimate of a pair that is not rejected has to
stay below nbins + 1 wherever the FP32 geometry runs.  The estimate is formed here as the kernel does it, with the
square root or logarithm off by a unit in the last place either way."""
import ctypes
import os
import subprocess
import textwrap

import numpy as np
import pytest

from gramsci_amd import _lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = textwrap.dedent("""
    #include "gs_api_internal.h"
    // wide, rej_lo, rej_hi, ua, ub for n points in a box of edge len at the origin
    extern "C" int pair_bins(const gs_params* p, long n, double len, double* out)
    {
        double t[gs::kMaxBins + 2];
        int rc = gs_bin_thresholds(p, t);
        if (rc) return rc;
        const double bbox[6] = {0, 0, 0, len, len, len};
        gs::BinDesc B;
        const gs::PairGrid q = gs::pair_grid(n, bbox, p->rmax, p->cell_div, 1 << 24);
        if ((rc = gs::fill_pair_bins(*p, t, q, len, 1.0, 1.0, B))) return rc;
        out[0] = B.wide; out[1] = B.rej_lo; out[2] = B.rej_hi; out[3] = B.ua; out[4] = B.ub;
        return 0;
    }
""")


@pytest.fixture(scope="module")
def pair_bins(tmp_path_factory):
    L.lib()
    d = tmp_path_factory.mktemp("pair_bins")
    (d / "pair_bins.cpp").write_text(SOURCE)
    so = str(d / "pair_bins.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I" + os.path.join(ROOT, "gramsci_amd", "csrc"), "-I/opt/rocm/include",
                           str(d / "pair_bins.cpp"), "-o", so, L.LIB_PATH, "-Wl,-rpath," + os.path.dirname(L.LIB_PATH)])
    f = ctypes.CDLL(so).pair_bins
    f.argtypes = [ctypes.c_void_p, ctypes.c_long, ctypes.c_double, ctypes.c_void_p]

    def call(rmin, rmax, nbins, log, n, length):
        p = L.make_params(rmin, rmax, nbins, 1, log)
        out = np.zeros(5)
        rc = f(ctypes.addressof(p), n, length, out.ctypes.data)
        return None if rc else out          # None: the bins themselves are refused

    return call


def _largest_estimate(rej_lo, rej_hi, ua, ub, log):
    lo, hi = np.float32(rej_lo), np.float32(rej_hi)
    width = hi - lo
    s = hi
    while np.nextafter(s, np.float32(np.inf)) - lo <= np.nextafter(width, np.float32(np.inf)):
        s = np.nextafter(s, np.float32(np.inf))         # the last s that the kernel does not reject
    with np.errstate(all="ignore"):
        f = np.log2(np.float64(s)) if log else np.sqrt(np.float64(s))
        f = np.float32(f)
        fs = [np.nextafter(f, np.float32(-np.inf)), f, np.nextafter(f, np.float32(np.inf))]
        u = [np.float32(np.float64(x) * np.float64(np.float32(ua)) + np.float64(np.float32(ub))) for x in fs]
    return float(np.max(u))


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("rmax", [88.8, 1.0, 0.37, 5000.0, 3e-4, 1e-12, 2e-39])
@pytest.mark.parametrize("nbins", [1, 10, 100, 127])
def test_estimates_stay_within_the_table(pair_bins, log, rmax, nbins):
    seen = narrow = 0
    for rel in np.concatenate([10.0 ** -np.arange(0.05, 7.0, 0.05), [1.02e-4, 1.35e-4]]):
        for length in (2.0, 50.0):
            out = pair_bins(rmax * (1.0 - rel), rmax, nbins, log, 3000, length * rmax)
            if out is None:
                continue
            seen += 1
            wide, rej_lo, rej_hi, ua, ub = out
            narrow += wide != 0
            if not wide:
                assert _largest_estimate(rej_lo, rej_hi, ua, ub, log) < nbins + 1, (rel, length)
    assert seen
    if rmax >= 0.3:
        # the FP32 geometry still takes every range but the narrow ones
        out = pair_bins(0.9 * rmax, rmax, min(nbins, 30), log, 3000, 50.0 * rmax)
        assert out[0] == 0
