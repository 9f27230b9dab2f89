"""CPU check of the 4PCF's LDS layout (quad4_lds_bytes): the longest neighbour list that fits a work-group's LDS, for
every number of bins.  Apexes with more neighbours run with their lists in device memory, several times as slow."""
import ctypes
import os
import subprocess
import textwrap

import pytest

from gramsci_amd import _lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = textwrap.dedent("""
    #include <cmath>
    #include "gs_api_internal.h"
    // bytes of a work-group with lists of kmax and the fewest masks, on cells of rmax / m
    extern "C" long quad_bytes(int nb, int tetra, int weighted, int wave, int kmax, int m)
    {
        gs::QuadArgs a{};
        a.tetra = tetra;
        a.ncell = tetra ? nb : nb * (nb + 1) * (nb + 2) * (nb + 3) / 24 * nb * nb;
        a.nrows = (int)gs::full_stencil(1.0 / m, 0.25 / m, 1.0, m).size();
        a.lds_hist = (size_t)a.ncell * 64 <= 16 * 1024;
        a.kmax = kmax;
        return (long)gs::quad4_lds_bytes(a, nb, weighted != 0, wave != 0);
    }
""")


@pytest.fixture(scope="module")
def quad_bytes(tmp_path_factory):
    L.lib()
    d = tmp_path_factory.mktemp("quad_lists")
    (d / "quad_lists.cpp").write_text(SOURCE)
    so = str(d / "quad_lists.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I" + os.path.join(ROOT, "gramsci_amd", "csrc"), "-I/opt/rocm/include",
                           str(d / "quad_lists.cpp"), "-o", so, L.LIB_PATH, "-Wl,-rpath," + os.path.dirname(L.LIB_PATH)])
    f = ctypes.CDLL(so).quad_bytes
    f.restype = ctypes.c_long
    return f


BUDGET = 160 * 1024 - 256       # gfx950's LDS, less the kernel's static part


@pytest.mark.parametrize("weighted", [0, 1])
@pytest.mark.parametrize("m", [1, 2, 4])
def test_longest_lists(quad_bytes, weighted, m):
    for nb in range(1, 17):
        # beside the perimeter table of nb^4 entries
        assert quad_bytes(nb, 0, weighted, 0, 256 if nb <= 14 else 128, m) <= BUDGET, nb
    for nb in range(1, 128):
        assert quad_bytes(nb, 1, weighted, 0, 256, m) <= BUDGET, nb


def test_wave_lists(quad_bytes):
    # four lists of 64 a work-group
    for nb in range(1, 14):
        assert quad_bytes(nb, 0, 0, 1, 64, 2) <= BUDGET, nb
    for nb in range(1, 128):
        assert quad_bytes(nb, 1, 0, 1, 64, 2) <= BUDGET, nb
