"""The 4PCF's teams and masks at their edges: neighbour lists around 64, 128 and 256 (one wave, the work-group, each
number of mask words), one wave per apex or not, weighted sums in LDS and in global memory, tetrahedra, buffer points,
16 bins (the largest table).  Counts equal the oracle's exactly; sums within the tolerances of the 4PCF's other tests."""
import numpy as np
import pytest

import oracle as O
from gramsci_amd import catalog as C
from gramsci_amd.engine import Engine
from test_gpu_34pcf import _close, _close_disc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


def _check(eng, xyz, w, nd, p, tetra, buf=None):
    ref = (O.pcf4_tetra if tetra else O.pcf4)(xyz, w, nd, p, buf=buf)
    eng.set_catalogue(xyz, w, nd, buf)
    r = (eng.pcf4_tetra if tetra else eng.pcf4)(p.rmin, p.rmax, p.nbins, p.log_bins)
    assert np.array_equal(r["cnt"], ref["cnt"])
    if not tetra:
        assert r["stats"]["n_units"] == ref["n_quads"]
    # the sums whose terms have one sign (N2 and discN cancel between classes: a relative tolerance of the result
    # says nothing about FP64 sums there)
    assert _close(r["n3"], ref["n3"]) and _close_disc(r["disc_r"], ref["disc_r"])
    return r


@pytest.mark.parametrize("wave", ["0", "1"])
@pytest.mark.parametrize("tetra", [False, True])
@pytest.mark.parametrize("n", [0, 1, 3, 4, 5, 6, 33, 63, 64, 65, 66, 67, 127, 128, 129, 130])
def test_list_lengths(eng, monkeypatch, wave, tetra, n):
    # n points within reach of each other: every apex has n - 1 neighbours
    monkeypatch.setenv("GS_T4_WAVE", wave)
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 4.0, (n, 3))
    w = np.exp(rng.normal(0, 0.3, n))
    # rmin leaves out some sides, rmax none
    _check(eng, xyz, w, n // 3, O.Params(1.5, 7.0, 3, 1, False), tetra)
    buf = (rng.random(n) < 0.4).astype(np.int32)
    _check(eng, xyz, np.ones(n), n // 3, O.Params(1.0, 7.0, 2, 1, True), tetra, buf)


@pytest.mark.parametrize("n", [256, 257, 258])
def test_four_mask_words(eng, n):
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 4.0, (n, 3))
    _check(eng, xyz, np.exp(rng.normal(0, 0.3, n)), n // 3, O.Params(2.8, 7.0, 2, 1, False), False)


@pytest.mark.parametrize("nbins", [1, 2, 3, 4, 6, 16])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("wave", ["0", "1"])
def test_bins(eng, monkeypatch, nbins, weighted, wave):
    # count histograms in LDS (up to 3 bins) and global memory, weighted sums likewise, the table up to its limit
    monkeypatch.setenv("GS_T4_WAVE", wave)
    d, r = C.clustered(900, 40.0, 51), C.uniform(1500, 40.0, 52)
    xyz = np.concatenate([d, r])
    w = C.lognormal_weights(len(xyz), 0.2, 53) if weighted else np.ones(len(xyz))
    _check(eng, xyz, w, 900, O.Params(2.0, 7.0, nbins, 1, False), False)


@pytest.mark.parametrize("tetra", [False, True])
def test_every_pass(eng, monkeypatch, tetra):
    # lists of 3 to several hundred neighbours: the wave, 64 / 128 / 256 and device-memory passes in one count
    d = C.clustered(1200, 30.0, 61)
    xyz = np.concatenate([d, C.uniform(2500, 60.0, 62)])
    w = C.lognormal_weights(len(xyz), 0.2, 63)
    p = O.Params(3.0, 8.0, 2, 1, False)
    base = _check(eng, xyz, w, 1200, p, tetra)
    for k in ("64", "128"):
        monkeypatch.setenv("GS_T4_KMAX_LDS", k)
        r = _check(eng, xyz, w, 1200, p, tetra)
        for q in ("n_candidates", "n_units", "n_overflow"):
            assert r["stats"][q] == base["stats"][q], q


def test_largest_tables(eng):
    # 16 bins and cells of rmax / 16: the perimeter table and the stencil rows beside the shortest list
    d, r = C.clustered(300, 20.0, 71), C.uniform(500, 20.0, 72)
    xyz = np.concatenate([d, r])
    w = C.lognormal_weights(len(xyz), 0.2, 73)
    ref = O.pcf4(xyz, w, 300, O.Params(1.0, 6.0, 16, 1, False))
    eng.set_catalogue(xyz, w, 300)
    for div in (2, 16):
        out = eng.pcf4(1.0, 6.0, 16, False, cell_div=div)
        assert np.array_equal(out["cnt"], ref["cnt"]) and out["stats"]["n_units"] == ref["n_quads"], div
        assert _close(out["n3"], ref["n3"]) and _close_disc(out["disc_r"], ref["disc_r"])


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("nbins,tetra", [(9, False), (10, False), (14, False), (16, False), (11, True), (40, True), (127, True)])
@pytest.mark.parametrize("n", [60, 129, 200])
def test_many_bins(eng, weighted, nbins, tetra, n):
    # lists for which no mask per bin fits the LDS: one mask a neighbour, or (tetrahedra) always one, their bins so wide
    # that the first few hold all sides
    rng = np.random.default_rng(n + nbins)
    xyz = rng.uniform(0, 4.0, (n, 3))
    w = np.exp(rng.normal(0, 0.3, n)) if weighted else np.ones(n)
    p = O.Params(0.5, 0.5 + 1.2 * nbins, nbins, 1, False) if tetra else O.Params(2.6, 7.0, nbins, 1, False)
    _check(eng, xyz, w, n // 3, p, tetra)


def test_time_of_the_kernels(eng):
    # the reported time is the kernels': with 16 bins the host prepares 127 MB for the results meanwhile, 20 ms, and
    # 200 points' quads take less than a millisecond
    xyz = np.random.default_rng(1).uniform(0, 30.0, (200, 3))
    eng.set_catalogue(xyz, None, 100)
    assert min(eng.pcf4(1.0, 6.0, 16, False)["stats"]["ms_count"] for _ in range(3)) < 5.0
