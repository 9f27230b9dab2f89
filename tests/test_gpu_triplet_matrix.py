"""The isotropic 3PCF of unit weights on the matrix cores: neighbour lists around its 16-point blocks, both team
sizes, every pass, buffer points, regions, scales, and the bins beyond its histogram (the general kernel's).  Counts
are integers and equal the oracle's, and those of the FP64 kernel, exactly."""
import numpy as np
import pytest

import oracle as O
from gramsci_amd import catalog as C
from gramsci_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


def _check(eng, xyz, nd, p, buf=None):
    ref = O.pcf3(xyz, np.ones(len(xyz)), nd, p, buf=buf)
    eng.set_catalogue(xyz, None, nd, buf)
    a = eng.pcf3(p.rmin, p.rmax, p.nbins, 1, p.log_bins, "fp32")
    b = eng.pcf3(p.rmin, p.rmax, p.nbins, 1, p.log_bins, "fp64")
    assert np.array_equal(a["cnt"], b["cnt"]) and np.array_equal(a["cnt"].reshape(ref["cnt"].shape), ref["cnt"])
    for k in ("n_candidates", "n_units", "n_overflow"):
        assert a["stats"][k] == b["stats"][k], k
    return a


@pytest.mark.parametrize("team", ["64", "256", ""])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 15, 16, 17, 18, 32, 33, 34, 63, 64, 65, 66, 81, 129])
def test_list_lengths(eng, monkeypatch, team, n):
    # n points within reach of each other: lists of n - 1, n - 2, ..., 0 neighbours, around whole blocks of 16
    monkeypatch.setenv("GS_T3_WG", team)
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 4.0, (n, 3))
    _check(eng, xyz, n // 3, O.Params(0.5, 7.0, 4, 1, False))
    buf = (rng.random(n) < 0.4).astype(np.int32)
    _check(eng, xyz, n // 3, O.Params(0.2, 3.0, 3, 1, True), buf)


@pytest.mark.parametrize("team", ["64", "256"])
@pytest.mark.parametrize("kmax,kmax_lds", [("", ""), ("64", ""), ("64", "128"), ("128", "64")])
@pytest.mark.parametrize("buffered", [False, True])
def test_passes(eng, monkeypatch, team, kmax, kmax_lds, buffered):
    # lists beyond the first pass's go to the second, beyond its to the one with lists in device memory
    monkeypatch.setenv("GS_T3_WG", team)
    monkeypatch.setenv("GS_T3_KMAX", kmax)
    monkeypatch.setenv("GS_T3_KMAX_LDS", kmax_lds)
    rng = np.random.default_rng(3)
    xyz = np.concatenate([C.clustered(2500, 60.0, 31), C.uniform(4000, 60.0, 32)])
    buf = (rng.random(len(xyz)) < 0.2).astype(np.int32) if buffered else None
    _check(eng, xyz, 2500, O.Params(1.0, 9.0, 5, 1, True), buf)


@pytest.mark.parametrize("rmin,rmax,nbins,log", [(0.0, 8.0, 1, False), (0.0, 8.0, 7, False), (7.9, 8.0, 3, False),
                                                 (0.001, 8.0, 12, True), (2.0, 8.0, 13, False), (1.0, 8.0, 20, True)])
def test_bins(eng, rmin, rmax, nbins, log):
    # 12 bins: the largest histogram of the matrix kernel; 13 and 20: the general kernel
    xyz = np.concatenate([C.clustered(1500, 50.0, 41), C.uniform(2500, 50.0, 42)])
    _check(eng, xyz, 1500, O.Params(rmin, rmax, nbins, 1, log))


@pytest.mark.parametrize("scale", [2.0 ** -60, 3e-9, 1.0, 7e5, 2.0 ** 60])
@pytest.mark.parametrize("at", [0.0, 1e4])
def test_scales(eng, scale, at):
    # the squared sides are computed in units of rmax's power of two; `at`: far from the origin
    rng = np.random.default_rng(5)
    xyz = (rng.uniform(0, 20.0, (1500, 3)) + at) * scale
    _check(eng, xyz, 500, O.Params(1.0 * scale, 6.0 * scale, 4, 1, False))


def test_edges_and_duplicates(eng):
    # a lattice: many sides exactly on bin edges, and coincident points (FP64 decides)
    g = np.stack(np.meshgrid(*[np.arange(8.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
    xyz = np.concatenate([g, g[::3], g[::7] + 1e-9])
    a = _check(eng, xyz, 300, O.Params(1.0, 4.0, 3, 1, False))
    assert a["stats"]["n_recheck"] > 0
    _check(eng, xyz, 300, O.Params(0.0, 3.0, 3, 1, False))


@pytest.mark.parametrize("team", ["64", "256"])
@pytest.mark.parametrize("buffered", [False, True])
def test_regions(eng, monkeypatch, team, buffered):
    # regions of different sizes (empty, single-point) in one launch; work items span them
    monkeypatch.setenv("GS_T3_WG", team)
    rng = np.random.default_rng(9)
    sizes = [0, 1, 700, 2, 0, 1300, 64, 900, 3]
    off = np.concatenate([[0], np.cumsum(sizes)])
    nd = np.array([s // 3 for s in sizes])
    xyz = np.concatenate([rng.uniform(0, 30.0 * (s / 1000.0) ** (1 / 3) + 3.0, (s, 3)) + 100.0 * k
                          for k, s in enumerate(sizes)])
    buf = (rng.random(len(xyz)) < 0.3).astype(np.int32) if buffered else None
    p = O.Params(0.5, 8.0, 4, 1, False)
    for kmax in ("", "64"):
        monkeypatch.setenv("GS_T3_KMAX", kmax)
        eng.set_catalogue_batched(xyz, None, buf, off, nd)
        out = eng.pcf3_batched(p.rmin, p.rmax, p.nbins, 1, p.log_bins, "fp32", cell_div=2)
        for _ in range(2):      # replays of the captured pipeline
            again = eng.pcf3_batched(p.rmin, p.rmax, p.nbins, 1, p.log_bins, "fp32", cell_div=2)
            assert np.array_equal(again["cnt"], out["cnt"])
        for r in range(len(sizes)):
            s = slice(off[r], off[r + 1])
            ref = O.pcf3(xyz[s], np.ones(sizes[r]), nd[r], p, buf=None if buf is None else buf[s])
            assert np.array_equal(out["cnt"][r].reshape(ref["cnt"].shape), ref["cnt"]), r
