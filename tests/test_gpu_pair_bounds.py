"""The bounds that make a pair's bin certain in the pair kernel, where they are easily too small: midpoints close to
the origin in every unit of length, points that are not numbers, bins of a narrow range, distances whose square no
float holds.  Counts equal the oracle's exactly."""
import numpy as np
import pytest

import oracle as O
from gramsci_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("scale", [1e-29, 1e-25, 1e-20, 1e-15, 1e-12, 1e-10, 8e-9, 8e-8, 1e-5, 1.0, 1e6, 1e15])
@pytest.mark.parametrize("eps", [1e-9, 1e-8, 1e-7, 1e-5])
def test_midpoints_at_the_origin(eng, scale, eps):
    # 1,500 pairs of points opposite each other, their midpoints within eps of the origin: the angle of such a pair
    # hangs on the last bits of its coordinates.  FP64 at every scale (FP32 rechecks all pairs below rmax = 1e-5)
    rng = np.random.default_rng(3)
    h = rng.normal(size=(1500, 3))
    h *= rng.uniform(0.1, 0.45, (1500, 1)) / np.linalg.norm(h, axis=1)[:, None]
    m = rng.normal(size=(1500, 3)) * eps
    xyz = np.concatenate([m + h, m - h]) * scale
    p = O.Params(0.05 * scale, 0.8 * scale, 3, 5, False)
    ref = O.pcf2(xyz, None, 1000, p)
    eng.set_catalogue(xyz, None, 1000)
    for prec in ("fp32", "fp64"):
        r = eng.pcf2(p.rmin, p.rmax, p.nbins, p.nmu, p.log_bins, prec)
        assert np.array_equal(r["cnt"], ref["cnt"]), prec


@pytest.mark.parametrize("weighted,buffered,nmu", [(True, False, 4), (False, False, 1), (True, True, 3)])
@pytest.mark.parametrize("share", [0.02, 0.5])
def test_points_that_are_not_numbers(eng, weighted, buffered, nmu, share):
    # a point with a NaN coordinate has no pairs, as in the reference's arithmetic (no comparison with NaN holds), and
    # takes none from the points beside it in its chunk
    rng = np.random.default_rng(5)
    n = 3000
    xyz = rng.uniform(0, 25.0, (n, 3))
    w = rng.uniform(0.5, 2.0, n) if weighted else None
    buf = (rng.random(n) < 0.3).astype(np.int32) if buffered else None
    for axis in range(3):
        bad = rng.random(n) < share
        bad[:2] = False
        x = xyz.copy()
        x[bad, axis] = np.nan
        g = ~bad
        p = O.Params(0.5, 5.0, 4, nmu, False)
        ref = O.pcf2(xyz[g], None if w is None else w[g], int(g[:1000].sum()), p, buf=None if buf is None else buf[g])
        eng.set_catalogue(x, w, 1000, buf)
        for prec in ("fp32", "fp64"):
            r = eng.pcf2(p.rmin, p.rmax, p.nbins, p.nmu, p.log_bins, prec)
            assert np.array_equal(r["cnt"], ref["cnt"]), (axis, prec)
            assert np.allclose(r["wsum"], ref["wsum"], rtol=1e-12, atol=0.0)
        if weighted:
            # no pairs, no gradient but that of the normalisation: dL/dwn of such a point is 0
            ga, gb = (eng.adjoint2(np.ones((4, nmu)), np.zeros((4, nmu)), 0.5, 5.0, 4, nmu, False, prec) for prec in ("fp32", "fp64"))
            assert np.all(np.isfinite(ga)) and np.max(np.abs(ga - gb)) <= 1e-11 * np.max(np.abs(gb))


@pytest.mark.parametrize("rmax", [1.7e19, 1.9e19, 3e25, 1e60])
@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("nmu", [1, 5])
def test_squared_distances_beyond_float(eng, rmax, log, nmu):
    # above 1.8e19 no float holds a squared distance: the bin's estimate is infinite, and has to stay within the table
    rng = np.random.default_rng(12)
    xyz = rng.uniform(0, 3.0, (600, 3)) * rmax
    p = O.Params(0.1 * rmax, rmax, 6, nmu, log)
    ref = O.pcf2(xyz, None, 250, p)
    eng.set_catalogue(xyz, None, 250)
    for prec in ("fp32", "fp64"):
        assert np.array_equal(eng.pcf2(p.rmin, p.rmax, 6, nmu, log, prec)["cnt"], ref["cnt"]), prec


@pytest.mark.parametrize("rel", [1e-2, 1e-3, 1.35e-4, 1.02e-4, 1e-5])
@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("nbins,nmu", [(100, 1), (127, 1), (20, 6)])
def test_narrow_ranges_of_bins(eng, rel, log, nbins, nmu):
    # the FP32 estimate of a bin is off by a sizeable part of it, or by more: FP64 geometry takes over
    rng = np.random.default_rng(14)
    xyz = rng.uniform(0, 100.0, (3000, 3))
    w = rng.uniform(0.5, 2.0, 3000)
    p = O.Params(88.8 * (1.0 - rel), 88.8, nbins, nmu, log)
    ref = O.pcf2(xyz, w, 1000, p)
    eng.set_catalogue(xyz, w, 1000)
    for prec in ("fp32", "fp64"):
        r = eng.pcf2(p.rmin, p.rmax, nbins, nmu, log, prec)
        assert np.array_equal(r["cnt"], ref["cnt"]) and r["stats"]["n_overflow"] == ref["overflow"], prec
    g2, g3 = rng.normal(size=(2, nbins, nmu))
    ref = O.adjoint2(xyz, w, 1000, p, g2, g3)
    for prec in ("fp32", "fp64"):
        got = eng.adjoint2(g2, g3, p.rmin, p.rmax, nbins, nmu, log, prec)
        # terms rounded to 2^-50 of the largest, at most 3000 a point
        assert np.max(np.abs(got - ref)) <= 1e-11 * np.max(np.abs(ref)), prec


@pytest.mark.parametrize("rmax", [1e148, 1e150, 1e151, 1e153])
@pytest.mark.parametrize("nmu", [1, 4])
def test_largest_rmax(eng, rmax, nmu):
    # up to the largest rmax with a finite square: the lanes without a point are beyond it
    rng = np.random.default_rng(15)
    xyz = rng.uniform(0, 3.0, (300, 3)) * rmax
    p = O.Params(0.1 * rmax, rmax, 3, nmu, nmu > 1)
    ref = O.pcf2(xyz, None, 100, p)
    eng.set_catalogue(xyz, None, 100)
    for prec in ("fp32", "fp64"):
        assert np.array_equal(eng.pcf2(p.rmin, p.rmax, 3, nmu, p.log_bins, prec)["cnt"], ref["cnt"]), prec


@pytest.mark.parametrize("weighted", [False, True])
def test_triplets_and_quads_beside_points_that_are_not_numbers(eng, weighted):
    rng = np.random.default_rng(6)
    n = 700
    xyz = rng.uniform(0, 12.0, (n, 3))
    w = rng.uniform(0.5, 2.0, n) if weighted else None
    bad = rng.random(n) < 0.2
    x = xyz.copy()
    x[bad, rng.integers(0, 3, int(bad.sum()))] = np.nan
    g = ~bad
    wg = np.ones(int(g.sum())) if w is None else w[g]
    nd = int(g[:250].sum())
    eng.set_catalogue(x, w, 250)
    for nmu in (1, 3):
        ref = O.pcf3(xyz[g], wg, nd, O.Params(0.5, 3.0, 3, nmu, False))
        for prec in ("fp32", "fp64"):
            assert np.array_equal(eng.pcf3(0.5, 3.0, 3, nmu, False, prec)["cnt"], ref["cnt"]), (nmu, prec)
    ref = O.pcf4(xyz[g], wg, nd, O.Params(0.5, 3.0, 2, 1, False))
    assert np.array_equal(eng.pcf4(0.5, 3.0, 2)["cnt"], ref["cnt"])
