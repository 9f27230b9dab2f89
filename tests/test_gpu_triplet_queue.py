"""The general triplet kernel's queue of binned pairs and its packed weighted histogram: lists around a queue's
length, every work-group size and mode, and lists so long that an apex's pairs are taken in pieces and the packed
counts are drained within it.  Counts equal the oracle's exactly; sums are exact integers, equal between geometries
and to those of the pass with lists in device memory, which has neither queue nor packed planes."""
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


def _close(a, b):
    # 1e-12 of the largest entry: the oracle adds the signed class sums in another order (no entry without data points)
    b = np.asarray(b).reshape(np.shape(a))
    fin = np.isfinite(b)
    return np.all(np.abs(a - b)[fin] <= 1e-12 * np.max(np.abs(b[fin]), initial=0.0))


@pytest.mark.parametrize("team", ["64", "128", "256"])
@pytest.mark.parametrize("nmu,weighted,equi", [(1, True, False), (3, False, False), (3, True, False), (1, False, True),
                                               (1, True, True), (2, True, True)])
@pytest.mark.parametrize("n", [1, 2, 3, 12, 13, 24, 65, 130])
def test_list_lengths(eng, monkeypatch, team, nmu, weighted, equi, n):
    monkeypatch.setenv("GS_T3_WG", team)
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 4.0, (n, 3)) + 20.0
    w = C.lognormal_weights(n, 0.4, 7) if weighted else None
    for buf in (None, (rng.random(n) < 0.3).astype(np.int32)):
        p = O.Params(0.5, 5.0, 3, nmu, buf is not None)
        ref = (O.pcf3_equi if equi else O.pcf3)(xyz, np.ones(n) if w is None else w, n // 3, p, buf=buf)
        eng.set_catalogue(xyz, w, n // 3, buf)
        run = eng.pcf3_equi if equi else eng.pcf3
        a, b = (run(p.rmin, p.rmax, p.nbins, nmu, p.log_bins, prec) for prec in ("fp32", "fp64"))
        assert np.array_equal(a["cnt"], b["cnt"]) and np.array_equal(a["cnt"].reshape(ref["cnt"].shape), ref["cnt"])
        if weighted:
            assert np.array_equal(a["wsum"], b["wsum"])
            assert _close(a["n2"], ref["n2"])


@pytest.mark.parametrize("nmu,weighted", [(1, True), (2, True), (2, False)])
def test_long_lists(eng, monkeypatch, nmu, weighted):
    # 1,500 points within reach of each other in one bin: 1.1 million pairs an apex, more than a piece, and more than
    # 2^22 increments of a bin within four apexes; equal weights make every term the largest
    rng = np.random.default_rng(21)
    xyz = rng.uniform(0, 1.0, (1500, 3)) + 5.0
    w = np.ones(1500) if weighted else None
    eng.set_catalogue(xyz, w, 500, None)
    a = eng.pcf3(0.0, 2.0, 1, nmu, False, "fp32")
    monkeypatch.setenv("GS_T3_KMAX", "64")
    monkeypatch.setenv("GS_T3_KMAX_LDS", "64")
    b = eng.pcf3(0.0, 2.0, 1, nmu, False, "fp32")
    assert a["cnt"].sum() == 1500 * 1499 * 1498 // 2
    assert np.array_equal(a["cnt"], b["cnt"])
    if weighted:
        assert np.array_equal(a["wsum"], b["wsum"])


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("batched", [False, True])
def test_packed_counts_beyond_their_width(eng, prec, batched):
    # 2,000 points within reach of each other, every side in the first of 6 bins: a histogram of 224 entries has one
    # replica, and lists of 28 bytes an entry (FP64: 44) leave the LDS of a compute unit room for two work-groups (FP64:
    # one), so that the triangles, counted three times, average more than 2^22 a histogram: without the drains some
    # packed count would run over
    import torch
    groups = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    n = 2000
    assert n * (n - 1) * (n - 2) // 2 > groups * 2 ** 22 * 1.5
    rng = np.random.default_rng(22)
    xyz = rng.uniform(0, 1.0, (n, 3)) + 5.0
    w = rng.uniform(0.5, 1.0, n)
    if batched:
        eng.set_catalogue_batched(xyz, w, None, np.array([0, n]), np.array([n]))
        a = eng.pcf3_batched(0.0, 12.0, 6, 1, False, prec, cell_div=2)
        cnt, wsum = a["cnt"][0, :, 0], a["wsum"][0, :, 0]
    else:
        eng.set_catalogue(xyz, w, n)
        a = eng.pcf3(0.0, 12.0, 6, 1, False, prec)
        cnt, wsum = a["cnt"], a["wsum"]
    assert cnt[0, 0] == n * (n - 1) * (n - 2) // 2 and cnt.sum() == cnt[0, 0]
    p1, p2, p3 = (np.sum(w.astype(np.longdouble) ** k) for k in (1, 2, 3))
    exact = float((p1 ** 3 - 3 * p1 * p2 + 2 * p3) / 2)
    # each product is rounded down to 2^-60 of the largest, and twice in FP64 before: 4e-16 of it
    assert abs(wsum[0, 0] - exact) <= 2e-15 * exact


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("nmu,weighted,equi", [(1, True, False), (3, False, False), (2, True, False), (1, False, True)])
@pytest.mark.parametrize("n", [449, 450, 451, 577, 900])
def test_lists_by_rows(eng, prec, nmu, weighted, equi, n):
    # n points within reach of each other: every apex has n - 1 neighbours (isotropic: those after it), on both sides of
    # the 448 entries from which the pairs go to the waves by rows
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 4.0, (n, 3)) + 20.0
    w = C.lognormal_weights(n, 0.4, 7) if weighted else None
    p = O.Params(2.0, 8.0, 3, nmu, False)
    ref = (O.pcf3_equi if equi else O.pcf3)(xyz, np.ones(n) if w is None else w, n // 3, p)
    eng.set_catalogue(xyz, w, n // 3)
    a = (eng.pcf3_equi if equi else eng.pcf3)(p.rmin, p.rmax, p.nbins, nmu, False, prec)
    assert np.array_equal(a["cnt"].reshape(ref["cnt"].shape), ref["cnt"])
    if weighted:
        assert _close(a["n2"], ref["n2"])
