"""The pair kernel's work decomposition at its edges: chunk sizes, items per chunk, partial chunks and
tiles, the drains of its packed weighted histogram, and the ranges outside the FP32 error bounds."""
import numpy as np
import pytest

import oracle as O
from gramsci_amd import catalog as C
from gramsci_amd._lib import GsError
from gramsci_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


def _check(eng, xyz, w, nd, p, buf=None):
    ref = O.pcf2(xyz, w, nd, p, buf=buf)
    for prec in ("fp32", "fp64"):
        eng.set_catalogue(xyz, w, nd, buf)
        r = eng.pcf2(p.rmin, p.rmax, p.nbins, p.nmu, p.log_bins, prec)
        assert np.array_equal(r["cnt"], ref["cnt"]), prec
        for k in ("wsum", "n2", "n3"):      # sums of at most n^2 rounded products, exact in fixed point
            assert np.all(np.abs(r[k] - ref[k]) <= 1e-13 * max(np.abs(ref[k]).max(), 1e-300)), (prec, k)


@pytest.mark.parametrize("group", ["16", "32", "64"])
@pytest.mark.parametrize("parts", ["1", "8", "64"])
@pytest.mark.parametrize("weighted,buffered,nmu", [(True, False, 6), (True, True, 5), (False, True, 1), (False, False, 4)])
def test_groups_and_parts(eng, monkeypatch, group, parts, weighted, buffered, nmu):
    monkeypatch.setenv("GS_PAIR_GROUP", group)
    monkeypatch.setenv("GS_PAIR_PARTS", parts)
    rng = np.random.default_rng(7)
    # a dense cluster (long tiles), sparse rows (chunks cut into pieces) and single points
    xyz = np.concatenate([C.clustered(1203, 40.0, 5), rng.uniform(0, 40.0, (805, 3)), rng.uniform(0, 400.0, (61, 3))])
    w = np.exp(rng.normal(0, 0.3, len(xyz))) if weighted else None
    buf = (rng.random(len(xyz)) < 0.4).astype(np.int32) if buffered else None
    _check(eng, xyz, w, 1203, O.Params(0.5, 9.0, 5, nmu, True), buf)


@pytest.mark.parametrize("n", [2, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129])
def test_chunk_edges(eng, monkeypatch, n):
    # one x-row of n points: chunks of 16 / 32 / 64 and their remainders
    rng = np.random.default_rng(n)
    xyz = np.column_stack([np.sort(rng.uniform(0, 30.0, n)), rng.uniform(0, 1.0, n), rng.uniform(0, 1.0, n)])
    w = rng.uniform(0.5, 2.0, n)
    for group in ("16", "32", "64"):
        monkeypatch.setenv("GS_PAIR_GROUP", group)
        _check(eng, xyz, w, n // 2, O.Params(0.0, 12.0, 4, 3, False))


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_packed_histogram_drains(eng, prec):
    # every pair in one bin: each work-group passes 2^20 increments of it, so the waves' scans drain it
    # before the 22-bit counts run over; closed form n (n - 1), (sum w)^2 - sum w^2
    n = 60000
    rng = np.random.default_rng(3)
    xyz = 100.0 + rng.uniform(0.0, 1.0, (n, 3))
    w = rng.uniform(0.1, 1.0, n)
    eng.set_catalogue(xyz, w, n)
    r = eng.pcf2(0.0, 2.0, 1, 1, False, prec)
    assert int(r["cnt"][0, 0, 0]) == n * (n - 1)
    s, s2 = np.sum(w.astype(np.longdouble)), np.sum(w.astype(np.longdouble) ** 2)
    exact = float(s * s - s2)
    assert abs(r["wsum"][0, 0, 0] - exact) <= 1e-14 * exact


@pytest.mark.parametrize("scale", [1e-40, 1e-12, 1e-7, 1e-3, 1e6, 1e9, 1e40])
def test_scales_beyond_the_fp32_bounds(eng, scale):
    # coordinates scaled by powers of ten: beyond the range of the FP32 mu estimate every pair is
    # rechecked, and beyond that of its bin table the FP64 geometry runs
    rng = np.random.default_rng(9)
    xyz = (rng.uniform(0, 30.0, (700, 3)) - 7.0) * scale
    _check(eng, xyz, None, 300, O.Params(1.0 * scale, 8.0 * scale, 4, 5, True))


def test_cells_much_wider_than_rmax(eng):
    # a few points in a box of 1e6 rmax: the grid's cells are widened to ~1e3 rmax and the FP32 guard
    # bands with them
    rng = np.random.default_rng(11)
    a = rng.uniform(0, 1e6, (60, 3))
    xyz = np.concatenate([a + rng.normal(0, 0.4, a.shape) for _ in range(6)])
    _check(eng, xyz, None, 100, O.Params(0.1, 2.0, 4, 3, False))


@pytest.mark.parametrize("group", ["16", "32", "64"])
@pytest.mark.parametrize("parts", ["1", "16"])
@pytest.mark.parametrize("buffered,nmu,log", [(False, 6, True), (True, 5, False), (True, 1, True)])
def test_adjoint_groups_and_parts(eng, monkeypatch, group, parts, buffered, nmu, log):
    monkeypatch.setenv("GS_PAIR_GROUP", group)
    monkeypatch.setenv("GS_PAIR_PARTS", parts)
    rng = np.random.default_rng(17)
    # dense points (more than 64 tiles to a chunk, so that its sums are flushed within an item), sparse ones
    xyz = np.concatenate([rng.uniform(10.0, 22.0, (4700, 3)), rng.uniform(0, 60.0, (301, 3))])
    w = np.exp(rng.normal(0, 0.3, len(xyz)))
    buf = (rng.random(len(xyz)) < 0.4).astype(np.int32) if buffered else None
    p = O.Params(0.5 if log else 0.0, 12.0, 5, nmu, log)
    g2, g3 = rng.normal(size=(2, 5, nmu))
    ref = O.adjoint2(xyz, w, 2000, p, g2, g3, buf=buf)
    eng.set_catalogue(xyz, w, 2000, buf)
    got = eng.adjoint2(g2, g3, p.rmin, p.rmax, p.nbins, p.nmu, log)
    # each term is rounded to 2^-50 of the largest; at most 5000 terms a point
    assert np.max(np.abs(got - ref)) <= 1e-11 * np.max(np.abs(ref))


@pytest.mark.parametrize("nbins,nmu", [(127, 106), (106, 127), (116, 116)])
def test_largest_histograms(eng, nbins, nmu):
    # 40,386 and 40,368 counts: the whole LDS of a compute unit but 2 KB
    rng = np.random.default_rng(8)
    xyz = rng.uniform(0, 10.0, (500, 3)) + 3.0
    _check(eng, xyz, None, 200, O.Params(0.5, 6.0, nbins, nmu, False))


@pytest.mark.parametrize("weighted,fits", [(False, 3900), (True, 780)])
def test_batched_histogram_limit(eng, weighted, fits):
    # four histograms in 64 KiB: 3,966 counts, 793 with sums
    rng = np.random.default_rng(9)
    xyz = rng.uniform(0, 10.0, (400, 3)) + 3.0
    w = rng.uniform(0.5, 2.0, 400) if weighted else None
    eng.set_catalogue_batched(xyz, w, None, np.array([0, 150, 400]), np.array([70, 100]))
    nm = fits // 3 // 13
    out = eng.pcf2_batched(0.5, 6.0, 13, nm, False, "fp32", cell_div=2)
    assert out["cnt"].sum() > 0
    with pytest.raises(GsError, match="do not fit in LDS"):
        eng.pcf2_batched(0.5, 6.0, 13, nm + 5, False, "fp32", cell_div=2)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("buffered", [False, True])
def test_packed_counts_beyond_their_width(eng, monkeypatch, prec, buffered):
    # one replica and 1,024 threads a work-group, at most two of those on a compute unit: the pairs of one bin average
    # more than 2^22 a histogram, the width of a packed count, so without the scans some count would run over
    import torch
    monkeypatch.setenv("GS_PAIR_REPS", "1")
    monkeypatch.setenv("GS_PAIR_WG", "1024")
    groups = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    n = 90000
    rng = np.random.default_rng(4)
    xyz = 100.0 + rng.uniform(0.0, 1.0, (n, 3))
    w = rng.uniform(0.1, 1.0, n)
    buf = (rng.random(n) < 0.02).astype(np.int32) if buffered else None
    k = 0 if buf is None else int(buf.sum())
    assert (n - k) * (n - k - 1) // 2 > groups * 2 ** 22 * 1.5
    eng.set_catalogue(xyz, w, n, buf)
    r = eng.pcf2(0.0, 2.0, 1, 1, False, prec)
    assert int(r["cnt"][0, 0, 0]) == (n - k) * (n - 1)
    wl = w.astype(np.longdouble)
    apex = wl if buf is None else wl[buf == 0]
    exact = float(np.sum(apex) * np.sum(wl) - np.sum(apex ** 2))
    # each product is rounded to 2^-52 of the largest, one: 1e-16 of the mean product of 0.3 in the end
    assert abs(r["wsum"][0, 0, 0] - exact) <= 1e-14 * exact


def test_packed_counts_of_waves_beyond_their_width(eng):
    # a batch has a histogram for every wave, at most 32 on a compute unit
    import torch
    waves = 32 * torch.cuda.get_device_properties(0).multi_processor_count
    n = 280000
    assert n * (n - 1) // 2 > waves * 2 ** 22 * 1.1
    rng = np.random.default_rng(5)
    xyz = 100.0 + rng.uniform(0.0, 1.0, (n, 3))
    w = rng.uniform(0.1, 1.0, n)
    eng.set_catalogue_batched(xyz, w, None, np.array([0, n]), np.array([n]))
    r = eng.pcf2_batched(0.0, 2.0, 1, 1, False, cell_div=2)
    assert int(r["cnt"][0, 0, 0, 0]) == n * (n - 1)
    s, s2 = np.sum(w.astype(np.longdouble)), np.sum(w.astype(np.longdouble) ** 2)
    exact = float(s * s - s2)
    assert abs(r["wsum"][0, 0, 0, 0] - exact) <= 1e-14 * exact


def test_largest_weighted_histograms(eng):
    # 10,098 entries of 16 bytes fill the LDS; one bin more is refused
    rng = np.random.default_rng(10)
    xyz = rng.uniform(0, 10.0, (400, 3)) + 3.0
    w = rng.uniform(0.5, 2.0, 400)
    _check(eng, xyz, w, 150, O.Params(0.5, 6.0, 33, 102, False))
    with pytest.raises(GsError, match="does not fit in LDS"):
        eng.pcf2(0.5, 6.0, 99, 35, False)
