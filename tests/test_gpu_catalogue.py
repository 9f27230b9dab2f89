"""The pass that takes a catalogue over and the cell sort, at the edges of their blocks and of the pieces that
host memory is staged in: exact weight sums, counts against a kd-tree, invalid input wherever it stands."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from gramsci_amd._lib import GsError
from gramsci_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


# one point; a block of the pass (192 threads x 4 coordinates); a staged piece of 2^20 bytes of coordinates or
# weights, less one, plus one; more than four pieces; more blocks than the pass has at most
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 43690, 43691, 131072, 131073, 300007])
@pytest.mark.parametrize("device", [False, True])
def test_sizes(eng, n, device):
    import torch
    rng = np.random.default_rng(n)
    box = 40.0 * max(n / 20000.0, 1.0) ** (1 / 3)
    xyz = rng.uniform(-box / 2, box / 2, (n, 3))
    w = np.exp(rng.normal(0, 1, n))
    buf = (rng.random(n) < 0.2).astype(np.int32)
    nd = n // 3
    put = (lambda a: torch.from_numpy(a).cuda()) if device else (lambda a: a)
    eng.set_catalogue(put(xyz), put(w), nd, put(buf))
    r = eng.pcf2(0.0, 2.0, 1)
    # apexes without the buffer flag: every ordered pair from a non-buffer point, by class
    cls = [slice(0, nd), slice(nd, n)]
    free = buf != 1
    tree = [cKDTree(xyz[s]) if xyz[s].size else None for s in cls]
    apex = [cKDTree(xyz[s][free[s]]) if free[s].any() else None for s in cls]
    own = [int(free[s].sum()) for s in cls]

    def pairs(a, b):
        return int(apex[a].count_neighbors(tree[b], 2.0)) if apex[a] is not None and tree[b] is not None else 0

    assert [int(v) for v in r["cnt"].reshape(-1)] == [pairs(0, 0) - own[0], pairs(0, 1) + pairs(1, 0), pairs(1, 1) - own[1]]
    # the normalised sums divide by the weight sums of each class, exact to the last bits
    W = [np.sum(w[s].astype(np.longdouble)) for s in cls]
    ws = r["wsum"].reshape(-1).astype(np.longdouble)
    if nd:
        n2 = ws[0] / W[0] ** 2 - ws[1] / (W[0] * W[1]) + ws[2] / W[1] ** 2
        n3 = ws[2] / W[1] ** 2
        scale = max(abs(ws[0] / W[0] ** 2), abs(ws[1] / (W[0] * W[1])), abs(n3), 1e-300)
        assert abs(r["n2"].reshape(-1)[0] - n2) <= 1e-14 * scale
        assert abs(r["n3"].reshape(-1)[0] - n3) <= 1e-14 * scale


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("at", [0, 767, 131071, 131072, 300006])
def test_invalid_input_is_found_and_leaves_no_catalogue(eng, device, at):
    import torch
    n = 300007
    rng = np.random.default_rng(1)
    xyz = rng.uniform(0, 50.0, (n, 3))
    put = (lambda a: torch.from_numpy(a).cuda()) if device else (lambda a: a)
    for bad in (-1.0, np.nan, np.inf):
        w = np.ones(n)
        w[at] = bad
        w[n - 1] = bad
        with pytest.raises(GsError, match=rf"w\[{at}\]"):
            eng.set_catalogue(put(xyz), put(w), n // 2)
        assert eng.pcf2(0.0, 2.0, 1)["cnt"].sum() == 0
    x = xyz.copy()
    x[at, at % 3] = np.inf
    with pytest.raises(GsError, match="non-finite"):
        eng.set_catalogue(put(x), None, n // 2)


def test_wide_grid_of_empty_cells(eng):
    # many blocks of cell counts, nearly all of them zero, with pairs across rows and blocks
    rng = np.random.default_rng(4)
    a = rng.uniform(0, 3000.0, (400, 3))
    xyz = np.concatenate([a, a + rng.normal(0, 3.0, a.shape)])
    eng.set_catalogue(xyz, None, 400)
    r = eng.pcf2(0.0, 12.0, 1)
    t = [cKDTree(xyz[:400]), cKDTree(xyz[400:])]
    cc = [int(t[i].count_neighbors(t[j], 12.0)) for i, j in ((0, 0), (0, 1), (1, 1))]
    assert [int(v) for v in r["cnt"].reshape(-1)] == [cc[0] - 400, 2 * cc[1], cc[2] - 400]


def test_outlying_point_widens_the_cells(eng):
    # one point far away widens the cells until most points are an apex's candidates: triangles of unit weights leave the
    # matrix kernel, four-point sums the LDS; counts are those without that point
    rng = np.random.default_rng(5)
    n = 12000
    x = rng.uniform(0, 20.0, (n, 3))
    w = rng.uniform(0.5, 2.0, n)
    far = np.concatenate([x, [[5000.0, 5000.0, 5000.0]]])
    got = []
    for xyz, weights in ((x, w), (far, np.append(w, 1.0))):
        eng.set_catalogue(xyz, None, 3000)
        r3 = eng.pcf3(0.2, 1.2, 4)
        eng.set_catalogue(xyz, weights, 3000)
        r3w, r4w = eng.pcf3(0.2, 1.2, 4), eng.pcf4(0.3, 0.9, 3)
        got.append((r3, r3w, r4w))
    a, b = got
    for k in range(3):
        assert a[k]["cnt"].sum() > 0 and np.array_equal(a[k]["cnt"], b[k]["cnt"]), k
        assert b[k]["stats"]["n_candidates"] > 8192 * n
    assert np.array_equal(a[1]["wsum"], b[1]["wsum"])


def test_engine_knows_that_a_failed_hand_over_left_nothing(eng):
    import torch
    x = np.random.default_rng(2).uniform(0, 9.0, (50, 3))
    eng.set_catalogue(x, np.ones(50), 20)
    with pytest.raises(GsError):
        eng.set_catalogue(x, -np.ones(50), 20)
    assert (eng.n_data, eng.n_rand) == (0, 0)
    g = np.ones((2, 1))
    assert eng.adjoint2(g, g, 0.0, 5.0, 2).size == 0
    with pytest.raises(ValueError):         # an output for 50 points would stay as it was
        eng.adjoint2(g, g, 0.0, 5.0, 2, out=torch.empty(50, dtype=torch.float64, device="cuda"))
    # arguments that never reach the context leave its catalogue and the engine's sizes alone
    eng.set_catalogue(x, None, 20)
    with pytest.raises(ValueError):
        eng.set_catalogue(x, np.ones(49), 20)
    assert (eng.n_data, eng.n_rand) == (20, 30)
    assert eng.adjoint2(g, g, 0.0, 5.0, 2).size == 50
