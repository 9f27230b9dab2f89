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
