"""The one-launch preparation of sets of up to 8,192 particles: results and
validation verdicts at the edges of its range (32 particles a workgroup, 1,024
threads, the first size of the general preparation), and where its curve order
has nothing to go by (all particles at one point, or on one axis)."""
import numpy as np
import pytest

import oracle
from starsmasher_amd import Gravity, SG_PREC_FP64, SphgravError, _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _set(n, kind="cloud"):
    rng = np.random.default_rng(n)
    pos = rng.normal(size=(n, 3))
    if kind == "axis":
        pos[:, 1:] = 0.0
    if kind == "point":
        pos[:] = 1.5
    return (*pos.T.copy(), rng.uniform(0.5, 1.0, n) / n, rng.uniform(0.01, 0.2, n))


@pytest.mark.parametrize("n,kind", [(1, "cloud"), (31, "cloud"), (32, "cloud"), (33, "axis"),
                                    (512, "point"), (1023, "cloud"), (1025, "cloud"), (4097, "axis"),
                                    (8191, "cloud"), (8192, "cloud"), (8193, "cloud")])
def test_sizes(grav, n, kind):
    args = _set(n, kind)
    res = grav.compute(*args, nkernel=0, precision=SG_PREC_FP64)
    rows = np.unique(np.linspace(0, n - 1, min(n, 400)).astype(int))
    ref = oracle.direct(*args, nkernel=0, rows=rows)
    scale = np.sqrt(np.mean(np.stack(ref[:3]) ** 2)) + 1e-300
    for k in range(3):
        assert np.abs(res[k][rows] - ref[k]).max() <= 1e-11 * max(scale, np.abs(ref[3]).max())
    assert (np.abs(res[3][rows] - ref[3]) / np.maximum(np.abs(ref[3]), 1e-300)).max() < 1e-11


@pytest.mark.parametrize("n", [1, 40, 1500, 8192])
def test_verdicts(grav, n):
    for field, value, status in ((3, 0.0, _lib.SG_ERR_MASS), (3, -1.0, _lib.SG_ERR_MASS),
                                 (4, 0.0, _lib.SG_ERR_RANGE2), (0, np.nan, _lib.SG_ERR_NONFINITE),
                                 (2, -np.inf, _lib.SG_ERR_NONFINITE), (3, np.nan, _lib.SG_ERR_NONFINITE)):
        for at in {0, n // 2, n - 1}:
            args = [a.copy() for a in _set(n)]
            args[field][at] = value
            with pytest.raises(SphgravError) as e:
                grav.compute(*args)
            assert e.value.status == status
    grav.compute(*_set(n))
