"""The grad-h term alone (k_psi_only) against the oracle: the number of parts a
group's chunks are cut into changes with the i-range (64 at one group, fewer
from there), chunks and tiles are ragged, and a set of large supports lists more
pairs of a visit than fit the list.  Bound 1e-11, as in the other tests of the
term: its pairs are FP64, and the largest polynomial coefficients cancel.
"""
import numpy as np
import pytest

import oracle
from starsmasher_amd import Gravity
from test_gpu_unordered import _set

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


@pytest.mark.parametrize("kind,n,ibeg,ni,nk", [
    ("plummer", 1, 0, 1, 0), ("plummer", 63, 0, 63, 1), ("plummer", 65, 0, 65, 2),
    ("plummer", 257, 0, 257, 0), ("two", 3000, 0, 3000, 1), ("two", 3000, 2999, 1, 0),
    ("bigH", 3001, 100, 1025, 2), ("twins", 20011, 0, 20011, 0), ("giant", 33333, 5, 33000, 0),
    ("giant", 70000, 0, 70000, 2),
])
@pytest.mark.parametrize("length", [1.0, 1e-30, 1e25])
def test_against_oracle(grav, kind, n, ibeg, ni, nk, length):
    if kind == "bigH":
        d = _set("plummer", n)
        d["range2"][::7] = 4.0e4
    else:
        d = _set(kind, n)
    x, y, z, r2 = d["x"] * length, d["y"] * length, d["z"] * length, d["range2"] * length ** 2
    psi = grav.psi(x, y, z, d["m"], r2, nkernel=nk, ibeg=ibeg, ni=ni)
    rows = np.unique(np.concatenate([np.random.default_rng(2).choice(ni, min(ni, 150), replace=False),
                                     [0, ni - 1]]))
    ref = oracle.psi(d["x"], d["y"], d["z"], d["m"], d["range2"], nkernel=nk, rows=rows + ibeg)
    gas = d["range2"][rows + ibeg] > 0
    assert np.all(psi[rows][~gas] == 0.0)
    got = psi[rows][gas] * length ** 2
    assert np.max(np.abs(got - ref[gas]) / np.abs(ref[gas])) <= 1e-11


@pytest.mark.parametrize("nk", [0, 2])
@pytest.mark.parametrize("H", [1e-5, 1e-7, 1e-8])
def test_supports_of_the_size_of_fp32_rounding(grav, H, nk):
    """Tight clumps of 64 + 32 particles, 0.6 H apart, all over a set 1e5 to 1e8
    times larger than H: chunks that straddle two clumps test boxes whose FP32
    corners, relative to the group's origin, are off by more than H."""
    rng = np.random.default_rng(0)
    pos = []
    for c in rng.uniform(-1.0, 1.0, (60, 3)):
        d = rng.normal(size=3)
        d *= 0.6 * H / np.linalg.norm(d)
        pos += [c + 0.01 * H * rng.normal(size=(64, 3)), c + d + 0.01 * H * rng.normal(size=(32, 3))]
    pos = np.concatenate(pos)
    n = len(pos)
    args = [*(p.copy() for p in pos.T), rng.uniform(0.5, 1.5, n) / n, np.full(n, H * H)]
    want = oracle.psi(*args, nkernel=nk)
    # positions relative to the group's origin are off by 2^-53 of the distance to it
    tol = 1e-11 + 8.0 * 2.0 ** -53 / H
    np.testing.assert_allclose(grav.psi(*args, nkernel=nk), want, rtol=tol, atol=0)
