"""The grad-h term formed by the unordered whole-set pass: all its pairs are in
the visits left to the ordered rest kernel.

Against the pass without the term (the same forces, bit for bit), the term of
the ordered pass, the term alone, and oracle rows.  The term's pairs are FP64 in
every pass; only the order of the sums differs (1e-11 relative, as in the other
tests of the term).
"""
import numpy as np
import pytest

import oracle
from starsmasher_amd import SG_PREC_FP32C, SG_PREC_FP64, Gravity
from test_gpu_unordered import _set

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


# the smallest set of either precision's pass and one particle fewer, coincident
# pairs and point particles, supports that hold the whole set
@pytest.mark.parametrize("kind,n,nk,prec", [
    ("plummer", 49151, 0, SG_PREC_FP32C), ("giant", 49152, 0, SG_PREC_FP32C),
    ("twins", 65537, 1, SG_PREC_FP32C), ("bigH", 50001, 2, SG_PREC_FP32C),
    ("plummer", 32768, 1, SG_PREC_FP64), ("bigH", 32769, 0, SG_PREC_FP64),
    ("twins", 40001, 2, SG_PREC_FP64),
])
def test_grad_h_term(grav, kind, n, nk, prec):
    d = _set(kind, n)
    args = (d["x"], d["y"], d["z"], d["m"], d["range2"])
    plain = grav.compute(*args, nkernel=nk, precision=prec)
    *force, psi = grav.compute_psi(*args, nkernel=nk, precision=prec)
    for a, b in zip(plain, force):
        np.testing.assert_array_equal(a, b)
    old = grav.get_config(prec)
    grav.set_config(prec, 256, 1, 3)
    try:
        ordered = grav.compute_psi(*args, nkernel=nk, precision=prec)[4]
    finally:
        grav.set_config(prec, *old)
    np.testing.assert_allclose(psi, ordered, rtol=1e-11, atol=0)
    np.testing.assert_allclose(psi, grav.psi(*args, nkernel=nk), rtol=1e-11, atol=0)
    assert np.all(psi[d["range2"] < 0] == 0.0)
    rows = np.unique(np.concatenate([np.random.default_rng(1).choice(n, 150, replace=False),
                                     [0, n - 1]]))
    ref = oracle.psi(*args, nkernel=nk, rows=rows)
    gas = d["range2"][rows] > 0
    assert np.max(np.abs(psi[rows][gas] - ref[gas]) / np.abs(ref[gas])) <= 1e-11
