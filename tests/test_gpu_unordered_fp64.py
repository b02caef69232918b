"""The whole-set FP64 pass that evaluates each unordered far pair once
(sg_sym64.hip), against the oracle and against the ordered pass.

A context takes it at its automatic configuration from 32,769 particles on; an
explicit j-split asks for the ordered pass.  Bounds: the FP64 errors of the other
parity tests (1e-11 on the acceleration, 1e-12 on the potential); the two passes
differ by no more than twice that.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_errors
from starsmasher_amd import SG_PREC_FP64, Gravity, ics
from test_gpu_unordered import _set

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


# 32,768 and 32,769: the two sides of the rule; 32,769 and 65,537 end in a chunk
# of one particle; from 65,537 on a superblock has two column groups, from
# 131,073 three; 69,889 leaves one tile behind whole superblocks
@pytest.mark.parametrize("kind,n,nk", [
    ("plummer", 32768, 0), ("two", 32769, 1), ("plummer", 34000, 2), ("bigH", 40011, 0),
    ("giant", 65536, 0), ("twins", 65537, 1), ("two", 69889, 2), ("plummer", 131073, 0),
])
def test_against_oracle_and_ordered_pass(grav, kind, n, nk):
    d = _set(kind, n)
    args = (d["x"], d["y"], d["z"], d["m"], d["range2"])
    res = grav.compute(*args, nkernel=nk, precision=SG_PREC_FP64)
    visits, nearv, widev, fp64 = grav.last_precision_stats()
    again = grav.compute(*args, nkernel=nk, precision=SG_PREC_FP64)
    for a, b in zip(res, again):
        np.testing.assert_array_equal(a, b)     # fixed order of every sum
    chunks = -(-n // 256) * 4
    assert 0 < nearv < visits and widev == 0 and fp64 == 0
    if n >= 32769:
        assert visits == chunks * chunks
    rng = np.random.default_rng(1)
    rows = np.unique(np.concatenate([rng.choice(n, 200, replace=False), [0, n - 1]]))
    ref = oracle.direct(*args, nkernel=nk, rows=rows)
    ea, ep = rel_errors(np.stack(res[:3], -1)[rows], res[3][rows], np.stack(ref[:3], -1), ref[3])
    assert ea.max() <= 1e-11 and ep.max() <= 1e-12, (ea.max(), ep.max())
    old = grav.get_config(SG_PREC_FP64)
    grav.set_config(SG_PREC_FP64, 256, 1, 3)
    try:
        ordered = grav.compute(*args, nkernel=nk, precision=SG_PREC_FP64)
    finally:
        grav.set_config(SG_PREC_FP64, *old)
    ea, ep = rel_errors(np.stack(res[:3], -1), res[3], np.stack(ordered[:3], -1), ordered[3])
    assert ea.max() <= 2e-11 and ep.max() <= 2e-12, (ea.max(), ep.max())


@pytest.mark.parametrize("length,mass", [(1e11, 1e33), (1e-60, 1e-30)])
def test_units(grav, length, mass):
    """r^-3 of FP64 pairs in units far from one."""
    d = ics.plummer(33000, seed=3)
    g = grav.compute(d["x"], d["y"], d["z"], d["m"], d["range2"], precision=SG_PREC_FP64)
    s = grav.compute(d["x"] * length, d["y"] * length, d["z"] * length, d["m"] * mass,
                     d["range2"] * length ** 2, precision=SG_PREC_FP64)
    ea, ep = rel_errors(np.stack(s[:3], -1) * (length ** 2 / mass), s[3] * (length / mass),
                        np.stack(g[:3], -1), g[3])
    assert ea.max() <= 2e-11 and ep.max() <= 2e-12
