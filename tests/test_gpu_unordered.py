"""The whole-set FP32C pass that evaluates each unordered far pair once
(sg_sym.hip), against the oracle and against the ordered pass.

A context takes it at its automatic configuration from 49,152 particles on;
an explicit j-split asks for the ordered pass.  Bounds: the library's stated
FP32C errors (1e-5 on the acceleration, 1e-6 on the potential, as in the other
parity tests); both passes round each pair to FP32 and sum pairs in FP32 (the
ordered one 32 in sequence; this one 16 and a tree over 16 lanes for a row, 16 and a tree
over four for a column), so they differ from each other by no more than twice that.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_errors
from starsmasher_amd import SG_PREC_FP32C, Gravity, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _set(kind, n):
    if kind == "giant":
        return ics.giant_with_core(n, seed=n)
    if kind == "two":
        return ics.two_polytropes(n, seed=n)
    d = ics.plummer(n, seed=n)
    if kind == "bigH":   # particles whose support holds the whole set
        d["range2"][np.random.default_rng(n).choice(n, 9, replace=False)] = 4.0e4
    if kind == "twins":  # coincident pairs and point particles
        for k in ("x", "y", "z"):
            d[k][1::997] = d[k][0:-1:997][:d[k][1::997].size]
        d["range2"][5::1009] *= -1.0
    return d


# 49,152 is the smallest set of the pass and 49,151 the largest before it;
# 49,153 and 65,537 end in a chunk of one particle, 69,889 and 131,073 leave
# a superblock of one tile behind whole ones; up to 65,536 particles a
# workgroup has two waves, then four
@pytest.mark.parametrize("kind,n,nk", [
    ("plummer", 49151, 0), ("plummer", 49152, 0), ("two", 49153, 1), ("giant", 50000, 2),
    ("bigH", 65537, 0), ("twins", 69889, 1), ("two", 100003, 2), ("giant", 131073, 0),
])
def test_against_oracle_and_ordered_pass(grav, kind, n, nk):
    d = _set(kind, n)
    args = (d["x"], d["y"], d["z"], d["m"], d["range2"])
    res = grav.compute(*args, nkernel=nk)
    visits, nearv, widev, fp64 = grav.last_precision_stats()
    again = grav.compute(*args, nkernel=nk)
    for a, b in zip(res, again):
        np.testing.assert_array_equal(a, b)     # fixed order of every sum
    chunks = -(-n // 256) * 4
    assert 0 < nearv + widev < visits and fp64 >= n - (d["range2"] < 0).sum()
    if n >= 49152:
        assert visits == chunks ** 2            # every chunk pair, each order once
    old = grav.get_config(SG_PREC_FP32C)
    grav.set_config(SG_PREC_FP32C, 256, 1, 7)
    try:
        other = grav.compute(*args, nkernel=nk)
    finally:
        grav.set_config(SG_PREC_FP32C, *old)
    acc, ref = np.stack(res[:3], -1), np.stack(other[:3], -1)
    ea, ep = rel_errors(acc, res[3], ref, other[3])
    print(f"[{kind} {n}] against the ordered pass: acc {ea.max():.2e} {np.median(ea):.2e} "
          f"pot {ep.max():.2e}")
    assert ea.max() < 2e-5 and np.median(ea) < 2e-7 and ep.max() < 2e-6
    rng = np.random.default_rng(n)
    rows = np.unique(np.concatenate([rng.choice(n, 150, replace=False), [0, n - 1],
                                     np.argsort(ea)[-20:],
                                     np.argsort(np.abs(d["range2"]))[-9:]]))
    o = oracle.direct(*args, nkernel=nk, rows=rows)
    ea, ep = rel_errors(acc[rows], res[3][rows], np.stack(o[:3], -1), o[3])
    print(f"[{kind} {n}] against the oracle: acc {ea.max():.2e} {np.median(ea):.2e} pot {ep.max():.2e}")
    assert ea.max() < 1e-5 and ep.max() < 1e-6


def test_particles_on_a_line(grav):
    """All chunks of a set on one axis: boxes of zero width, no far chunk
    rejected by two of the three axes."""
    n = 50000
    rng = np.random.default_rng(8)
    x = np.sort(rng.uniform(-50.0, 50.0, n))
    z = np.zeros(n)
    m = rng.uniform(0.5, 2.0, n)
    r2 = np.full(n, 1e-4)
    res = grav.compute(x, z, z, m, r2)
    rows = rng.choice(n, 100, replace=False)
    o = oracle.direct(x, z, z, m, r2, nkernel=0, rows=rows)
    scale = np.sqrt(np.mean(o[0] ** 2))
    assert np.abs(res[0][rows] - o[0]).max() < 1e-5 * scale
    assert np.abs(res[1]).max() == 0.0 and np.abs(res[2]).max() == 0.0
    assert (np.abs(res[3][rows] - o[3]) / np.abs(o[3])).max() < 1e-6


@pytest.mark.parametrize("length,mass", [(1.0e13, 1.0e30), (1.0e-13, 1.0e-20)])
def test_units(grav, length, mass):
    """The same set in other units (metres and kilograms of a wide system, and
    the reverse): r^-3 by itself leaves the FP32 range, the result scales
    exactly up to FP32 rounding of the scaled inputs."""
    d = _set("plummer", 50000)
    base = grav.compute(d["x"], d["y"], d["z"], d["m"], d["range2"])
    res = grav.compute(d["x"] * length, d["y"] * length, d["z"] * length, d["m"] * mass,
                       d["range2"] * length ** 2)
    back = [r / (mass / length ** 2) for r in res[:3]]
    ea, ep = rel_errors(np.stack(back, -1), res[3] / (mass / length), np.stack(base[:3], -1), base[3])
    print(f"[units {length:g} {mass:g}] acc {ea.max():.2e} pot {ep.max():.2e}")
    assert ea.max() < 1e-5 and ep.max() < 1e-6
