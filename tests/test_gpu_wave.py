"""The wave-sized work items of small i-ranges (k_pair_wave), against the
oracle and against the block kernel (an explicit j-split asks for it).

Bounds as in the other parity tests of the FP32C pass: 1e-5 on the
acceleration, 1e-6 on the potential; where a few particles' pair terms cancel
(a handful of coincident ones) relative to the set's rms.
"""
import numpy as np
import pytest

import oracle
from starsmasher_amd import SG_PREC_FP32C, Gravity, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _set(n, hscale=1.0):
    rng = np.random.default_rng(n)
    pos = rng.normal(size=(n, 3))
    if n > 20:   # a coincident pair, a coincident triple with a point particle
        pos[7] = pos[3]
        pos[11] = pos[12] = pos[13]
    m = rng.uniform(0.1, 1.0, n) / n
    h = hscale * rng.uniform(0.5, 1.5, n) * (64.0 / n) ** (1.0 / 3.0)
    r2 = h * h
    if n > 20:
        r2[[5, 12]] *= -1.0
    return pos[:, 0].copy(), pos[:, 1].copy(), pos[:, 2].copy(), m, r2


def _check(res, ref, what):
    acc, racc = np.stack(res[:3], -1), np.stack(ref[:3], -1)
    norm = np.maximum(np.linalg.norm(racc, axis=1), 0.1 * np.sqrt(np.mean(racc ** 2)) + 1e-300)
    ea = np.linalg.norm(acc - racc, axis=1) / norm
    ep = np.abs(res[3] - ref[3]) / np.maximum(np.abs(ref[3]), 1e-300)
    print(f"[{what}] acc {ea.max():.2e} pot {ep.max():.2e}")
    assert ea.max() < 1e-5 and ep.max() < 1e-6, what


# one to two i chunks; 5,760 / 5,888: 8,190 and 8,464 visits, each in four
# parts up to 8,192; 16,385: 257 i chunks
@pytest.mark.parametrize("n,nk", [(1, 0), (2, 1), (63, 0), (64, 1), (65, 2), (128, 0), (257, 1),
                                  (1000, 2), (5760, 0), (5888, 1), (16385, 0)])
def test_sizes(grav, n, nk):
    args = _set(n)
    res = grav.compute(*args, nkernel=nk)
    _check(res, oracle.direct(*args, nkernel=nk), f"n {n} nk {nk}")
    for a, b in zip(res, grav.compute(*args, nkernel=nk)):
        np.testing.assert_array_equal(a, b)


# few softened pairs a visit, lists of all lengths, and more than the list
# holds (every pair softened)
@pytest.mark.parametrize("nk", [0, 1, 2])
@pytest.mark.parametrize("hscale", [0.05, 0.6, 1.7, 30.0])
def test_softened_shares(grav, hscale, nk):
    args = _set(1500, hscale)
    res = grav.compute(*args, nkernel=nk)
    fp64 = grav.last_precision_stats()[3]
    _check(res, oracle.direct(*args, nkernel=nk), f"H x {hscale} nk {nk}")
    pos = np.stack(args[:3], 1)
    r2 = ((pos[:, None] - pos[None]) ** 2).sum(-1)
    want = int((r2 < np.maximum(np.abs(args[4])[:, None], np.abs(args[4])[None])).sum())
    assert abs(fp64 - want) <= 1e-3 * want


@pytest.mark.parametrize("n,ibeg,ni", [(3000, 0, 1), (3000, 2999, 1), (3000, 1234, 65),
                                       (40000, 12345, 6789), (120000, 60001, 49151)])
def test_partial_ranges(grav, n, ibeg, ni):
    d = ics.plummer(n, seed=n)
    args = (d["x"], d["y"], d["z"], d["m"], d["range2"])
    res = grav.compute(*args, nkernel=2, ibeg=ibeg, ni=ni)
    rows = np.unique(np.linspace(ibeg, ibeg + ni - 1, min(ni, 300)).astype(int))
    ref = oracle.direct(*args, nkernel=2, rows=rows)
    _check([r[rows - ibeg] for r in res], ref, f"{ni} of {n}")
    old = grav.get_config(SG_PREC_FP32C)
    grav.set_config(SG_PREC_FP32C, 128, 1, 3)
    try:
        block = grav.compute(*args, nkernel=2, ibeg=ibeg, ni=ni)
    finally:
        grav.set_config(SG_PREC_FP32C, *old)
    _check(res, block, f"{ni} of {n} against the block kernel")
