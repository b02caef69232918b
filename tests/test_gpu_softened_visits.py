"""Chunk visits with many softened pairs, in FP64, with the grad-h term and in the
gradient.  After a visit with more than half of its pairs softened the next one of an
FP64 pass or a gradient is evaluated pair by pair, so the sets mix dense clumps, of more
and of less than a chunk, with particles that soften nothing.

Bounds as in test_gpu_instantiations.py: FP64 1e-11 (acceleration) and 1e-12
(potential), grad-h term 1e-11, gradient 1e-5 in FP32C of the rms; accelerations that
cancel relative to the set's rms.
"""
import numpy as np
import pytest

import oracle
from starsmasher_amd import SG_PREC_FP32C, SG_PREC_FP64, Gravity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _set(n, clump, hscale, seed=1):
    """Clumps of `clump` particles softened among themselves (all of the set where
    hscale is large), the others with supports that hold nobody."""
    rng = np.random.default_rng(seed)
    pos = rng.normal(size=(n, 3))
    k = n // (2 * clump)
    centre = rng.normal(size=(k, 3))
    pos[: k * clump] = np.repeat(centre, clump, 0) + 1e-2 * rng.normal(size=(k * clump, 3))
    h = np.full(n, 1e-3)
    h[: k * clump] = hscale * 1e-2 * rng.uniform(1.0, 4.0, k * clump)
    if n > 100:
        pos[7] = pos[3]                  # coincident
        pos[n - 1] = pos[n - 2]
    r2 = h * h
    if n > 100:
        r2[[5, n // 2]] *= -1.0          # point particles
    mix = rng.permutation(n)
    m = rng.uniform(0.1, 1.0, n) / n
    return [a[mix].copy() for a in (*pos.T, m, r2)]


def _rows(n, args):
    rng = np.random.default_rng(n)
    big = np.argsort(-np.abs(args[4]))[:60]
    return np.unique(np.concatenate([rng.choice(n, min(n, 150), replace=False), big,
                                     np.flatnonzero(args[4] < 0), [0, n - 1]]))


def _check(res, ref, rows, acc, pot):
    a, r = np.stack(res[:3], 1)[rows], np.stack(ref[:3], 1)
    scale = np.maximum(np.linalg.norm(r, axis=1), 0.1 * np.sqrt((r ** 2).sum(1).mean()))
    assert (np.linalg.norm(a - r, axis=1) / scale).max() <= acc
    assert (np.abs(res[3][rows] - ref[3]) / np.abs(ref[3])).max() <= pot


# clumps of 40, 64 and 200 particles; supports of a clump, of some and of the
# whole set; 33,000: the whole-set pass (FP64 from 32,769 on), 4,096 and below the
# visits of 16 columns
@pytest.mark.parametrize("nk", [0, 1, 2])
@pytest.mark.parametrize("n,clump,hscale", [(700, 40, 1.0), (4096, 64, 1.0), (9000, 200, 100.0),
                                            (33000, 200, 1.0), (33000, 64, 600.0)])
def test_dense_and_sparse_visits(grav, n, clump, hscale, nk):
    args = _set(n, clump, hscale)
    rows = _rows(n, args)
    ref = oracle.direct(*args, nkernel=nk, rows=rows)
    psi = oracle.psi(*args, nkernel=nk, rows=rows)
    gas = psi != 0.0
    for prec, acc, pot in ((SG_PREC_FP64, 1e-11, 1e-12), (SG_PREC_FP32C, 1e-5, 1e-6)):
        plain = grav.compute(*args, nkernel=nk, precision=prec)
        res = grav.compute_psi(*args, nkernel=nk, precision=prec)
        _check(res, ref, rows, acc, pot)
        if prec == SG_PREC_FP32C or n > 32768:   # one pass for both: the same forces
            for a, b in zip(plain, res):
                np.testing.assert_array_equal(a, b)
        _check(plain, ref, rows, acc, pot)
        got = res[4][rows]
        assert np.abs(got[gas] / psi[gas] - 1.0).max() <= 1e-11 and np.all(got[~gas] == 0.0)
        again = grav.compute_psi(*args, nkernel=nk, precision=prec)
        for a, b in zip(res, again):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nk", [0, 1, 2])
@pytest.mark.parametrize("n,clump,hscale", [(700, 40, 1.0), (9000, 200, 100.0), (33000, 64, 600.0)])
def test_gradient(grav, n, clump, hscale, nk):
    args = _set(n, clump, hscale)
    rng = np.random.default_rng(n)
    cot = [rng.normal(size=n).astype(np.float32).astype(np.float64) for _ in range(4)]
    rows = _rows(n, args)
    res = grav.vjp(*args, *cot, nkernel=nk, precision=SG_PREC_FP32C)
    ref = oracle.vjp(*args, np.stack(cot[:3], 1), cot[3], nkernel=nk, rows=rows)
    for a, b in zip(res, ref):
        assert np.abs(a[rows] - b).max() <= 1e-5 * np.sqrt(np.mean(b ** 2))
    for a, b in zip(res, grav.vjp(*args, *cot, nkernel=nk, precision=SG_PREC_FP32C)):
        np.testing.assert_array_equal(a, b)
