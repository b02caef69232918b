"""Sets much wider than the distances within them: two stars between two particles
so far away that the distances between the stars, in units of the set's extent, leave the
FP32 range in r^-3 (forces) or r^-4 (gradients).

The stars come one after the other in the arrays: all of them lie in one cell of
the space-filling curve, which then keeps the input order.  Sizes leave more than 33
particles in the last chunk: its origin is then one of the stars'.  Bounds as in
test_gpu_unordered.py and test_gpu_adjoint_sizes.py.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_errors
from starsmasher_amd import SG_PREC_FP32C, SG_PREC_FP64, Gravity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _set(n, far):
    rng = np.random.default_rng(n)
    pos = 0.1 * rng.normal(size=(n, 3))
    pos[n // 2:, 0] += 3.0
    pos[-1] = (0.3 * far, far, -0.2 * far)
    pos[0] = -pos[-1]
    h = np.full(n, 0.6 * n ** (-1.0 / 3.0))
    return [c.copy() for c in pos.T] + [rng.uniform(0.5, 1.5, n) / n, h * h]


def _rows(n):
    return np.unique(np.random.default_rng(2).choice(np.arange(1, n - 1), 150, replace=False))


def _check(res, args):
    rows = _rows(args[0].size)      # the far particles' forces are zero to rounding
    ref = oracle.direct(*args, rows=rows)
    ea, ep = rel_errors(np.stack(res[:3], -1)[rows], res[3][rows], np.stack(ref[:3], -1), ref[3])
    print(f"[wide {args[0].size}] acc {ea.max():.2e} pot {ep.max():.2e}")
    assert ea.max() <= 1e-5 and ep.max() <= 1e-6
    assert all(np.isfinite(r).all() for r in res)


@pytest.mark.parametrize("far", [1e4, 1e8, 1e14, 1e17])
def test_forces(grav, far):
    args = _set(50040, far)
    _check(grav.compute(*args), args)


@pytest.mark.parametrize("far", [1e8, 1e14, 1e17])
def test_batch(grav, far):
    sets = [_set(n, far) for n in (3000, 20090)]
    names = ("x", "y", "z", "m", "range2")
    for args, res in zip(sets, grav.compute_batch([dict(zip(names, a)) for a in sets])):
        _check(res, args)


@pytest.mark.parametrize("far", [1e4, 1e8, 1e11, 1e14])
def test_gradient(grav, far):
    n = 33001
    args = _set(n, far)
    rng = np.random.default_rng(3)
    cot = [rng.normal(size=n).astype(np.float32).astype(np.float64) for _ in range(4)]
    res = grav.vjp(*args, *cot, precision=SG_PREC_FP32C)
    rows = _rows(n)
    ref = oracle.vjp(*args, np.stack(cot[:3], 1), cot[3], rows=rows)
    for a, b in zip(res, ref):
        assert np.isfinite(a).all()
        assert np.abs(a[rows] - b).max() <= 1e-5 * np.sqrt(np.mean(b ** 2))


def test_masses_and_extents_at_the_ends_of_the_range(grav):
    """A set of coincident particles (no extent), one of extent 1e-160 and one of
    masses below the smallest normal number: finite results."""
    n = 49152
    rng = np.random.default_rng(5)
    z = np.zeros(n)
    for pos, m, h in ((np.zeros((n, 3)), 1.0 / n, 0.1), (1e-160 * rng.normal(size=(n, 3)), 1.0 / n, 0.1),
                      (rng.normal(size=(n, 3)), 1e-310, 0.1)):
        res = grav.compute(*(c.copy() for c in pos.T), z + m, z + h * h)
        assert all(np.isfinite(r).all() for r in res)


def _clumps(k, H):
    """Tight clumps of 64 + 32 particles 0.6 H apart: FP32 positions relative to an
    origin in another clump are off by up to 1e-7, more than H."""
    rng = np.random.default_rng(0)
    pos = []
    for c in rng.uniform(-1.0, 1.0, (k, 3)):
        d = rng.normal(size=3)
        d *= 0.6 * H / np.linalg.norm(d)
        pos += [c + 0.01 * H * rng.normal(size=(64, 3)), c + d + 0.01 * H * rng.normal(size=(32, 3))]
    pos = np.concatenate(pos)
    n = len(pos)
    return [*(p.copy() for p in pos.T), rng.uniform(0.5, 1.5, n) / n, np.full(n, H * H)]


# small sets run one wave per 64 particles, the larger ones the rest kernels
@pytest.mark.parametrize("k,prec", [(60, SG_PREC_FP32C), (560, SG_PREC_FP32C), (560, SG_PREC_FP64)])
@pytest.mark.parametrize("H", [1e-5, 1e-7, 1e-8])
def test_supports_of_the_size_of_fp32_rounding(grav, k, prec, H):
    args = _clumps(k, H)
    rows = np.arange(0, args[0].size, k // 20)
    ref = oracle.direct(*args, rows=rows)
    res = grav.compute(*args, precision=prec)
    ea, ep = rel_errors(np.stack(res[:3], -1)[rows], res[3][rows], np.stack(ref[:3], -1), ref[3])
    assert ea.max() <= 1e-5 and ep.max() <= 1e-6
    if prec == SG_PREC_FP32C:
        rng = np.random.default_rng(1)
        cot = [rng.normal(size=args[0].size).astype(np.float32).astype(np.float64) for _ in range(4)]
        ref = oracle.vjp(*args, np.stack(cot[:3], 1), cot[3], rows=rows)
        for a, b in zip(grav.vjp(*args, *cot), ref):
            assert np.abs(a[rows] - b).max() <= 1e-5 * np.sqrt(np.mean(b ** 2))
