"""The FP32C adjoint over its two forms: one wave per 64 particles (below
32,768) and each unordered far pair once, against the FP64 pass on all particles and
against the oracle on rows, which shares no preparation, order or gather with either.

Bounds as in test_gpu_adjoint.py: the largest difference over the rms of the gradient
at most 1e-5 (the FP32 rounding of pair terms that cancel under random cotangents).
"""
import numpy as np
import pytest

import oracle
from starsmasher_amd import SG_PREC_FP32C, SG_PREC_FP64, Gravity, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _set(n, kind):
    rng = np.random.default_rng(n)
    if kind == "two":
        d = ics.two_polytropes(n, seed=n)
    elif kind == "giant":
        d = ics.giant_with_core(n, seed=n)
    else:
        d = ics.plummer(n, seed=n)
    args = [d[k].copy() for k in ("x", "y", "z", "m", "range2")]
    if n > 100:   # coincident pairs, point particles
        for k in range(3):
            args[k][7] = args[k][3]
            args[k][n - 1] = args[k][n - 2]
        args[4][[5, n // 2]] *= -1.0
    if kind == "bigH":
        args[4][rng.choice(n, 5, replace=False)] = 4.0e4
    cot = [rng.normal(size=n).astype(np.float32).astype(np.float64) for _ in range(4)]
    return args, cot


# 1 .. 257: one to five i chunks; 32,767 / 32,768 / 32,769: the two forms'
# border and a last chunk of one; 65,793: a superblock of one tile at the end
@pytest.mark.parametrize("n,kind,nk", [(1, "cloud", 0), (64, "cloud", 1), (65, "cloud", 2),
                                       (257, "cloud", 0), (3000, "bigH", 1), (5000, "two", 0),
                                       (32767, "cloud", 0), (32768, "giant", 1), (32769, "two", 2),
                                       (40000, "bigH", 0), (65793, "cloud", 1)])
def test_against_fp64_and_oracle(grav, n, kind, nk):
    args, cot = _set(n, kind)
    res = grav.vjp(*args, *cot, nkernel=nk, precision=SG_PREC_FP32C)
    for a, b in zip(res, grav.vjp(*args, *cot, nkernel=nk, precision=SG_PREC_FP32C)):
        np.testing.assert_array_equal(a, b)
    ref = grav.vjp(*args, *cot, nkernel=nk, precision=SG_PREC_FP64)
    for name, a, b in zip(("x", "y", "z", "m", "H"), res, ref):
        rms = np.sqrt(np.mean(b ** 2))
        err = np.abs(a - b)
        print(f"[{kind} {n} nk {nk}] {name}: median {np.median(err) / max(rms, 1e-300):.2e} "
              f"max {err.max() / max(rms, 1e-300):.2e}")
        assert err.max() <= 1e-5 * rms + 1e-300
    # first, last, coincident and point particles, the largest supports, and others
    rows = np.unique(np.concatenate([
        np.random.default_rng(1).choice(n, min(n, 100), replace=False), [0, n - 1],
        np.argsort(-np.abs(args[4]))[:6], np.flatnonzero(args[4] < 0), [3, 7, n - 2] if n > 100 else []]))
    rows = rows.astype(int)
    exact = oracle.vjp(*args, np.stack(cot[:3], 1), cot[3], nkernel=nk, rows=rows)
    for a, b, whole in zip(res, exact, ref):
        assert np.abs(a[rows] - b).max() <= 1e-5 * np.sqrt(np.mean(whole ** 2)) + 1e-300


@pytest.mark.parametrize("length,mass", [(1.0e11, 1.0e24), (1.0e-8, 1.0e-18)])
def test_units(grav, length, mass):
    """Another system of units: r^-5 by itself leaves the FP32 range (the near
    pairs, unscaled, need r^-3 within it)."""
    args, cot = _set(40000, "cloud")
    base = grav.vjp(*args, *cot)
    u = cot[3] * length ** -1.0
    scaled = [args[0] * length, args[1] * length, args[2] * length, args[3] * mass,
              args[4] * length ** 2]
    res = grav.vjp(*scaled, *cot[:3], u)
    units = [mass / length ** 3] * 3 + [1.0 / length ** 2] + [mass / length ** 3]
    for a, b, f in zip(res, base, units):
        rms = np.sqrt(np.mean(b ** 2))
        assert np.abs(a / f - b).max() <= 1e-5 * rms
