"""What runs where the device memory of the unordered passes is not to be had: the
ordered kernels, bit for bit those an explicit configuration asks for, in the same
context as before and after."""
import numpy as np
import pytest

from starsmasher_amd import SG_PREC_FP32C, SG_PREC_FP64, Gravity, ics

pytestmark = pytest.mark.gpu
N = 50001


def _args(d):
    return [d[k] for k in ("x", "y", "z", "m", "range2")]


@pytest.fixture
def limited():
    """A context that has run the unordered pass and then lost its memory."""
    with Gravity(0) as g, Gravity(0) as other:
        yield g, other


@pytest.mark.parametrize("prec", [SG_PREC_FP32C, SG_PREC_FP64])
@pytest.mark.parametrize("psi", [False, True])
def test_whole_set(limited, prec, psi):
    g, other = limited
    d = _args(ics.two_polytropes(N, seed=3))
    run = lambda c: (c.compute_psi if psi else c.compute)(*d, nkernel=2, precision=prec)
    first = run(g)
    slabs = g.last_config()[2]
    g.set_scratch_limit(0)
    second = run(g)
    wg, ipl, js = g.last_config()
    assert js != slabs
    other.set_config(prec, wg, ipl, js)
    for a, b in zip(second, run(other)):
        np.testing.assert_array_equal(a, b)
    g.set_scratch_limit()
    for a, b in zip(first, run(g)):
        np.testing.assert_array_equal(a, b)


def test_gradient(limited):
    g, other = limited
    d = _args(ics.plummer(N, seed=4))
    rng = np.random.default_rng(0)
    cot = [rng.normal(size=N) for _ in range(4)]
    first = g.vjp(*d, *cot)
    g.set_scratch_limit(1 << 20)
    second = g.vjp(*d, *cot)
    other.set_config(SG_PREC_FP32C, 256, 1, 0)
    for a, b in zip(second, other.vjp(*d, *cot)):
        np.testing.assert_array_equal(a, b)
    g.set_scratch_limit()
    for a, b, c in zip(first, g.vjp(*d, *cot), second):
        np.testing.assert_array_equal(a, b)
        # two FP32C forms: the bound of either against FP64, twice
        assert np.abs(a - c).max() <= 2e-5 * np.sqrt(np.mean(c ** 2))


@pytest.mark.parametrize("prec,acc,pot", [(SG_PREC_FP32C, 1e-5, 1e-6), (SG_PREC_FP64, 1e-11, 1e-12)])
def test_batch_graph(limited, prec, acc, pot):
    """The captured graph follows the limit both ways."""
    g, _ = limited
    sets = [ics.plummer(n, seed=n) for n in (5000, 300, 9000, 20001)]
    run = lambda graph: g.compute_batch(sets, precision=prec, use_graph=graph)
    first = run(True)
    for limit in (0, None, 0):
        g.set_scratch_limit(limit)
        for graph in (True, True, False, True):
            for r, q in zip(run(graph), first):
                a, b = np.stack(r[:3], 1), np.stack(q[:3], 1)
                ea = np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
                assert ea.max() <= 2 * acc and (np.abs(r[3] / q[3] - 1.0)).max() <= 2 * pot
                if limit is None:
                    np.testing.assert_array_equal(a, b)
