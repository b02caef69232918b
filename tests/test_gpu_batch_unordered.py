"""Batches that evaluate each unordered far pair once (the default batch shape,
both precisions), against the oracle and against the ordered batch kernel, which other
shapes still run.

Bounds: the library's stated FP32C errors (1e-5 on the acceleration, 1e-6 on
the potential); both passes round each pair to FP32 and sum pairs in FP32 (32 in
sequence, or 16 and a tree over the lanes), so they differ by no more than twice that.  FP64: 1e-11 and 1e-12, as in the
other parity tests.
"""
import numpy as np
import pytest

import oracle
from conftest import rel_errors
from starsmasher_amd import SG_PREC_FP32C, SG_PREC_FP64, Gravity, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grav():
    g = Gravity(0)
    yield g
    g.close()


def _scaled(d, length, mass):
    e = dict(d)
    for k in ("x", "y", "z"):
        e[k] = d[k] * length
    e["m"] = d["m"] * mass
    e["range2"] = d["range2"] * length * length
    return e


def _check(grav, sets, nk, prec=SG_PREC_FP32C):
    amax, pmax = (1e-5, 1e-6) if prec == SG_PREC_FP32C else (1e-11, 1e-12)
    eager = grav.compute_batch(sets, nkernel=nk, precision=prec)
    for _ in range(2):   # capture, then replay
        for r, g in zip(eager, grav.compute_batch(sets, nkernel=nk, precision=prec, use_graph=True)):
            for a, b in zip(r, g):
                np.testing.assert_array_equal(a, b)
    old = grav.get_batch_config(prec)
    grav.set_batch_config(prec, 128, 1)
    try:
        ordered = grav.compute_batch(sets, nkernel=nk, precision=prec)
    finally:
        grav.set_batch_config(prec, *old)
    rng = np.random.default_rng(4)
    for k, (d, r, o) in enumerate(zip(sets, eager, ordered)):
        n = d["x"].size
        rows = np.unique(np.concatenate([rng.choice(n, min(n, 200), replace=False), [0, n - 1]]))
        ref = oracle.direct(d["x"], d["y"], d["z"], d["m"], d["range2"], nkernel=nk, rows=rows)
        if n > 1:
            ea, ep = rel_errors(np.stack(r[:3], -1)[rows], r[3][rows], np.stack(ref[:3], -1), ref[3])
            assert ea.max() <= amax and ep.max() <= pmax, (k, n, ea.max(), ep.max())
            ea, ep = rel_errors(np.stack(r[:3], -1), r[3], np.stack(o[:3], -1), o[3])
            assert ea.max() <= 2 * amax and ep.max() <= 2 * pmax, (k, n, ea.max(), ep.max())
        else:
            np.testing.assert_allclose(r[3], ref[3], rtol=1e-12)


# 255 and 256: the two sides of the rule on the mean set; sets of one particle,
# of a tile and one more, of a superblock (1,024) and one more, of more than
# 64 chunks (two words of bits); the largest last, first and alone; 320 chunks
# and superblocks of 32 in a batch of 40 x 20,480
@pytest.mark.parametrize("prec", [SG_PREC_FP32C, SG_PREC_FP64])
@pytest.mark.parametrize("sizes,nk", [
    ([255] * 5, 0), ([256] * 5, 1),
    ([1, 1024, 1025, 257, 1, 4097, 70001], 0),
    ([16385, 3, 2048, 12289], 2),
    ([33333], 1),
    ([20480] * 39 + [20481], 0),
])
def test_sizes(grav, sizes, nk, prec):
    _check(grav, [ics.plummer(int(n), seed=17 * k + n) for k, n in enumerate(sizes)], nk,
           prec)


def test_each_set_in_its_own_units(grav):
    """Lengths and masses that differ by 1e16 and 1e20 between the sets of a
    batch, one set far from the origin: scales and boxes are the set's own."""
    base = [ics.plummer(n, seed=n) for n in (5000, 6000, 7000, 8000)]
    sets = [_scaled(base[0], 1e-8, 1e-10), _scaled(base[1], 1e8, 1e10), base[2], dict(base[3])]
    sets[3]["x"] = sets[3]["x"] + 1e3
    _check(grav, sets, 0)


def test_changed_sizes_replan(grav):
    """The captured graph is not replayed for other offsets."""
    for sizes in ([3000, 5000], [5000, 3000], [8000], [3000, 5000]):
        _check(grav, [ics.plummer(n, seed=n) for n in sizes], 0)


def _visits(grav, sizes, prec):
    grav.compute_batch([ics.plummer(n, seed=n) for n in sizes], precision=prec)
    return grav.last_tile_stats()[0]


def test_chunks_of_padding_are_not_visited(grav):
    """A set fills its last tile of 256 with padding; the visits are those of the
    chunks with particles, each pair of them in both orders."""
    sizes = [300, 700, 70, 513, 256, 3, 2500]
    assert _visits(grav, sizes, SG_PREC_FP32C) == sum((-(-n // 64)) ** 2 for n in sizes)


def test_fp64_batches_of_small_sets_run_the_ordered_kernel(grav):
    """The ordered kernel visits by tiles; in FP64 it is the shorter one up to a
    mean set of 2,560."""
    for n, unordered in ((300, False), (2449, False), (3001, True)):
        assert (_visits(grav, [n] * 8, SG_PREC_FP64) == 8 * (-(-n // 64)) ** 2) == unordered
        assert _visits(grav, [n] * 8, SG_PREC_FP32C) == 8 * (-(-n // 64)) ** 2
