"""The host code of a context when device memory runs short, on the CPU:
sg_capi.cpp linked against a device made of bookkeeping (fake_device.cpp), whose
launches are checked for the buffers they would work in."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OK, HIP = 0, 6


@pytest.fixture(scope="session")
def built(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake") / "libfake.so"
    csrc = os.path.join(ROOT, "starsmasher_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{ROOT}/include", f"-I{csrc}",
                    os.path.join(csrc, "sg_capi.cpp"),
                    os.path.join(ROOT, "tests", "fake_device.cpp"), "-o", str(so)], check=True)
    return load(str(so))


def load(path):
    # RTLD_DEEPBIND: its own hipMalloc and not that of a runtime loaded before
    L = C.CDLL(path, mode=os.RTLD_LOCAL | os.RTLD_DEEPBIND)
    L.fake_used.restype = C.c_longlong
    L.fake_ran.restype = L.fake_fault.restype = C.c_char_p
    return L


class Context:
    """Calls on a fake context.  Device arrays are any non-null address."""

    def __init__(self, lib):
        self.L, self.h = lib, C.c_void_p()
        self.reset()
        self.base = lib.fake_used()
        assert lib.sg_create(0, C.byref(self.h)) == OK

    def reset(self, budget=-1, fail=0):
        self.L.fake_reset(C.c_longlong(budget), fail)

    def state(self):
        fault = self.L.fake_fault().decode()
        assert not fault, fault
        return self.L.fake_ran().decode().split()

    def used(self):
        return self.L.fake_used() - self.base

    def compute(self, n, prec=0, psi=False, ibeg=0, ni=-1):
        a = C.c_void_p(4096)
        f = self.L.sg_compute_psi_device if psi else self.L.sg_compute_device
        return f(self.h, n, ibeg, n - ibeg if ni < 0 else ni, a, a, a, a, a, 0, prec,
                 *[a] * (5 if psi else 4))

    def vjp(self, n, prec=0):
        a = C.c_void_p(4096)
        return self.L.sg_vjp_device(self.h, n, a, a, a, a, a, 0, prec, *[a] * 9)

    def batch(self, sizes, prec=0, graph=1):
        off = (C.c_longlong * (len(sizes) + 1))(*np.concatenate([[0], np.cumsum(sizes)]).tolist())
        a = C.c_void_p(4096)
        return self.L.sg_compute_batch_device(self.h, len(sizes), off, a, a, a, a, a, 0, prec,
                                              graph, a, a, a, a)

    def host(self, call, n):
        v = np.ones(n)
        p = v.ctypes.data_as(C.c_void_p)
        if call == "compute":
            return self.L.sg_compute_host(self.h, n, 0, n, p, p, p, p, p, 0, 0, p, p, p, p)
        if call == "psi":
            return self.L.sg_psi_host(self.h, n, 0, n, p, p, p, p, p, 0, p)
        return self.L.sg_vjp_host(self.h, n, p, p, p, p, p, 0, 0, *[p] * 9)


@pytest.fixture
def ctx(built):
    c = Context(built)
    yield c
    c.reset()
    assert built.sg_destroy(c.h) == OK
    assert c.used() == 0


CALLS = {
    "compute": lambda c, n: c.compute(n),
    "part": lambda c, n: c.compute(2 * n, ibeg=n, ni=n),
    "vjp": lambda c, n: c.vjp(n),
    "host": lambda c, n: c.host("compute", n),
    "host_psi": lambda c, n: c.host("psi", n),
    "host_vjp": lambda c, n: c.host("vjp", n),
    "batch": lambda c, n: c.batch([n, 300]),
}


@pytest.mark.parametrize("call", sorted(CALLS))
def test_buffers_after_a_failed_allocation(ctx, call):
    """A call whose k-th allocation fails returns an error, and the calls after it, of
    any size, work in buffers of their own size again."""
    f = CALLS[call]
    assert f(ctx, 2000) == OK
    for k in range(1, 60):
        n = 3000 + 500 * k
        ctx.reset(fail=k)
        status = f(ctx, n)
        if ctx.L.fake_mallocs() < k:
            assert status == OK
            break
        assert status in (OK, HIP)
        ctx.reset()
        assert f(ctx, 1000) == OK and f(ctx, n - 1) == OK, k
        ctx.state()
    else:
        raise AssertionError("every allocation failed")


BIG = 1 << 20
# what runs where the device holds the slabs of each unordered far pair once,
# and where it does not
UNORDERED = {
    "compute": (lambda c: c.compute(BIG), "sym", "ordered"),
    "fp64": (lambda c: c.compute(BIG, prec=1), "sym64", "ordered"),
    "psi": (lambda c: c.compute(BIG, psi=True), "sym", "ordered"),
    "vjp": (lambda c: c.vjp(BIG), "adj_sym", "adj_ordered256"),
    "batch": (lambda c: c.batch([BIG // 2] * 4), "sym", "ordered_batch"),
    "batch64": (lambda c: c.batch([BIG // 2] * 4, prec=1), "sym64", "ordered_batch"),
}


@pytest.mark.parametrize("call", sorted(UNORDERED))
def test_a_refused_size_is_not_asked_for_again(ctx, call):
    f, unordered, ordered = UNORDERED[call]
    assert f(ctx) == OK and ctx.state() == [unordered]
    full = ctx.used()
    other = Context(ctx.L)
    other.reset(budget=ctx.L.fake_used() + full // 2)
    assert f(other) == OK and other.state() == [ordered]
    graphs = ctx.L.fake_graphs()
    for _ in range(3):   # no allocation, no wait, no other graph
        other.reset(budget=ctx.L.fake_used())
        assert f(other) == OK
        assert other.state() == ([] if graphs else [ordered])
        assert ctx.L.fake_mallocs() == ctx.L.fake_frees() == ctx.L.fake_graphs() == 0
    # a smaller set's slabs fit
    other.reset(budget=ctx.L.fake_used() + full // 2)
    assert other.compute(100000) == OK and other.state() == ["sym"]
    other.reset()
    assert ctx.L.sg_destroy(other.h) == OK


@pytest.mark.parametrize("call", sorted(UNORDERED))
def test_whatever_fits_the_ordered_pass_runs(ctx, call):
    """From the memory on that a call succeeds with, it succeeds with any more:
    slabs are taken last and never from what the call needs."""
    f, unordered, ordered = UNORDERED[call]
    assert f(ctx) == OK
    full = ctx.used()
    seen = []
    for percent in range(1, 221):
        c = Context(ctx.L)
        c.reset(budget=ctx.L.fake_used() + full * percent // 100)
        seen.append((f(c), c.state()))
        c.reset()
        assert ctx.L.sg_destroy(c.h) == OK
    status = [s for s, _ in seen]
    first = status.index(OK)
    assert status[first:] == [OK] * len(status[first:])
    passes = [r for s, r in seen if s == OK]
    assert passes[0] == [ordered] and passes[-1] == [unordered]
    assert sorted(passes, key=lambda r: r == [unordered]) == passes


def test_slabs_are_given_back_for_what_a_call_needs(ctx):
    assert ctx.compute(BIG) == OK and ctx.state() == ["sym"]
    held = ctx.used()
    # one set too large for the pass, on a device with 200 MB left
    ctx.reset(budget=ctx.L.fake_used() + (200 << 20))
    assert ctx.compute((1 << 22) + 1) == OK and ctx.state() == ["ordered"]
    assert ctx.used() < held
    ctx.reset(budget=ctx.L.fake_used() + held)
    assert ctx.compute(BIG) == OK and ctx.state() == ["ordered"]


def test_a_batch_without_its_optional_tables(ctx):
    """The tables of the unordered pass are as optional as its slabs: a batch that
    cannot have one of these five allocations runs the ordered kernel."""
    ran = []
    for k in range(1, 100):
        c = Context(ctx.L)
        ctx.reset(fail=k)
        status = c.batch([5000, 300, 5000])
        reached = ctx.L.fake_mallocs() >= k
        if status == OK:
            ran.append(c.state())
        ctx.reset()
        assert c.batch([5000, 300, 5000]) == OK and c.batch([4000] * 2) == OK
        c.state()
        assert ctx.L.sg_destroy(c.h) == OK
        if not reached:
            break
    assert ran == [["ordered_batch"]] * 5 + [["sym"]]


@pytest.mark.parametrize("n,automatic", [(4096, "adj_wave"), (40000, "adj_sym")])
def test_the_gradient_runs_at_the_workgroup_size_asked_for(ctx, n, automatic):
    for wg in (64, 128, 256):
        assert ctx.L.sg_set_config(ctx.h, 0, wg, 1, 0) == OK
        assert ctx.vjp(n) == OK and ctx.state() == [f"adj_ordered{wg}"]
        ctx.reset()
    assert ctx.L.sg_set_config(ctx.h, 0, 0, 1, 0) == OK
    assert ctx.vjp(n) == OK and ctx.state() == [automatic]


@pytest.mark.parametrize("call", sorted(UNORDERED))
def test_scratch_limit(ctx, call):
    """A limit holds for the memory of the unordered passes only, gives back what
    is held above it, and a new one lets a refused size be asked for again."""
    f, unordered, ordered = UNORDERED[call]
    replay = [[]] if call.startswith("batch") else []   # of a graph: nothing is launched anew
    limit = lambda b: ctx.L.sg_set_scratch_limit(ctx.h, C.c_longlong(b))
    assert ctx.L.sg_set_scratch_limit(None, C.c_longlong(0)) == 1
    assert f(ctx) == OK and ctx.state() == [unordered]
    full = ctx.used()
    assert limit(0) == OK and ctx.used() < full
    ctx.reset()
    assert f(ctx) == OK and ctx.state() == [ordered]
    assert limit(1 << 30) == OK
    ctx.reset()
    assert f(ctx) == OK and ctx.state() in [[ordered]] + replay
    assert ctx.compute(100000) == OK and ctx.state()[-1] == "sym"
    assert limit(-1) == OK
    ctx.reset(budget=ctx.L.fake_used() + (1 << 20))
    assert f(ctx) == OK and ctx.state() in [[ordered]] + replay
    ctx.reset()
    assert f(ctx) == OK and ctx.state() in [[ordered]] + replay   # remembered
    assert limit(-1) == OK
    ctx.reset()
    assert f(ctx) == OK and ctx.state() == [unordered]


def test_slabs_leave_as_much_free_as_they_take(ctx):
    """A program that shares the device (torch's allocator) finds at least as much
    memory free as the unordered pass took."""
    assert ctx.compute(BIG) == OK
    held = ctx.used()
    seen = set()
    for percent in range(60, 260, 5):
        c = Context(ctx.L)
        budget = ctx.L.fake_used() + held * percent // 100
        c.reset(budget=budget)
        assert c.compute(BIG) == OK
        pass_, free = c.state()[0], budget - ctx.L.fake_used()
        seen.add(pass_)
        assert pass_ == "ordered" or free >= 0.9 * held
        c.reset()
        assert ctx.L.sg_destroy(c.h) == OK
    assert seen == {"ordered", "sym"}


_NO_MEMORY = r"""
import resource, sys
sys.path.insert(0, {tests!r})
import test_allocation as t
L = t.load({lib!r})
c = t.Context(L)
used = int(open("/proc/self/statm").read().split()[0]) * 4096
resource.setrlimit(resource.RLIMIT_AS, (used + (60 << 20),) * 2)
print(c.batch([1 << 30, 1 << 29, 300]))
print(c.batch([5000, 300]), c.state())
"""


def test_a_plan_that_host_memory_does_not_hold(built):
    """An exception never leaves a C entry point: the call reports the error."""
    code = _NO_MEMORY.format(tests=os.path.join(ROOT, "tests"), lib=built._name)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])
    assert r.stdout.split("\n")[:2] == ["6", "0 ['sym']"]
