"""The host code of a context when device memory runs short, on the CPU:
sg_capi.cpp linked against a device made of bookkeeping (fake_device.cpp), whose
launches are checked for the buffers they would work in."""
import ctypes as C
import os
import subprocess

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
    # RTLD_DEEPBIND: its own hipMalloc and not that of a runtime loaded before
    L = C.CDLL(str(so), mode=os.RTLD_LOCAL | os.RTLD_DEEPBIND)
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
