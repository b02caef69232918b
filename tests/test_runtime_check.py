"""The check that torch and the library share one HIP runtime is made anew
when the process loads a shared object, and only then."""
import ctypes
import os
import shutil
import subprocess
import sys

import pytest

from starsmasher_amd import _lib, gravity

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_verdict_stands_until_an_object_is_loaded(monkeypatch, tmp_path):
    _lib.load()
    found, calls = ["/a/libamdhip64.so"], []
    monkeypatch.setattr(gravity, "hip_runtimes", lambda: calls.append(1) or found)
    monkeypatch.setattr(gravity, "_one_runtime_at", None)
    for _ in range(3):
        gravity._check_shared_runtime("x")
    assert len(calls) == 1
    copy = tmp_path / "liboracle_copy.so"
    shutil.copy(os.path.join(ROOT, "oracle", "liboracle.so"), copy)
    lib = ctypes.CDLL(str(copy))
    found.append("/b/libamdhip64.so")
    for _ in range(2):   # a refusal is not kept: every call reads the maps
        with pytest.raises(TypeError):
            gravity._check_shared_runtime("x")
    assert len(calls) == 3 and lib


_BOTH = r"""
import _ctypes, sys, threading
sys.path.insert(0, {root!r})
from starsmasher_amd import _lib, gravity
_lib.load()
gravity.hip_runtimes = lambda: ["one"]
sys.setswitchinterval(1e-5)
stop = threading.Event()
def load():   # as an import of an extension module does, with the GIL held
    while not stop.is_set():
        _ctypes.dlclose(_ctypes.dlopen({lib!r}, 2))
t = threading.Thread(target=load)
t.start()
for _ in range(20000):
    gravity._check_shared_runtime("x")
stop.set()
t.join()
print("done")
"""


def test_check_while_another_thread_loads_objects(tmp_path):
    """The dynamic linker's lock is never held while waiting for the GIL."""
    copy = tmp_path / "liboracle_copy.so"
    shutil.copy(os.path.join(ROOT, "oracle", "liboracle.so"), copy)
    r = subprocess.run([sys.executable, "-c", _BOTH.format(root=ROOT, lib=str(copy))],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "done\n", r.stderr
