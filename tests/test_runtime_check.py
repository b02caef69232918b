"""The check that torch and the library share one HIP runtime is made anew
when the process loads a shared object, and only then."""
import ctypes
import os
import shutil

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
