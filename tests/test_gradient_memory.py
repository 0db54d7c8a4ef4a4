"""A gradient's device memory: what it cannot do without comes first, the tapes that
save it time only from what is left (CPU: an allocator of a given capacity; GPU:
somebody else holds most of the memory)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from lbmcl_amd import capi
from lbmcl_amd.adjoint import cavity_gradient, gaussian_random_field
from tests.native import build_native


@pytest.mark.parametrize("sanitize", [None, "asan"])
def test_memory_of_a_gradient(sanitize):
    r = subprocess.run([build_native.build("tapes_test", sanitize)], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1"))
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stderr[-2000:]


@pytest.mark.gpu
def test_gradient_beside_somebody_elses_memory():
    """64^3 FP64 x 150: 1 GB that it needs, and 6 GB where memory is plentiful."""
    kw = dict(dim=64, steps=150, precision="f64", force=gaussian_random_field(64, 8.0, 1e-6, seed=2))
    want = cavity_gradient(**kw)
    capi.trim()
    h = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library uses
    h.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    h.hipFree.argtypes = [ctypes.c_void_p]
    held = []
    try:
        while True:
            free, total = ctypes.c_size_t(), ctypes.c_size_t()
            assert h.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            take = min(free.value - (4 << 30), 32 << 30)
            if take < (64 << 20):
                break
            p = ctypes.c_void_p()
            assert h.hipMalloc(ctypes.byref(p), take) == 0
            held.append(p)
        got = cavity_gradient(**kw)
    finally:
        for p in held:
            assert h.hipFree(p) == 0
        capi.trim()
    assert got["device_bytes"] < 3e9 < 5e9 < want["device_bytes"]
    for k in ("objective", "d_velocity", "d_viscosity"):
        assert got[k] == want[k]
    assert np.array_equal(got["d_force"], want["d_force"])
