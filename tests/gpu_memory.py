"""Device memory beside the library, for tests: what is free, and somebody who holds
most of it."""
from __future__ import annotations

import contextlib
import ctypes
import time

from lbmcl_amd import capi


def _hip():
    capi.lib()  # the library first: its libamdhip64 is the one loaded below
    h = ctypes.CDLL("libamdhip64.so.7")
    h.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    h.hipFree.argtypes = [ctypes.c_void_p]
    return h


def free_memory() -> int:
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def settled_free_memory() -> int:
    """What is free once it has not changed for a while (see is_free_soon)."""
    reads = [free_memory()]
    while len(reads) < 100 and (len(reads) < 8 or len(set(reads[-8:])) > 1):
        time.sleep(0.03)
        reads.append(free_memory())
    return reads[-1]


def is_free_soon(at_least: int) -> bool:
    """Whether that much is free within a few seconds: the driver counts freed memory
    as free a while after hipFree."""
    for _ in range(100):
        if free_memory() >= at_least:
            return True
        time.sleep(0.05)
    return False


@contextlib.contextmanager
def memory_held(leave: int):
    """Hold all of the device's memory but about `leave` bytes."""
    h, held = _hip(), []
    try:
        while (take := min(free_memory() - leave, 32 << 30)) >= 64 << 20:
            p = ctypes.c_void_p()
            assert h.hipMalloc(ctypes.byref(p), take) == 0
            held.append(p)
        yield
    finally:
        for p in held:
            assert h.hipFree(p) == 0
