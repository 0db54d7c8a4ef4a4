"""Long ranges on lattices with short runs, which are iterated in another layout:
the same bits as iterations one by one, in both lattices and in the caller's
layout, with what may come before and after (a force, an odd first iteration,
stores, single iterations, a second range)."""
import ctypes

import numpy as np
import pytest

from lbmcl_amd import capi

pytestmark = pytest.mark.gpu


def _words(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32 if a.dtype.itemsize == 4 else np.uint16)


def _agree(a, b):
    for buffer in (0, 1):
        x, y = a.read_state(buffer), b.read_state(buffer)
        if x.dtype == np.uint16:
            assert np.array_equal(x, y)
        else:
            assert np.array_equal(x, y, equal_nan=True)
            ok = ~np.isnan(x)
            assert np.array_equal(_words(x)[ok], _words(y)[ok])
    assert np.array_equal(a.read_rho(), b.read_rho(), equal_nan=True)
    assert np.array_equal(a.read_u(), b.read_u(), equal_nan=True)


@pytest.mark.parametrize("n, stride, precision, storage, arith, count, every, force", [
    (64, 1, "f32", "native", "reference", 12, 0, False), (64, 4, "f32", "native", "reference", 13, 2, False),
    (64, 1, "f32", "native", "reference", 11, 0, False), (64, 16, "f32", "native", "reference", 31, 0, False), (64, 16, "f32", "native", "fused", 33, 5, True),
    (64, 4, "f64", "native", "exact", 35, 7, True), (64, 8, "f64", "native", "reference", 32, 1, False),
    (64, 1, "f32", "fp16", "reference", 34, 0, True), (64, 32, "f32", "bf16", "reference", 33, 33, False),
    (128, 2, "f32", "native", "reference", 37, 10, False), (128, 8, "f32", "native", "exact", 32, 0, True),
    (128, 2, "f64", "native", "reference", 33, 4, True), (256, 16, "f32", "fp16", "reference", 32, 9, False)])
def test_range_matches_single_iterations(n, stride, precision, storage, arith, count, every, force):
    kw = dict(stride=stride, precision=precision, storage=storage, arith=arith, velocity=0.07, viscosity=0.01)
    with capi.Context(n, profile=False, **kw) as a, capi.Context(n, profile=True, **kw) as b:
        if force:
            g = (np.random.default_rng(n).standard_normal(3 * n ** 3) * 1e-6).astype(a.dtype)
            a.set_force(g)
            b.set_force(g)
        for c in (a, b):
            c.initialize()
            c.compute_range(1, count, every)
        _agree(a, b)
        for c in (a, b):
            c.compute(count + 1, update_macro=True)
            c.compute_range(count + 2, 32, 3)
        _agree(a, b)


def test_written_walls_keep_single_iterations():
    """Wall slots with values of the caller's: the other layout would lose them."""
    n, out = 64, []
    for profile in (False, True):
        with capi.Context(n, stride=1, profile=profile) as g:
            g.initialize()
            state = g.read_state(0).reshape(n, n, n, 19)
            state[3, 0, 5, 2] = 0.06
            g.write_state(0, state)
            g.compute_range(1, 40, 8)
            out.append([g.read_state(0), g.read_state(1), g.read_rho(), g.read_u()])
    assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(*out))


def test_first_range_while_a_graph_is_recorded():
    """The third lattice is allocated by the first range, which may fall into
    somebody's recording of a graph on another stream: the recording stays valid."""
    n = 64
    capi.lib()
    h = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library uses
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    assert h.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0  # non-blocking
    capi.trim()
    with capi.Context(n, stride=1, profile=False) as a, capi.Context(n, stride=1, profile=True) as b:
        for c in (a, b):
            c.initialize()
        b.compute_range(1, 40, 8)
        a.finish()
        b.finish()
        assert h.hipStreamBeginCapture(stream, 0) == 0  # global: no thread may allocate
        try:
            a.compute_range(1, 40, 8)
        finally:
            rc = h.hipStreamEndCapture(stream, ctypes.byref(graph))
        assert rc == 0 and graph.value
        assert h.hipGraphDestroy(graph) == 0 and h.hipStreamDestroy(stream) == 0
        _agree(a, b)
