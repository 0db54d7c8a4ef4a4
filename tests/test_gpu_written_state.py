"""States that lbm_write_state brings, and the ranges of iterations that follow: wall
slots keep their bytes, whatever the launches, and a restored state takes the
launches that the run it came from took."""
import numpy as np
import pytest

from lbmcl_amd import capi
from tests.gpu_memory import free_memory, settled_free_memory

pytestmark = pytest.mark.gpu


def _words(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32 if a.dtype.itemsize == 4 else np.uint16)


def _isnan(a, storage):
    if storage == "bf16":
        return (a & 0x7fff) > 0x7f80
    return np.isnan(a.view(np.float16) if storage == "fp16" else a)


@pytest.mark.parametrize("n, stride, precision, storage, count", [
    (8, 8, "f32", "native", 3), (16, 16, "f64", "native", 5), (32, 32, "f32", "fp16", 3), (32, 32, "f32", "bf16", 3),
    (64, 1, "f32", "native", 40), (64, 2, "f32", "fp16", 40), (128, 4096, "f32", "native", 5),
    (128, 4096, "f64", "native", 5)])
def test_payloads_of_wall_slots_stay(n, stride, precision, storage, count):
    """The NaNs of one lattice's wall slots with a payload of the caller's."""
    got = []
    for profile in (True, False):  # per-launch events: one launch an iteration
        with capi.Context(n, stride=stride, precision=precision, storage=storage, profile=profile) as g:
            g.initialize()
            s = g.read_state(0)
            nan = _isnan(s, storage)
            _words(s)[nan] |= 0x15
            g.write_state(0, s)
            g.compute_range(1, count, 2)
            got.append([_words(g.read_state(b)) for b in (0, 1)])
    assert nan.any()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("change", [False, True])
@pytest.mark.parametrize("n, stride, precision, storage", [
    (64, 1, "f32", "native"), (64, 4, "f64", "native"), (64, 2, "f32", "fp16"), (128, 2, "f32", "bf16"),
    (128, 1, "f64", "native"), (128, 8, "f32", "native")])
def test_restored_states_take_the_fast_layout(n, stride, precision, storage, change):
    """A range of a restored lattice with short runs allocates the third lattice that
    the other layout needs, unless a wall slot holds something else than the initial
    lattice's; the same bits as single iterations in either case."""
    kw = dict(stride=stride, precision=precision, storage=storage)
    with capi.Context(n, profile=False, **kw) as a, capi.Context(n, profile=True, **kw) as b:
        b.initialize()
        b.compute_range(1, 3)
        state = [b.read_state(k) for k in (0, 1)]
        if change:  # cell (0, 3, 5) is a wall; population 1 leaves it for (1, 3, 5)
            c = n * (3 + n * 5)
            state[1][((c // stride) * 19 + 1) * stride + c % stride] = state[1][19 * 8]
        for c in (a, b):
            c.initialize()
            for k in (0, 1):
                c.write_state(k, state[k])
        capi.trim()
        a.finish()
        before = settled_free_memory()
        a.compute_range(4, 64, 5)
        a.finish()
        taken = before - free_memory()
        b.compute_range(4, 64, 5)
        lattice = 19 * n ** 3 * a.sdtype(0).itemsize
        # a lattice or none; what else the runtime allocates and frees is megabytes
        assert (taken < lattice // 2) if change else (taken > lattice // 2), (taken, lattice)
        for k in (0, 1):
            x, y = _words(a.read_state(k)), _words(b.read_state(k))
            assert np.array_equal(x, y)
        assert np.array_equal(a.read_rho(), b.read_rho(), equal_nan=True)
        assert np.array_equal(a.read_u(), b.read_u(), equal_nan=True)
