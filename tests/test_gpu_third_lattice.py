"""The third lattice of a context whose ranges are iterated in another layout comes
back without the end of the context: by lbm_trim, and for another allocation of the
library's."""
import numpy as np
import pytest

from lbmcl_amd import capi
from tests.gpu_memory import free_memory, is_free_soon, memory_held, settled_free_memory

pytestmark = pytest.mark.gpu


def _agree(a, b):
    for k in (0, 1):
        assert np.array_equal(a.read_state(k).view(np.uint32), b.read_state(k).view(np.uint32))
    assert np.array_equal(a.read_rho(), b.read_rho(), equal_nan=True)


def test_trim_takes_it_back():
    n = 128
    lattice = 19 * 4 * n ** 3
    with capi.Context(n, stride=1, profile=False) as a, capi.Context(n, stride=1, profile=True) as b:
        for c in (a, b):
            c.initialize()
        capi.trim()
        a.finish()
        before = settled_free_memory()
        a.compute_range(1, 40, 7)
        assert before - free_memory() > lattice // 2
        capi.trim()  # the range may still be under way
        assert is_free_soon(before - lattice // 2)
        a.compute_range(41, 40, 7)
        assert before - free_memory() > lattice // 2
        b.compute_range(1, 80, 7)
        _agree(a, b)
    capi.trim()


def test_another_allocation_takes_it_back():
    n = 256  # 1.3 GB a lattice
    lattice = 19 * 4 * n ** 3
    kw = dict(stride=1, velocity=0.06)
    with capi.Context(n, profile=True, **kw) as b:
        b.initialize()
        b.compute_range(1, 80, 7)
        with capi.Context(n, profile=False, **kw) as a:
            a.initialize()
            capi.trim()
            a.compute_range(1, 40, 7)
            a.finish()
            with memory_held(2 * lattice - (512 << 20)):  # not enough for two lattices, rho and u
                with capi.Context(n, profile=False, stride=4096) as c:
                    c.initialize()
                    c.compute_range(1, 4)
                    c.finish()
            capi.trim()
            a.compute_range(41, 40, 7)
            _agree(a, b)
    capi.trim()


@pytest.mark.parametrize("n, stride, precision, storage, from_", [
    (64, 8, "f64", "native", 96), (64, 1, "f32", "fp16", 24), (64, 16, "f32", "bf16", 24)])
def test_ranges_about_the_length_that_pays(n, stride, precision, storage, from_):
    """One iteration less stays in the layout, one more goes through the other: the
    same bits as single iterations."""
    kw = dict(stride=stride, precision=precision, storage=storage, velocity=0.07)
    for count in (from_ - 1, from_, from_ + 1):
        with capi.Context(n, profile=False, **kw) as a, capi.Context(n, profile=True, **kw) as b:
            for c in (a, b):
                c.initialize()
                c.compute_range(1, count, 5)
            for k in (0, 1):
                assert np.array_equal(a.read_state(k).view(np.uint8), b.read_state(k).view(np.uint8))
            assert np.array_equal(a.read_rho(), b.read_rho(), equal_nan=True)
            assert np.array_equal(a.read_u(), b.read_u(), equal_nan=True)
