"""States that lbm_write_state brings, and the ranges of iterations that follow: wall
slots keep their bytes, whatever the launches."""
import numpy as np
import pytest

from lbmcl_amd import capi

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
