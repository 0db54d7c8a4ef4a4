"""A gradient's device memory: what it cannot do without comes first, the tapes that
save it time only from what is left (CPU: an allocator of a given capacity; GPU:
somebody else holds most of the memory)."""
import os
import subprocess

import numpy as np
import pytest

from lbmcl_amd import capi
from lbmcl_amd.adjoint import cavity_gradient, gaussian_random_field
from tests.gpu_memory import is_free_soon, memory_held
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
    with memory_held(4 << 30):
        got = cavity_gradient(**kw)
        capi.trim()
    assert got["device_bytes"] < 3e9 < 5e9 < want["device_bytes"]
    for k in ("objective", "d_velocity", "d_viscosity"):
        assert got[k] == want[k]
    assert np.array_equal(got["d_force"], want["d_force"])


@pytest.mark.gpu
def test_as_much_stays_free_as_is_kept():
    """What the library keeps after a gradient and after its context is no more than
    what is free beside it: of 2 GiB, half."""
    with memory_held(2 << 30):
        r = cavity_gradient(64, 150, precision="f64")  # 1.5 GB
        assert r["device_bytes"] > 1.2e9
        assert is_free_soon(1_000_000_000)
        with capi.Context(256, stride=4096, profile=False, storage="fp16") as c:  # 1.5 GB, of which the pool has most
            c.initialize()
            c.finish()
        assert is_free_soon(1_000_000_000)
    capi.trim()


@pytest.mark.gpu
@pytest.mark.parametrize("n, precision, steps, every, grad", [
    (32, "f64", 150, 12, True), (32, "f32", 150, 12, False), (64, "f32", 40, 40, True), (64, "f32", 40, 1, True)])
def test_checkpoint_interval_bounds_the_memory(n, precision, steps, every, grad):
    """With an interval of the caller's: checkpoints, one tape, two lattices and two
    adjoint states, and the gradient's buffers."""
    r = cavity_gradient(n, steps, precision=precision, checkpoint_every=every, grad_force=grad)
    size = 8 if precision == "f64" else 4
    states = -(-steps // every) - 1 + every - 1 + 2 + 2
    fields = (4 * size + 4) + (0 if not grad else 24 + (12 if precision == "f32" else 0))
    assert r["device_bytes"] == n ** 3 * (states * 19 * size + fields)


@pytest.mark.gpu
@pytest.mark.parametrize("steps, every", [(20_000, 1), (100_000_000, 20_000), (10 ** 15, 1)])
def test_state_survives_a_gradient_without_memory(steps, every):
    """A gradient that finds no memory has not touched the context's lattices."""
    n = 64
    with capi.Context(n, precision="f64", profile=False) as a, capi.Context(n, precision="f64", profile=False) as b:
        for c in (a, b):
            c.initialize()
            c.compute_range(1, 5)
        with pytest.raises(capi.LbmError) as e:  # 800 GB at least
            a.adjoint(steps, checkpoint_every=every, grad_force=False)
        assert e.value.code == capi.LBM_ERR_MEMORY
        for c in (a, b):
            c.compute_range(6, 5, 5)
        for k in (0, 1):
            assert np.array_equal(a.read_state(k).view(np.uint64), b.read_state(k).view(np.uint64))
        assert np.array_equal(a.read_rho(), b.read_rho(), equal_nan=True)
