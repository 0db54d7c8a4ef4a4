"""Gradients in device memory that other runs have used: the states of a gradient
get their wall cells' slots set and nothing else, so memory that holds another
run's states (another lid velocity, hence other wall slots) must not show."""
import threading

import numpy as np
import pytest

from lbmcl_amd import capi
from lbmcl_amd.adjoint import cavity_gradient, gaussian_random_field

pytestmark = pytest.mark.gpu
KEYS = ("objective", "d_velocity", "d_viscosity")


def _same(a, b):
    return all(a[k] == b[k] for k in KEYS) and np.array_equal(a["d_force"], b["d_force"])


@pytest.mark.parametrize("n, precision, stride, steps, every, kernel", [
    (4, "f64", 4, 5, 2, 0), (8, "f32", 512, 7, 3, 0), (16, "f64", 1, 9, 1, 0), (32, "f32", 32, 12, 12, 0),
    (64, "f64", 4096, 11, 4, 0), (128, "f32", 2, 10, 3, 0), (128, "f32", 1, 6, 5, 0),
    (64, "f32", 64, 7, 3, capi.LBM_KERNEL_ROW), (32, "f64", 8, 7, 3, capi.LBM_KERNEL_GENERIC)])
def test_gradient_in_used_memory(n, precision, stride, steps, every, kernel):
    g = gaussian_random_field(n, 2.0, 1e-6, seed=n)
    kw = dict(force=g, precision=precision, stride=stride, checkpoint_every=every, kernel=kernel)
    capi.trim()
    want = cavity_gradient(n, steps, velocity=0.05, **kw)
    other = cavity_gradient(n, steps, velocity=-0.07, viscosity=0.02, **kw)
    assert n == 4 or not _same(want, other)  # 4^3 has boundary cells only
    assert _same(want, cavity_gradient(n, steps, velocity=0.05, **kw))
    # states of another arrangement in the same blocks
    cavity_gradient(n, steps, velocity=0.03, **dict(kw, stride=max(1, stride // 2)))
    assert _same(want, cavity_gradient(n, steps, velocity=0.05, **kw))
    capi.trim()
    assert _same(want, cavity_gradient(n, steps, velocity=0.05, **kw))


def test_gradients_of_several_threads():
    n, got = 32, {}
    force = gaussian_random_field(n, 2.0, 1e-6, seed=1)

    def run(i, out):
        for _ in range(3):
            out.setdefault(i, []).append(cavity_gradient(n, 20, velocity=0.03 + 0.01 * i, force=force, checkpoint_every=4))
            if i == 1:
                capi.trim()

    want = {}
    for i in range(3):
        run(i, want)
    threads = [threading.Thread(target=run, args=(i, got)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(3):
        assert len(got[i]) == 3 and all(_same(a, want[i][0]) for a in got[i])
