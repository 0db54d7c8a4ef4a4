"""Several iterations of a small lattice in one launch (compute_range without
per-launch events): both lattices, rho and u are those of single steps, bit for
bit, for every storage and arithmetic form, counts that are and are not
multiples of a launch's iterations, stored iterations anywhere, strides below and
above a row, a body force, and the smallest lattices.
"""
import numpy as np
import pytest

from lbmcl_amd import capi

pytestmark = pytest.mark.gpu

FORMS = [("f32", "native", "reference"), ("f32", "native", "fused"), ("f32", "native", "exact"),
         ("f64", "native", "reference"), ("f64", "native", "fused"), ("f64", "native", "exact"),
         ("f32", "fp16", "reference"), ("f32", "bf16", "reference")]


def _same(a, b):
    bits = {8: np.uint64, 4: np.uint32, 2: np.uint16}[a.dtype.itemsize]
    return np.array_equal(a.view(bits), b.view(bits)) or (a.dtype.kind == "f" and np.array_equal(a, b, equal_nan=True))


@pytest.mark.parametrize("precision, storage, arith", FORMS)
@pytest.mark.parametrize("n", [4, 8, 16, 32])
def test_launches_of_several_iterations_equal_single_steps(n, precision, storage, arith):
    for stride, steps, every, force in ((n ** 3, 7, 0, False), (min(32, n ** 3), 12, 3, False), (1, 9, 1, True),
                                        (4, 1, 2, False), (n, 2, 2, True)):
        print(n, precision, storage, arith, stride, steps, every, force, flush=True)
        got = []
        for profile in (True, False):  # per-launch events: one launch an iteration
            with capi.Context(n, stride=stride, precision=precision, storage=storage, arith=arith, profile=profile) as g:
                if force:
                    g.set_force((np.random.default_rng(5).standard_normal(3 * n ** 3) * 1e-5).astype(g.dtype))
                g.initialize()
                g.compute_range(1, steps, every)
                g.compute_range(1 + steps, 4, every)
                got.append((g.read_state(0), g.read_state(1), g.read_rho(), g.read_u()))
        for name, a, b in zip(("lattice 0", "lattice 1", "rho", "u"), *got):
            assert _same(a, b), name


def test_more_iterations_than_one_launch_takes():
    """8^3: a launch takes at most 1000 iterations."""
    got = []
    for profile in (True, False):
        with capi.Context(8, stride=32, precision="f64", profile=profile) as g:
            g.initialize()
            g.compute_range(1, 2003, 7)
            got.append((g.read_state(0), g.read_state(1), g.read_rho(), g.read_u()))
    for name, a, b in zip(("lattice 0", "lattice 1", "rho", "u"), *got):
        assert _same(a, b), name
