"""Two iterations in one launch (compute_range without per-launch events).

The two-step kernel evaluates the single-step kernels' expressions, so both
lattices, rho and u are theirs bit for bit.  Lattices with each kind of tile
(whole rows, two segments a row, segments with halo threads), strides below and
above a row, odd and even counts, stored iterations on either half of a pair,
restored states, and wall slots that are not the initial lattice's.
"""
import numpy as np
import pytest

from lbmcl_amd import capi

pytestmark = pytest.mark.gpu


def _same(a, b):
    bits = {8: np.uint64, 4: np.uint32}[a.dtype.itemsize]
    return np.array_equal(a.view(bits), b.view(bits)) or np.array_equal(a, b, equal_nan=True)


def _force(n, dtype):
    return (np.random.default_rng(5).standard_normal(3 * n ** 3) * 1e-5).astype(dtype)


@pytest.mark.parametrize("n, stride, precision, arith, steps, every, force", [
    (128, 32, "f32", "reference", 7, 0, False),
    (128, 128, "f32", "fused", 8, 2, False),
    (128, 8, "f32", "exact", 5, 3, False),
    (128, 4, "f64", "reference", 6, 1, False),
    (128, 4096, "f64", "fused", 7, 2, True),
    (128, 64, "f64", "exact", 4, 4, True),
    (128, 128 ** 3, "f64", "reference", 5, 0, False),
    (256, 4096, "f32", "reference", 6, 4, False),
    (256, 64, "f64", "reference", 5, 0, False),
    (128, 4096, "f32", "reference", 7, 2, True),  # FP32 with a force: single steps
])
def test_pairs_equal_single_steps(n, stride, precision, arith, steps, every, force):
    print(n, stride, precision, arith, steps, every, force, flush=True)
    got = []
    for profile in (True, False):  # per-launch events: one launch an iteration
        with capi.Context(n, stride=stride, precision=precision, arith=arith, profile=profile) as g:
            if force:
                g.set_force(_force(n, g.dtype))
            g.initialize()
            g.compute_range(1, 2, every)
            g.compute_range(3, steps, every)
            got.append((g.read_state(0), g.read_state(1), g.read_rho(), g.read_u()))
    for name, a, b in zip(("lattice 0", "lattice 1", "rho", "u"), *got):
        assert _same(a, b), name


@pytest.mark.parametrize("n, precision", [(512, "f32"), (512, "f64"), (1024, "f32")])
def test_pairs_equal_single_steps_large(n, precision):
    """Two segments a row, and halo threads in either precision."""
    print(n, precision, flush=True)
    got = []
    for profile in (True, False):
        with capi.Context(n, stride=4096, precision=precision, profile=profile) as g:
            g.initialize()
            g.compute_range(1, 6)
            g.compute(7, update_macro=True)
            got.append((g.read_rho(), g.read_u()))
    for name, a, b in zip(("rho", "u"), *got):
        assert _same(a, b), name


@pytest.mark.parametrize("precision", ["f32", "f64"])
def test_restored_state_and_other_walls(precision):
    """A restored state continues as the run it came from; a state whose wall slots
    differ from the initial lattice's keeps them (and takes single steps)."""
    n, stride = 128, 4096
    with capi.Context(n, stride=stride, precision=precision, profile=False) as g:
        g.initialize()
        g.compute_range(1, 4)
        s0, s1 = g.read_state(0), g.read_state(1)
        g.compute_range(5, 5)
        want = g.read_state(0), g.read_state(1)
        g.initialize()
        g.write_state(0, s0)
        g.write_state(1, s1)
        g.compute_range(5, 5)
        assert _same(g.read_state(0), want[0]) and _same(g.read_state(1), want[1])
    # cell (5, 0, 5) is a wall; population 2 leaves it for (5, 1, 5)
    c = 5 + n * n * 5
    slot = ((c // stride) * 19 + 2) * stride + c % stride
    s0[slot] = 0.06
    got = []
    for profile in (True, False):
        with capi.Context(n, stride=stride, precision=precision, profile=profile) as g:
            g.initialize()
            g.write_state(0, s0)
            g.write_state(1, s1)
            g.compute_range(5, 5)
            got.append((g.read_state(0), g.read_state(1)))
    assert _same(got[0][0], got[1][0]) and _same(got[0][1], got[1][1])
    assert not _same(got[0][0], want[0])
