"""Gradients of a run whose populations leave the range of the type: a lambda that is
not finite reaches every component of its cell's body-force gradient (its product
with the zeros of the lattice vectors too is a NaN), and none of them looks like a
gradient."""
import numpy as np
import pytest

from lbmcl_amd.adjoint import cavity_gradient

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("objective", ["kinetic_energy", "mean_ux_plane"])
@pytest.mark.parametrize("n, precision, steps, velocity", [
    (16, "f32", 1, 1e12), (16, "f32", 2, 1e8), (64, "f32", 1, 1e18), (64, "f32", 5, 1e8), (16, "f64", 1, 1e100),
    (64, "f64", 1, 1e153)])
def test_no_component_of_a_diverged_gradient_is_finite_alone(n, precision, steps, velocity, objective):
    r = cavity_gradient(n, steps, velocity=velocity, precision=precision, objective=objective, plane_z=n - 3)
    assert not np.isfinite(r["objective"]) and not np.isfinite(r["d_velocity"])
    finite = np.isfinite(r["d_force"])
    assert not finite.all()
    assert np.array_equal(finite[0], finite[1]) and np.array_equal(finite[0], finite[2])
