"""Blocking reads and what surrounds them: calls after the work that a read waits for
do not reach back."""
import numpy as np
import pytest

from lbmcl_amd import capi

pytestmark = pytest.mark.gpu


def _read(g):
    return [g.read_rho().view(np.uint32), g.read_u().view(np.uint32)] + [g.read_state(b).view(np.uint32) for b in (0, 1)]


@pytest.mark.parametrize("n, stride, count", [(32, 32, 50), (128, 64, 60), (128, 1, 60)])
def test_a_force_set_after_a_range_does_not_reach_back(n, stride, count):
    got = []
    for force in (False, True):
        with capi.Context(n, stride=stride, profile=False) as g:
            g.initialize()
            g.compute_range(1, count, count)  # rho and u of the last iteration
            if force:
                g.set_force(np.full(3 * n ** 3, 1e-3, np.float32))
            got.append(_read(g))
            g.compute_range(count + 1, 8, 8)
            got.append(_read(g))
    for a, b in zip(got[0], got[2]):
        assert np.array_equal(a, b)
    assert not np.array_equal(got[1][0], got[3][0])  # and after that it does

