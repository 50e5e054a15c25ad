"""Record columns read back to the host (states, control blocks, status):
dense copies in passes of 8 MiB, here at counts around a pass's row limit."""
import numpy as np
import pytest

import cantera_amd as ca
from cantera_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu

ROWS = 8 * 1024 * 1024 // (64 * 8)      # control blocks of one pass


@pytest.mark.parametrize("n", [1, ROWS - 1, ROWS, ROWS + 1, 5 * ROWS + 3 * ROWS // 7])
def test_readback_is_exact_around_a_pass(n):
    sol = ca.Solution("h2o2")
    g = np.random.default_rng(n)
    T, P = g.uniform(300.0, 2500.0, n), g.uniform(1e4, 1e6, n)
    Y = g.dirichlet(np.ones(sol.n_species), n)
    rb = ca.ReactorBatch(sol, T, P, Y)
    y = rb.state
    np.testing.assert_array_equal(y[:, 1], T)
    np.testing.assert_array_equal(y[:, 2:], Y)
    dev = DeviceArray.empty((n, rb.neq))
    rb.state_to_device(dev)
    assert ca.lib().cg_device_synchronize() == 0
    np.testing.assert_array_equal(dev.get(), y)
    ctl = np.full((n, 64), np.nan)
    assert ca.lib().cg_reactors_get_control(rb.handle, ctl) == 0
    np.testing.assert_array_equal(ctl[:, 45], P)
    assert not rb.status.any()
    assert not rb.stats["steps"].any()
