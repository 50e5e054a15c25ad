"""Device memory of the surrogate: a prediction holds its outputs (and, layer by
layer, two activations), not what training needs; a request that fails leaves
the net usable."""
import ctypes

import numpy as np
import pytest

from conftest import mech_file
from test_gpu_surrogate import synthetic_pairs

pytestmark = pytest.mark.gpu


def free_bytes():
    """hipMemGetInfo of the runtime that the library has loaded."""
    from cantera_amd._lib import check, lib
    check(lib().cg_device_synchronize())
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so.7").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.fixture(scope="module")
def gri30():
    import cantera_amd as ca
    from cantera_amd.workloads import MechInfo
    return ca.Solution("gri30"), synthetic_pairs(MechInfo(mech_file("gri30")), 4096, 5)


@pytest.mark.parametrize("hidden,per_row", [(256, 256), (320, 256 + 128 + 4 * 320)])
def test_predict_allocates_what_it_uses(gri30, hidden, per_row):
    from cantera_amd._lib import check, lib
    from cantera_amd.surrogate import DeviceArray, Surrogate
    sol, (y0, P, y1) = gri30
    n = 65536
    sur = Surrogate(sol, dt=1e-6, hidden=hidden, depth=4, seed=1)
    sur.fit_normalization(y0, P, y1)
    d0, dP = DeviceArray(np.tile(y0, (16, 1))), DeviceArray(np.tile(P, 16))
    out = DeviceArray.empty((n, y0.shape[1]))
    check(lib().cg_surrogate_predict(sur.handle, 64, d0.ptr, dP.ptr, out.ptr))   # code objects loaded
    before = free_bytes()
    check(lib().cg_surrogate_predict(sur.handle, n, d0.ptr, dP.ptr, out.ptr))
    assert before - free_bytes() <= n * per_row + (16 << 20)   # allocations come in blocks of 2 MiB


def test_a_failed_request_leaves_the_net_usable(gri30):
    """An epoch in batches of 2^31 - 1 rows (4.7 TB of activations) fails with an
    error; what was computed before it is computed again."""
    from cantera_amd._lib import lib
    from cantera_amd.surrogate import DeviceArray, Surrogate
    sol, (y0, P, y1) = gri30
    y0, P, y1 = y0[:64], P[:64], y1[:64]
    sur = Surrogate(sol, dt=1e-6, hidden=256, depth=4, seed=1)
    sur.fit_normalization(y0, P, y1)
    loss, grad = sur.loss_grad(y0, P, y1)
    pred = sur.predict(y0, P)
    d0, dP, d1 = DeviceArray(y0), DeviceArray(P), DeviceArray(y1)
    assert lib().cg_surrogate_train_epoch(sur.handle, 64, d0.ptr, dP.ptr, d1.ptr, 2 ** 31 - 1, 1e-3, None) == -999
    for _ in range(2):
        again, g = sur.loss_grad(y0, P, y1)
        assert again == loss
        np.testing.assert_array_equal(g, grad)
    np.testing.assert_array_equal(sur.predict(y0, P), pred)


def test_gradient_of_more_layers_than_are_held():
    """Above 256 MB the layers' gradient operands take turns.  Twice the rows:
    the mean loss and its gradient are the means over the halves, which are below
    that size; factors of 2 are exact in BF16, so only the order of FP32 sums of
    16,384 terms differs (random signs: 128 roundings, 8e-6 of the terms' norm,
    within a factor of 10 of the sum's)."""
    import cantera_amd as ca
    from cantera_amd.surrogate import Surrogate
    from cantera_amd.workloads import MechInfo
    sol = ca.Solution("h2o2")
    hidden, depth, n = 512, 16, 16384
    y0, P, y1 = synthetic_pairs(MechInfo(mech_file("h2o2")), n, 5)
    sur = Surrogate(sol, dt=1e-6, hidden=hidden, depth=depth, seed=1)
    sur.fit_normalization(y0, P, y1)
    halves = [sur.loss_grad(y0[s], P[s], y1[s]) for s in (slice(0, n // 2), slice(n // 2, n))]
    loss, grad = sur.loss_grad(y0, P, y1)
    assert abs(loss - (halves[0][0] + halves[1][0]) / 2) <= 1e-6 * loss
    mean = (halves[0][1].astype(np.float64) + halves[1][1]) / 2
    widths = [64] + [hidden] * depth + [64]
    off = 0
    for fi, fo in zip(widths, widths[1:]):
        a, b = grad[off:off + fo * fi + fo].astype(np.float64), mean[off:off + fo * fi + fo]
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b)
        off += fo * fi + fo


def test_gradient_operands_are_bounded(gri30):
    """Activations and pre-activations of every layer, outputs, and at most 256
    MB of gradient operands, not one of every layer (1.1 GB here)."""
    from cantera_amd._lib import check, lib
    from cantera_amd.surrogate import DeviceArray, Surrogate
    sol, (y0, P, y1) = gri30
    hidden, depth, n = 512, 16, 65536
    sur = Surrogate(sol, dt=1e-6, hidden=hidden, depth=depth, seed=1)
    sur.fit_normalization(y0, P, y1)
    sur.loss_grad(y0[:64], P[:64], y1[:64])   # code objects loaded
    d0, dP, d1 = (DeviceArray(np.tile(x, (16,) + (1,) * (x.ndim - 1))) for x in (y0, P, y1))
    before = free_bytes()
    check(lib().cg_surrogate_loss_grad(sur.handle, n, d0.ptr, dP.ptr, d1.ptr, None, None))
    partial = 3 * 4 * sur.n_params            # gradient copies of row splits, few at this size
    assert before - free_bytes() <= n * (6 * depth * hidden + 2 * 64 + 8 * 64) + (256 << 20) + partial + (32 << 20)
