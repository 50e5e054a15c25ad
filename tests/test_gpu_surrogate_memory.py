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
