"""The deepest network, 16 hidden layers and 17 parameter blocks (the last
entries of the layer tables of the fused inference and of the one-launch weight
gradient), with parameters that neither damp nor amplify: hidden layers near the
identity, activations near 3, where GELU is nearly the identity too.  Against the
float64 numpy restatements that round to BF16 where the device does.

Gradient: an activation within FP32 summation error of a BF16 rounding boundary
rounds the other way; with relative perturbations of 3e-7 of every pre-activation
the restatement's gradient moves by less than 1e-3 per layer, bar 2e-2 as for
shallow networks.  Prediction: such a rounding is 2^-6 in one activation and moves
a pre-activation of the layers behind by 2^-6 x 0.02 / 8, so that some tens of
activations of a row may differ at the end, each times an output weight of at
most 0.1: 30 x 2^-6 x 0.1 = 5e-2."""
import numpy as np
import pytest

from conftest import mech_file
from test_gpu_surrogate import pad, reference_loss_grad, synthetic_pairs
from test_gpu_surrogate_infer import network_output

pytestmark = pytest.mark.gpu
DEPTH = 16


def parameters(K, hidden, seed):
    g = np.random.default_rng(seed)
    ip, op, p = pad(K + 2), pad(K + 1), []
    for l in range(DEPTH + 1):
        fi, fo = (ip if l == 0 else hidden), (op if l == DEPTH else hidden)
        W, b = np.zeros((fo, fi)), np.zeros(fo)
        if l == 0:
            W[:, :K + 2] = g.normal(0, 0.3 / np.sqrt(K + 2), (fo, K + 2))
            b[:] = 3
        elif l < DEPTH:
            W[:] = np.eye(hidden) + g.normal(0, 0.02 / np.sqrt(hidden), (fo, fi))
        else:
            W[:K + 1] = g.normal(0, 0.3 / np.sqrt(hidden), (K + 1, fi))
            b[:K + 1] = g.normal(0, 0.1, K + 1)
        p += [W.ravel(), b]
    return np.concatenate(p).astype(np.float32)


@pytest.mark.parametrize("mech,hidden,rows", [("gri30", 128, 130), ("h2o2", 64, 200)])
def test_sixteen_layers(mech, hidden, rows):
    import cantera_amd as ca
    from cantera_amd.surrogate import Surrogate
    from cantera_amd.workloads import MechInfo
    sol = ca.Solution(mech)
    K = sol.n_species
    sur = Surrogate(sol, dt=1e-6, hidden=hidden, depth=DEPTH, seed=1)
    y0, P, y1 = synthetic_pairs(MechInfo(mech_file(mech)), 256, 5)
    sur.fit_normalization(y0, P, y1)
    sur.params = parameters(K, hidden, 1)
    y0, P, y1 = y0[:rows], P[:rows], y1[:rows]
    params, norm = sur.params, sur.normalization
    loss, g = sur.loss_grad(y0, P, y1)
    rl, rg, sizes = reference_loss_grad(params, norm, K, hidden, DEPTH, y0, P, y1)
    assert len(sizes) == 17
    assert abs(loss - rl) <= 1e-4 * rl
    off = 0
    for s in sizes:
        a, b = g[off:off + s].astype(np.float64), rg[off:off + s].astype(np.float64)
        assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b)
        off += s
    ip, op = pad(K + 2), pad(K + 1)
    mu, sd, sc = (norm[2 * ip + i * op:2 * ip + i * op + K + 1] for i in range(3))
    arg = network_output(params, norm, K, hidden, DEPTH, y0, P) * sd + mu
    got = sur.predict(y0, P)
    # the temperature is not projected
    assert np.all(np.abs(got[:, 1] - (y0[:, 1] + sc[0] * np.sinh(arg[:, 0])))
                  <= sc[0] * np.cosh(arg[:, 0]) * sd[0] * 5e-2 + 1e-12 * y0[:, 1])
