"""Batches large enough for several states per wavefront against the
one-state-per-wavefront kernel on the same states, for every reaction form:
ragged tile counts, negative mass fractions, both precisions."""
import os

import numpy as np
import pytest

from conftest import mech_file

pytestmark = pytest.mark.gpu

WIDE = 4096     # from here every mechanism's states go several to a wavefront, below 2,049 none's
MECHS = ["h2o2", "gri30", "nDodecane", "noxNeg", "pdep-test", "sri-falloff", "tsang-falloff",
         "chemically-activated-reaction", "frac", "gri30_ndodecane"]


@pytest.mark.parametrize("mech,n,fp32", [(m, WIDE + 5, False) for m in MECHS] +
                         [("gri30", n, False) for n in (WIDE, WIDE + 7, WIDE + 8, 5 * WIDE + 1)] +
                         [("gri30", WIDE + 7, True), ("nDodecane", WIDE + 3, True), ("pdep-test", WIDE + 1, True)])
def test_wide_matches_narrow(mech, n, fp32):
    import cantera_amd as ca
    path = os.path.join(os.path.dirname(__file__), "golden", mech + ".mech")
    sol = ca.Solution(path if os.path.exists(path) else mech_file(mech))
    g = np.random.default_rng(n + len(mech))
    K = sol.n_species
    T = g.uniform(300.0, 2500.0, n)
    P = 101325.0 * 10.0 ** g.uniform(-1.0, 1.7, n)
    Y = 10.0 ** g.uniform(-8.0, 0.0, (K, n))
    Y /= Y.sum(axis=0)
    Y[g.integers(0, K, n // 8), g.integers(0, n, n // 8)] *= -1e-3
    prec = ca.CG_FP32 if fp32 else ca.CG_FP64
    wide = sol.net_production_rates(T, P, Y, precision=prec)
    narrow = np.concatenate([sol.net_production_rates(T[i:i + 2048], P[i:i + 2048], Y[:, i:i + 2048], precision=prec)
                             for i in range(0, n, 2048)], axis=1)
    # the same formulas in the same precision: only the order of a species'
    # terms differs (at most 400 of them, each within the state's largest
    # rate of progress, which cancellation can leave far above the net rate)
    w2 = np.abs(wide - narrow)
    scale = np.maximum(np.abs(narrow).max(axis=0), 1e-300)
    assert np.isfinite(wide).all()
    assert np.median(w2.max(axis=0) / scale) <= 1e-13
    assert (w2.max(axis=0) / scale).max() <= 1e-9
