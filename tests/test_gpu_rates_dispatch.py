"""Rates on both sides of the sizes at which several states go to a wavefront
(2,049 states for a mechanism of at most 64 reactions, 4,096 for a larger one),
against the oracle: the first and the last tile, and a later one."""
import numpy as np
import pytest

from conftest import mech_file

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech,n", [(m, n) for m in ("h2o2", "pdep-test", "noxNeg") for n in (2048, 2049, 4095)] +
                         [(m, n) for m in ("gri30", "nDodecane") for n in (2049, 4095, 4096)])
def test_rates_match_oracle(mech, n, oracle_mod):
    import cantera_amd as ca
    sol = ca.Solution(mech)
    om = oracle_mod.Mech(mech_file(mech))
    r = np.random.Generator(np.random.Philox(n))
    Y = 10.0 ** r.uniform(-6, 0, (sol.n_species, n)) * sol.molecular_weights[:, None]
    Y /= Y.sum(axis=0)
    T, P = r.uniform(500.0, 2500.0, n), 101325.0 * 10.0 ** r.uniform(-1.0, 1.7, n)
    w = sol.net_production_rates(T, P, Y)
    for s in [*range(8), *range(n // 2, n // 2 + 8), *range(n - 9, n)]:
        o = om.rates(T[s], P[s], np.ascontiguousarray(Y[:, s]))
        # sums of rates of progress in another order: at most 400 terms, each
        # of the state's largest
        scale = max(np.abs(o["ropf"]).max(), np.abs(o["ropr"]).max())
        assert np.abs(w[:, s] - o["wdot"]).max() <= 1e-12 * scale
