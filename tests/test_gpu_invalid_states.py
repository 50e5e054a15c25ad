"""States that no gas can have (zero or infinite pressure, no mass, NaN): what
is defined whatever the state stays so, and a bad state spoils no other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BAD = ["P0", "Pinf", "Tnan", "Yzero", "Ynan"]


def states(sol, n, seed=11):
    r = np.random.Generator(np.random.Philox(seed))
    Y = 10.0 ** r.uniform(-6, 0, (sol.n_species, n)) * sol.molecular_weights[:, None]
    return r.uniform(800.0, 2500.0, n), 101325.0 * np.exp(r.uniform(-2, 3, n)), Y / Y.sum(0)


def spoil(kind, T, P, Y, s):
    if kind[0] == "T":
        T[s] = np.nan
    elif kind[0] == "P":
        P[s] = {"0": 0.0, "inf": np.inf}[kind[1:]]
    else:
        Y[:, s] = 0.0 if kind == "Yzero" else np.nan


@pytest.mark.parametrize("mech", ["gri30", "h2o2", "tsang-falloff", "pdep-test"])
def test_mass_row_and_column_are_zero(mech):
    """ydot does not depend on the mass: that row and column of the Jacobian are
    zero at every state, and states beside a bad one are those of a clean batch."""
    import cantera_amd as ca
    sol = ca.Solution(mech)
    T, P, Y = states(sol, 2 * len(BAD))
    clean = sol.reactor_jacobians(T, P, Y)
    for i, kind in enumerate(BAD):
        spoil(kind, T, P, Y, 2 * i)
    J = sol.reactor_jacobians(T, P, Y)
    assert np.array_equal(J[:, 0, :], np.zeros_like(J[:, 0, :]))
    assert np.array_equal(J[:, :, 0], np.zeros_like(J[:, :, 0]))
    # FP64 atomics in the general kernel: no fixed order
    scale = np.abs(clean[1::2]).max(axis=(1, 2), keepdims=True)
    assert np.abs(J[1::2] - clean[1::2]).max() <= 1e-12 * scale.max()
    assert np.all(np.abs(J[1::2] - clean[1::2]) <= 1e-12 * scale)


@pytest.mark.parametrize("mech", ["gri30", "h2o2", "pdep-test", "chemically-activated-reaction"])
@pytest.mark.parametrize("n", [20, 4100])
def test_exponents_beyond_any_range(mech, n):
    """Far outside the fits of the thermodynamics the exponent of an equilibrium
    constant passes 1e13: exp is then 0 or infinite, of no other sign, as in the
    oracle.  n on either side of the kernels' switch."""
    import cantera_amd as ca
    from conftest import mech_file
    from oracle.oracle import Mech
    sol, om = ca.Solution(mech), Mech(mech_file(mech))
    T, P, Y = states(sol, n)
    T[:10], T[10:20] = 1e10, 1e12
    w = sol.net_production_rates(T, P, Y)
    for s in range(20):
        ref = om.rates(T[s], P[s], np.ascontiguousarray(Y[:, s]))["wdot"]
        assert np.array_equal(np.isnan(w[:, s]), np.isnan(ref))
        assert np.array_equal(np.where(np.isinf(w[:, s]), w[:, s], 0.0), np.where(np.isinf(ref), ref, 0.0))
