"""Rates at the edges of the wavefront passes of 64 reactions: mechanisms cut to
reaction counts around whole passes and blocks of passes, reactions with four
products, and non-standard reactions mixed with standard ones."""
import numpy as np
import pytest

from conftest import mech_file

pytestmark = pytest.mark.gpu

TOL = 1e-12     # of each state's largest rate, as the other rate tests


def cut(src, dst, keep):
    """The mechanism with the reactions `keep` (indices, in that order)."""
    head, rxn, n = [], [], -1
    for line in open(src):
        t = line.split()
        if not t or t[0] in ("end", "reactions"):
            continue
        if t[0] == "R":
            n += 1
            rxn.append([])
        (rxn[n] if n >= 0 else head).append(line)
    with open(dst, "w") as f:
        f.writelines(head)
        f.write("reactions %d\n" % len(keep))
        for i, k in enumerate(keep):
            t = rxn[k][0].split()
            f.write(" ".join([t[0], str(i)] + t[2:]) + "\n")
            f.writelines(rxn[k][1:])
        f.write("end\n")
    return str(dst)


def check(path, oracle_mod, n=5, seed=3):
    import cantera_amd as ca
    om, sol = oracle_mod.Mech(path), ca.Solution(path)
    g = np.random.default_rng(seed)
    T = g.uniform(400.0, 2500.0, n)
    P = 101325.0 * 10.0 ** g.uniform(-1, 1.5, n)
    Y = g.dirichlet(0.3 * np.ones(sol.n_species), n)
    Y[0, ::5] *= -1e-6
    w = sol.net_production_rates(T, P, Y.T)
    for s in range(n):
        r = om.rates(T[s], P[s], Y[s])
        scale = max(np.abs(r["wdot"]).max(), np.abs(r["ropf"]).max(), np.abs(r["ropr"]).max(), 1e-300)
        assert np.abs(w[:, s] - r["wdot"]).max() <= TOL * scale
    return sol, T, P, Y


@pytest.mark.parametrize("mech,keep", [
    *[("gri30", range(325 - r, 325)) for r in (1, 63, 64, 65, 128, 129, 192, 193, 256, 257, 320)],
    ("gri30", range(64)),
    ("nDodecane", [13, 15]),                                   # four products only
    ("nDodecane", list(range(10)) + [13] + list(range(70)) + [15]),
])
def test_cut_mechanisms(mech, keep, tmp_path, oracle_mod):
    check(cut(mech_file(mech), tmp_path / "m.mech", list(keep)), oracle_mod)


def test_nan_is_not_hidden(oracle_mod):
    sol, T, P, Y = check(mech_file("gri30"), oracle_mod)
    Y[2, 10] = np.nan
    T[3] = np.nan
    w = sol.net_production_rates(T, P, Y.T)
    reacting = np.abs(sol.net_production_rates(T[:1], P[:1], Y[0])[:, 0]) > 0
    assert np.isnan(w[reacting][:, 2:4]).all()
    assert np.isfinite(w[:, [0, 1, 4]]).all()


@pytest.mark.parametrize("keep,n", [(range(325), 1), (range(325), 3), (range(325), 1025), (range(64), 4),
                                    (range(261, 325), 2), (range(40, 57), 5), ([0], 2)])
def test_jacobian_of_cut_mechanisms(keep, n, tmp_path, oracle_mod):
    """Jacobians at ragged tile counts, at whole passes of reactions, and with
    falloff, three-body or elementary reactions only.  Species columns against
    the oracle's analytic ones, as the Jacobian tests of whole mechanisms."""
    import cantera_amd as ca
    path = cut(mech_file("gri30"), tmp_path / "m.mech", list(keep))
    om, sol = oracle_mod.Mech(path), ca.Solution(path)
    g = np.random.default_rng(n)
    T = g.uniform(600.0, 2500.0, n)
    P = 101325.0 * 10.0 ** g.uniform(-1, 1.5, n)
    X = 10.0 ** g.uniform(-10, 0, (n, sol.n_species))
    Y = sol.mass_fractions_from_moles(X / X.sum(axis=1, keepdims=True))
    J = sol.reactor_jacobians(T, P, Y.T)
    J32 = sol.reactor_jacobians(T, P, Y.T, precision=ca.CG_FP32)
    np.testing.assert_array_equal(J32, J.astype(np.float32))
    assert not J[:, 0].any() and not J[:, :, 0].any()
    for s in {0, n // 2, n - 1}:
        Jo = om.jacobian(P[s], np.concatenate(([1.0, T[s]], Y[s])), analytic=True)
        scale = np.abs(Jo[:, 2:]).max(axis=1, keepdims=True) + 1e-300
        assert (np.abs(J[s][:, 2:] - Jo[:, 2:]) / scale).max() <= 1e-10
