"""The parameter terms of the adjoint's Hessian pass for pair tables that are gathered (six exchange pairs
that hold the DMI pairs) and that are not: several shells of both, shells without DMI, two basis atoms,
periodic and open axes, no pairs at all, and as many exchange parameters as there are slots.  Each
parameter against the tangent-linear run: both are exact derivatives of the same map, 1e-9 relative to
the larger of the two sides and of 1e-6 of all parameters' (the other way round of rounding in 12 steps)."""
import numpy as np
import pytest

from test_gpu_adjoint import FILM, state  # noqa: F401  (fixture)

from spirit_amd import configs

pytestmark = pytest.mark.gpu

OPEN = dict(FILM, ddi_method="none")
MODELS = {
    "one_shell_each": dict(OPEN, n_basis_cells=[9, 7, 5]),
    "one_shell_dipolar": dict(FILM, n_basis_cells=[7, 5, 4], boundary_conditions=[1, 0, 0]),
    "no_dmi": dict(OPEN, n_shells_dmi=0, dij=[], boundary_conditions=[1, 1, 1]),
    "three_shells_two_dmi": dict(OPEN, n_shells_exchange=3, jij=[5.0, 1.0, -0.5], n_shells_dmi=2, dij=[1.0, 0.3]),
    "eight_shells": dict(OPEN, n_basis_cells=[11, 9, 8], n_shells_exchange=8,
                         jij=[5.0, 1.0, -0.5, 0.2, 0.1, 0.1, -0.1, 0.05], boundary_conditions=[1, 0, 1]),
    "two_basis_atoms": dict(OPEN, basis=[[0, 0, 0], [0.5, 0.5, 0.5]], mu_s=[2.0, 1.0], n_basis_cells=[6, 5, 4],
                            n_shells_dmi=0, dij=[]),
    "no_pairs": dict(OPEN, n_shells_exchange=0, jij=[], n_shells_dmi=0, dij=[]),
}


@pytest.mark.parametrize("name", list(MODELS))
def test_parameter_terms(state, name):  # noqa: F811
    from spirit_amd import adjoint
    print("CASE adjoint parameters", name, flush=True)
    p = state(MODELS[name])
    sess = adjoint.Session(p, solver=2, n_steps=12, checkpoint_every=5)
    n = sess.nos
    rng = np.random.default_rng(11)
    s0, w = configs.random_spins(n, 4), rng.normal(size=(n, 3))
    sess.forward(s0)
    g = sess.backward(w)
    pairs = []
    for key, arg, m in [("J", "dJ", sess.n_exchange), ("D", "dD", sess.n_dmi), ("B", "dB", 1), ("K", "dK", sess.n_aniso)]:
        for k in range(m):
            d = np.zeros(m)
            d[k] = 1.0
            _, ds = sess.tangent(s0, np.zeros((n, 3)), **{arg: d})
            pairs.append((key, k, float(np.sum(w * ds)), float(g[key][k])))
    scale = max(abs(t) for _, _, t, _ in pairs)
    for key, k, t, a in pairs:
        print("  %s[%d] %.9e %.9e" % (key, k, t, a), flush=True)
        assert abs(t - a) <= 1e-9 * max(abs(t), abs(a), 1e-6 * scale), (key, k, t, a)
