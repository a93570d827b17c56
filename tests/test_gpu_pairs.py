"""Exchange and DMI over long or unequal pair tables (the offset-table loop and its fallback) against
the oracle: several shells, pairs reaching one to five cells, translations as long as the lattice,
periodic and open axes, two basis atoms, DMI pairs that are no exchange pairs.  Tolerances as the
other gradients': 1e-12 of the largest gradient (a sum of up to 40 products in another order),
energies 1e-11; 40 steps of the dynamics 1e-9."""
import numpy as np
import pytest

from test_gpu_parity import engine  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


def lattice(kind, cells, bc, **more):
    return dict(dict(bravais_lattice=kind, n_basis_cells=cells, boundary_conditions=bc, mu_s=[2.0],
                     external_field_magnitude=1.0, anisotropy_magnitude=0.2), **more)


SHELLS = dict(n_shells_exchange=3, jij=[5.0, 1.0, -0.5])
CASES = {
    "bcc_three_shells_periodic": lattice("bcc", [13, 9, 7], [1, 1, 1], **SHELLS),
    "fcc_dmi_open": lattice("fcc", [11, 6, 5], [0, 0, 0], n_shells_exchange=2, jij=[4.0, -1.0], n_shells_dmi=1,
                            dij=[0.7], dm_chirality=1),
    "sc_four_shells_mixed": lattice("sc", [9, 7, 5], [1, 0, 1], n_shells_exchange=4, jij=[3.0, 1.0, -1.0, 0.5],
                                    n_shells_dmi=2, dij=[0.7, 0.2], dm_chirality=2),
    "hex_dmi_more_than_exchange": lattice("hex2d", [17, 11, 1], [1, 1, 0], n_shells_exchange=1, jij=[4.0],
                                          n_shells_dmi=2, dij=[1.0, 0.5], dm_chirality=2),
    "two_basis_atoms": lattice("sc", [7, 6, 5], [1, 0, 1], basis=[[0, 0, 0], [0.5, 0.5, 0.5]], mu_s=[2.0, 1.0],
                               **SHELLS),
    "pairs_reach_three": lattice("sc", [8, 5, 4], [1, 1, 0], hamiltonian="heisenberg_pairs", pairs=[
        [0, 0, 3, 0, 0, 0.1, 0.2, 0.3, 1.5], [0, 0, 0, 3, 1, 0.0, 0.5, 0.0, -0.7], [0, 0, 1, 0, 0, 0.3, 0.0, 0.0, 4.0],
        [0, 0, 2, 2, 2, 0.0, 0.0, 0.0, 0.4]]),
    "pairs_reach_five": lattice("sc", [12, 6, 5], [1, 1, 0], hamiltonian="heisenberg_pairs", pairs=[
        [0, 0, 5, 0, 0, 0.1, 0.2, 0.3, 1.5], [0, 0, 0, 4, 1, 0.0, 0.5, 0.0, -0.7], [0, 0, 1, 0, 0, 0.3, 0.0, 0.0, 4.0]]),
    "pairs_as_long_as_the_lattice": lattice("sc", [3, 2, 1], [1, 0, 1], hamiltonian="heisenberg_pairs", pairs=[
        [0, 0, 3, 0, 0, 0.1, 0.2, 0.3, 1.5], [0, 0, 0, 2, 0, 0.0, 0.5, 0.0, -0.7], [0, 0, 0, 0, 1, 0.3, 0.0, 0.0, 4.0],
        [0, 0, 1, 1, 0, 0.3, 0.1, 0.0, 2.0]]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_pair_tables(engine, oracle, name):  # noqa: F811
    print("CASE pair tables", name, flush=True)
    cfg = CASES[name]
    e = engine(cfg)
    S = oracle.System(cfg)
    s = oracle.random_spins(S.nos, 5)
    e.set_spins(s)
    g, E = e.gradient()
    g0, E0 = S.gradient_and_energy(s)
    assert np.abs(g - g0).max() <= 1e-12 * np.abs(g0).max()
    assert abs(E - E0) <= 1e-11 * max(1.0, abs(E0))


@pytest.mark.parametrize("solver", [1, 2, 3, 4])
@pytest.mark.parametrize("name", ["bcc_three_shells_periodic", "sc_four_shells_mixed", "two_basis_atoms"])
def test_dynamics_over_pair_tables(engine, oracle, name, solver):  # noqa: F811
    from spirit_amd import simulation
    print("CASE pair tables dynamics", name, solver, flush=True)
    cfg = dict(CASES[name], llg_dt=1e-3, llg_damping=0.2, llg_force_convergence=1e-14)
    e = engine(cfg)
    S = oracle.System(cfg)
    s = oracle.random_spins(S.nos, 6)
    e.set_spins(s)
    simulation.start(e.p, simulation.METHOD_LLG, solver, single_shot=True)
    simulation.n_shot(e.p, 40)
    got = e.spins()
    simulation.stop(e.p)
    ref = S.llg(s, solver, 40, dt=1e-3, damping=0.2)
    assert np.abs(got - ref[0]).max() < 1e-9
