"""An observed step's energy and torque, reduced by the last block of its last stage (lattices of up to
512 blocks of 256 spins, which arrive in groups of 64) or by a kernel of its own (larger ones, and batches
that hold one): lattices of 1, 2, 64, 65, 128, 129, 512 and 513 blocks, full and with few spins in the
last, alone and in batches with and without a larger one.  Both reductions add in the same order:
spins, energies and torques are equal, and the oracle's to 1e-9 (30 steps); the interface hands out
energy and torque in single precision, which adds at most 6e-8 of them to 1e-11 of the sum's up to
10 meV a spin and to 1e-9."""
import numpy as np
import pytest

from test_gpu_batch import replica_cfg, spins, states  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

CELLS = [[5, 3, 1], [16, 16, 1], [257, 1, 1], [128, 128, 1], [127, 130, 1], [256, 128, 1], [331, 99, 1],
         [256, 512, 1], [257, 511, 1]]


def replica(k, cells, T):
    return replica_cfg(1, 0.5 + 0.1 * k, T, 40 + k, n_basis_cells=cells)


@pytest.mark.parametrize("solver", [1, 2, 3, 4])
@pytest.mark.parametrize("T", [0.0, 10.0])
def test_reductions(states, oracle, solver, T):  # noqa: F811
    from spirit_amd import hip, simulation, system
    print("CASE fold", solver, T, flush=True)
    cfgs = [replica(k, c, T) for k, c in enumerate(CELLS)]
    lone, lone2, bat = states(cfgs), states(cfgs), states(cfgs)
    small = [p for p, c in zip(lone2, CELLS) if c[0] * c[1] <= 512 * 256]
    for p in lone:
        simulation.start(p, simulation.METHOD_LLG, solver, n_iterations=30)
    hip.llg_start_batch(bat, solver, n_iterations=30)
    hip.llg_start_batch(small, solver, n_iterations=30)
    for k, (a, b) in enumerate(zip(lone, bat)):
        np.testing.assert_array_equal(spins(a), spins(b))
        assert system.get_energy(a) == system.get_energy(b)
        assert simulation.get_max_torque_norm(a) == simulation.get_max_torque_norm(b)
        c = lone2[k]
        if c in small:
            np.testing.assert_array_equal(spins(a), spins(c))
            assert system.get_energy(a) == system.get_energy(c)
        S = oracle.System(cfgs[k])
        s0 = np.array(oracle.random_spins(S.nos, 7 + k))
        ref, E, torque, _ = S.llg(s0, solver, 30, dt=1e-3, damping=0.2, temperature=T, seed=40 + k)
        assert np.abs(spins(a) - ref).max() <= 1e-9
        assert abs(system.get_energy(a) - E) <= 1e-11 * S.nos * 10.0 + 6e-8 * abs(E)
        assert abs(simulation.get_max_torque_norm(a) - torque) <= 1e-9 + 6e-8 * torque
