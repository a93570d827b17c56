"""The thermal field's normals (own logarithm of a uniform, sine and cosine of a multiple of pi) against
the oracle's: one step of free spins in a field (at rest a method would take no step) at a temperature
whose thermal rotation is of order one, so that the step shows the normals themselves.  20467 sites a
seed reach uniforms down to 5e-5 and up to 1 - 5e-5.  Tolerance: the oracle's normals are up to 6e-15 off (its rounded 2 pi u times the radius),
the engine's up to 3e-15; through xi + alpha s x xi with |f| < 1, the rotation and a normalisation this
is at most 3 times their sum, and 4e-15 for a dozen roundings of a unit vector."""
import numpy as np
import pytest

from test_gpu_parity import _run_llg, engine  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [1, 2, 3])
@pytest.mark.parametrize("seed", [1, 77, 2006])
def test_normals(engine, oracle, solver, seed):  # noqa: F811
    print("CASE normals", solver, seed, flush=True)
    cfg = dict(bravais_lattice="sc", n_basis_cells=[211, 97, 1], boundary_conditions=[1, 1, 0], mu_s=[2.0],
               external_field_magnitude=0.5, n_shells_exchange=0, n_shells_dmi=0, ddi_method="none", llg_dt=1e-3,
               llg_damping=0.3, llg_seed=seed, llg_temperature=1e4, llg_force_convergence=1e-14)
    e = engine(cfg)
    S = oracle.System(cfg)
    s0 = oracle.random_spins(S.nos, 3)
    e.set_spins(s0)
    s, _, _ = _run_llg(e, solver, 1)
    ref, _, _, _ = S.llg(s0, solver, 1, dt=1e-3, damping=0.3, temperature=1e4, seed=seed)
    moved = np.abs(ref - s0).max()
    err = np.abs(s - ref).max()
    print("  moved %.2f, max |s - s_oracle| = %.3e" % (moved, err), flush=True)
    assert moved > 0.5
    assert err <= 3 * 9e-15 + 4e-15
