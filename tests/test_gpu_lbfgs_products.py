"""L-BFGS iterations whose direction comes from the products of the gradient and the memory: lattices of
fewer spins than a block, of a block more or less, and of more blocks (1027) than the kernel of the
products has, over ten iterations (the memory of three pairs fills, then wraps three times), against the
oracle's vector-by-vector recursion.  Tolerance as the other minimiser trajectories', 1e-9; the products'
partial sums of up to 8 10^5 terms leave 1e-13 of a coefficient."""
import numpy as np
import pytest

from test_gpu_minimisers import MINIMISERS, make_state, run_n  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

CELLS = [[3, 2, 1], [5, 17, 3], [16, 16, 1], [257, 1, 1], [512, 513, 1]]


@pytest.mark.parametrize("name", ["lbfgs_oso", "lbfgs_atlas"])
@pytest.mark.parametrize("cells", CELLS, ids=["x".join(map(str, c)) for c in CELLS])
def test_lbfgs_products(make_state, oracle, name, cells):  # noqa: F811
    print("CASE lbfgs products", name, cells, flush=True)
    cfg = dict(bravais_lattice="sc", n_basis_cells=cells, boundary_conditions=[1, 1, 0], mu_s=[2.0],
               external_field_magnitude=1.0, anisotropy_magnitude=0.2, n_shells_exchange=1, jij=[10.0],
               n_shells_dmi=1, dij=[3.0], dm_chirality=2, ddi_method="none", llg_dt=1e-3, llg_damping=0.3,
               llg_force_convergence=1e-14)
    p = make_state(cfg)
    S = oracle.System(cfg)
    s0 = oracle.random_spins(S.nos, 23)
    for n in (1, 2, 3, 10):
        s, _, _ = run_n(p, s0, MINIMISERS[name], n)
        ref, _, _, _ = S.llg(s0, MINIMISERS[name], n, dt=cfg["llg_dt"], damping=cfg["llg_damping"],
                             direct_minimization=True)
        assert np.abs(s - ref).max() <= 1e-9, (n, np.abs(s - ref).max())
