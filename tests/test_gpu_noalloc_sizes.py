"""Spirit_HIP_Gradient_and_Energy_NoAlloc reads and writes arrays of spins, adds the energy in its gradient
kernel up to 128 blocks and beside it above, and keeps arrays that share memory apart: bit for bit
Spirit_HIP_Gradient_and_Energy over lattices at those edges (one spin; 128 and 129 blocks; more blocks
than the sum takes at a time), short and long pair tables, two basis atoms, twice in a row."""
import numpy as np
import pytest

from test_gpu_pairs import CASES as PAIR_CASES
from test_zz_no_alloc import SMALL, _state

pytestmark = pytest.mark.gpu


def sized(cells, **more):
    return dict(SMALL, bravais_lattice="sc", n_basis_cells=cells, **more)


CASES = dict(PAIR_CASES, one_spin=sized([1, 1, 1]), blocks_1=sized([16, 16, 1]), blocks_2=sized([257, 1, 1]),
             blocks_128=sized([128, 256, 1]), blocks_129=sized([331, 99, 1]), blocks_1025=sized([512, 513, 1]),
             long_blocks_129=sized([33, 32, 32], n_shells_exchange=2, jij=[10.0, 1.0]))


@pytest.mark.parametrize("shared", ["apart", "in_place", "energy_in_gradient", "energy_in_spins"])
@pytest.mark.parametrize("name", list(CASES))
def test_noalloc_sizes(tmp_path, name, shared):
    import torch

    from spirit_amd import hip, state, system
    print("CASE no-alloc", name, shared, flush=True)
    p = _state(tmp_path, CASES[name], "c.cfg")
    try:
        n = system.get_nos(p)
        rng = np.random.default_rng(3)
        for _ in range(2):
            s = rng.normal(size=(n, 3))
            s /= np.linalg.norm(s, axis=1)[:, None]
            system.get_spin_directions(p)[:] = s
            g_ref, e_ref = hip.gradient_and_energy(p, n)
            s_d = torch.tensor(s, device="cuda:0")
            g_d = s_d if shared == "in_place" else torch.full((n, 3), float("nan"), dtype=torch.float64, device="cuda:0")
            e_d = torch.full((1,), float("nan"), dtype=torch.float64, device="cuda:0")
            at = {"energy_in_gradient": g_d, "energy_in_spins": s_d}.get(shared, e_d)
            rc = hip.gradient_and_energy_noalloc(p, s_d.data_ptr(), g_d.data_ptr(), at.data_ptr(),
                                                 torch.cuda.current_stream().cuda_stream)
            assert rc == 0
            assert float(at.reshape(-1)[0].item()) == e_ref
            g = g_d.cpu().numpy()
            if shared == "energy_in_gradient":
                g[0, 0] = g_ref[0, 0]
            assert np.array_equal(g, g_ref)
    finally:
        state.delete(p)
