"""Every trial of a few Metropolis sweeps against the oracle's energies: the sweep is restated here with
the engine's counter-based random numbers (Philox4x32-10 of seed, step, colour and spin), each trial's
energy change is the difference of two whole-lattice energies of the oracle, and the engine's spins have
to be those of the restatement.  A decision that differs leaves one spin off by the whole move, so a wrong
factor in any term of the energy shows; decisions turn on the random number by less than the energies'
rounding (1e-13 of 1) once in 10^9 runs, moves differ by rounding alone (1e-15 each, bound 1e-11).  Short and long
pair tables, DMI pairs that are no exchange pairs, uniaxial, cubic and per-site anisotropy, open and
periodic axes, moves in a cone (fixed and adapted) and on the sphere."""
import itertools
import math

import numpy as np
import pytest

from test_gpu_parity import engine  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

K_B = 0.08617330350
M32 = 0xFFFFFFFF
SEED = 2006  # the default of mc_seed


def lattice(kind, cells, bc, **more):
    return dict(dict(bravais_lattice=kind, n_basis_cells=cells, boundary_conditions=bc, mu_s=[2.0],
                     external_field_magnitude=8.0, external_field_normal=[0.3, -0.4, 1.0], anisotropy_magnitude=0.0,
                     n_shells_exchange=0, n_shells_dmi=0), **more)


NN = dict(n_shells_exchange=1, jij=[1.0], n_shells_dmi=1, dij=[0.8], dm_chirality=1)
# configuration, pair translations (one of each +- pair), options of the moves, site anisotropy
CASES = {
    "nearest_neighbours": (lattice("sc", [6, 5, 4], [1, 0, 1], anisotropy_magnitude=1.5,
                                   anisotropy_normal=[0.2, 1, 0.5], **NN), None, {}),
    "bcc_two_shells": (lattice("bcc", [4, 5, 4], [1, 0, 1], n_shells_exchange=2, jij=[1.0, -0.7]), None, {}),
    "dmi_beyond_exchange": (lattice("sc", [6, 4, 4], [0, 0, 1], hamiltonian="heisenberg_pairs", pairs=[
        [0, 0, 1, 0, 0, 0, 0, 0, 1.0], [0, 0, 0, 1, 0, 0.6, 0.3, -0.9, 0.0], [0, 0, 3, 0, 0, 0.0, 0.7, 0.4, 0.0],
        [0, 0, 0, 0, 1, 0.5, 0, 0, 0.8]]), None, {}),
    "cubic": (lattice("sc", [5, 4, 4], [0, 1, 1], cubic_anisotropy_magnitude=4.0, **NN), None, {}),
    "site_anisotropy": (lattice("sc", [5, 5, 4], [0, 0, 1], site_anisotropy_normal=[0, 0.6, 0.8], **NN), "K", {}),
    "open_adaptive_cone": (lattice("sc", [4, 4, 5], [0, 0, 0], anisotropy_magnitude=1.0, **NN), None,
                           dict(adaptive=True)),
    "sphere": (lattice("sc", [4, 6, 4], [1, 1, 0], anisotropy_magnitude=1.0, **NN), None, dict(cone=False)),
}


def philox(c, seed):
    k0, k1 = seed & M32, seed >> 32
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [(p1 >> 32) ^ c[1] ^ k0, p1 & M32, (p0 >> 32) ^ c[3] ^ k1, p0 & M32]
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c


def uniforms(seed, step, colour, i):
    c = [i, colour | 0x40000000, step & M32, step >> 32]
    r = philox(list(c), seed) + philox([c[0], c[1] | 0x80000000, c[2], c[3]], seed)
    return [((r[k] >> 5) * 67108864.0 + (r[k + 1] >> 6)) / 9007199254740992.0 for k in (0, 2, 4, 6)]


def colouring(cells, bc, translations):
    """The first (K, c) with no pair inside a class (c . cell) mod K, K ascending."""
    for K in range(2, 9):
        for c in itertools.product(range(K), repeat=3):
            if any(bc[d] and cells[d] > 1 and c[d] * cells[d] % K for d in range(3)):
                continue
            if all(sum(c[d] * t[d] for d in range(3)) % K for t in translations):
                return K, c
    raise AssertionError("no colouring")


def trial(s, u, cone):
    ct = 1 - (1 - math.cos(cone)) * u[0] if cone is not None else u[0]
    st, phi = math.sqrt(1 - ct * ct), 2 * math.pi * u[1]
    local = np.array([st * math.cos(phi), st * math.sin(phi), ct])
    if cone is None:
        return local
    e0 = np.cross(s, [0.0, 0.0, 1.0])
    e0 /= np.linalg.norm(e0)
    return local[0] * e0 + local[1] * np.cross(s, e0) + local[2] * s


@pytest.mark.parametrize("name", list(CASES))
def test_trials_against_oracle_energies(engine, oracle, name):  # noqa: F811
    from spirit_amd import hamiltonian, simulation
    from spirit_amd.parameters import mc
    cfg, site, opt = CASES[name]
    cells, bc = cfg["n_basis_cells"], cfg["boundary_conditions"]
    print("CASE mc trials", name, flush=True)
    n = int(np.prod(cells))
    site_K = 3.0 * oracle.random_spins(n, 8)[:, 0] if site else None
    e = engine(cfg, site_K)
    S = oracle.System(cfg, site_K)
    s = oracle.random_spins(n, 9)
    e.set_spins(s)
    cone, adaptive, T, sweeps = opt.get("cone", True), opt.get("adaptive", False), 20.0, 4
    mc.set_temperature(e.p, T)
    mc.set_metropolis_cone(e.p, cone, 50.0, adaptive, 0.5)
    simulation.start(e.p, simulation.METHOD_MC, n_iterations=sweeps)
    got = e.spins()

    if cfg.get("hamiltonian") == "heisenberg_pairs":
        translations = [p[2:5] for p in cfg["pairs"]]
    else:
        translations = hamiltonian.get_exchange_pairs(e.p)[1].tolist()
    K, col = colouring(cells, bc, translations)
    angle = math.pi * 50.0 / 180.0
    rejected, decisions = 0, []
    _, E = S.gradient_and_energy(s)
    for step in range(sweeps):
        if adaptive:
            acc = 1 - rejected / n
            angle += 0.01 if acc > 0.5 else -0.01 if acc < 0.5 else 0.0
        rejected = 0
        for colour in range(K):
            for i in range(n):
                a, b, c = i % cells[0], i // cells[0] % cells[1], i // (cells[0] * cells[1])
                if (col[0] * a + col[1] * b + col[2] * c) % K != colour:
                    continue
                u = uniforms(SEED, step, colour, i)
                new = s.copy()
                new[i] = trial(s[i], u, angle if cone else None)
                _, E_new = S.gradient_and_energy(new)
                if E_new - E > 1e-14 and math.exp(-(E_new - E) / (K_B * T)) < u[2]:
                    rejected += 1
                    decisions.append(0)
                else:
                    s, E = new, E_new
                    decisions.append(1)
    assert 0.1 < np.mean(decisions) < 0.9  # both outcomes occur
    diff = np.abs(got - s).max(axis=1)
    assert diff.max() < 1e-11, "%d of %d spins differ" % ((diff > 1e-11).sum(), n)
