"""The measured work of the engine: what its users run, through the public entry points.

Each case is one call (or one short sequence of calls) of a user's program on a lattice of the
sizes this repository is configured, tested and benchmarked with:

* ``gradient``  one effective-field evaluation of spins the caller holds on the GPU (a caller's
                own solver or serving loop), hip.gradient_and_energy_noalloc;
* ``llg``       steps of LLG dynamics from a disordered state, simulation.n_shot of a started
                method, then the spins and the effective field: monolayers, films and bulk, with
                and without the dipolar FFT field, every solver, T = 0 and T > 0;
* ``minimise``  LBFGS_OSO direct minimisation, simulation.n_shot;
* ``mc``        Metropolis sweeps, simulation.n_shot;
* ``gneb``      a minimum-energy-path calculation, simulation.start;
* ``ensemble``  independent thermal replicas of uneven sizes, hip.llg_start_batch;
* ``adjoint``   a differentiable run: forward with checkpoints, then the gradients of a loss,
                adjoint.Session.

All arithmetic is FP64, as the engine's only precision.  ``exact`` restates each of them in
plain torch, without the engine.
"""
import math
import os
import shutil
import tempfile

import numpy as np
import torch

# Physical constants of the model (meV, T, ps, K, Angstrom)
MU_B, MU_0, K_B, GAMMA = 0.057883817555, 2.0133545e-28, 0.08617330350, 0.1760859644

SOLVERS = {"sib": 1, "depondt": 2, "heun": 3, "rk4": 4}
EVALS = {"sib": 2, "depondt": 2, "heun": 2, "rk4": 4}
# vector fields read or written per spin and step that no order of the stages avoids: every
# evaluation reads a configuration and every stage writes the next; Depondt and Heun keep the first
# virtual force for the corrector, which also reads the old spins; RK4 carries an accumulator
FIELDS = {"sib": 5, "depondt": 7, "heun": 7, "rk4": 17}

BRAVAIS = {
    "sc": ((1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (0.0, 0.0, 1.0)),
    "bcc": ((0.5, 0.5, -0.5), (-0.5, 0.5, -0.5), (0.5, -0.5, -0.5)),
    "fcc": ((0.5, 0.0, 0.5), (0.5, 0.5, 0.0), (0.0, 0.5, 0.5)),
    "hex2d": ((0.5 * math.sqrt(3.0), -0.5, 0.0), (0.5 * math.sqrt(3.0), 0.5, 0.0), (0.0, 0.0, 1.0)),
}
SHELL_J = (10.0, 2.0, -1.0)  # meV per exchange shell


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _lattice(na, nb, nc, lattice="sc", basis=1, bc="000", shells=1, D=1.0, chirality=1, K=0.0, B=0.5, site_K=False):
    return dict(na=na, nb=nb, nc=nc, lattice=lattice, basis=basis, bc=bc, shells=shells, D=D, chirality=chirality,
                K=K, B=B, site_K=site_K)


def listed():
    return [
        # one field evaluation of the smallest usual monolayer: launches and host work
        dict(_lattice(64, 64, 1, bc="110", D=6.0, chirality=2, K=0.2, B=2.0), name="gradient_square64",
             kind="gradient"),
        # the monolayer every first run of a user starts with: two tiny kernels a step
        dict(_lattice(64, 64, 1, bc="110", D=6.0, chirality=2, K=0.2, B=2.0), name="square64_depondt", kind="llg",
             solver="depondt", steps=200, dt=1e-3, damping=0.3, T=0.0, ddi="none"),
        # a bulk crystal with exchange to the third shell (8 + 6 + 12 neighbours), odd sizes, periodic
        dict(_lattice(97, 90, 85, lattice="bcc", bc="111", shells=3, D=0.0, K=0.1), name="bcc97_sib_3shells",
             kind="llg", solver="sib", steps=40, dt=1e-3, damping=0.2, T=0.0, ddi="none"),
        # the dipolar film of the benchmark's second workload: Heun at 10 K
        dict(_lattice(128, 128, 32, K=0.05), name="film128_heun_ddi", kind="llg", solver="heun", steps=50, dt=5e-4,
             damping=0.1, T=10.0, ddi="fft", images=0, padding=True),
        # the headline workload: per-site anisotropy, open cube, padded 512x512x256
        dict(_lattice(256, 256, 128, B=0.2, site_K=True), name="cube256_depondt_ddi", kind="llg", solver="depondt",
             steps=50, dt=5e-4, damping=0.3, T=0.0, ddi="fft", images=0, padding=True),
        # a film of a sample's own size: padded 400x300x24, no power of two
        dict(_lattice(200, 150, 12, K=0.05), name="film200x150_depondt_ddi", kind="llg", solver="depondt", steps=40,
             dt=5e-4, damping=0.3, T=0.0, ddi="fft", images=0, padding=True),
        # a dipolar monolayer, periodic in the plane with images, as skyrmion films are run
        dict(_lattice(500, 500, 1, bc="110", D=3.0, chirality=2, K=0.4), name="monolayer500_rk4_ddi", kind="llg",
             solver="rk4", steps=25, dt=1e-3, damping=0.3, T=0.0, ddi="fft", images=4, padding=True),
        # relaxation of a dipolar film by L-BFGS
        dict(_lattice(256, 256, 16, K=0.05), name="film256_lbfgs_ddi", kind="minimise", steps=50, dt=1e-3,
             ddi="fft", images=0, padding=True),
        # thermal equilibrium of a bulk magnet
        dict(_lattice(128, 128, 64, bc="111", K=0.05), name="bulk128_metropolis", kind="mc", steps=50, T=10.0),
        # skyrmion collapse: 32 images of the hexagonal monolayer, climbing image
        dict(_lattice(128, 128, 1, lattice="hex2d", bc="110", D=6.0, chirality=2, K=0.4, B=3.0),
             name="gneb32_hex128_vp", kind="gneb", images=32, steps=100, dt=1e-5),
        # 48 stochastic replicas of uneven sizes in one call
        dict(name="ensemble48_depondt", kind="ensemble", replicas=48, smallest=32, largest=256, steps=200, dt=1e-3,
             damping=0.2, solver="depondt"),
        # parameter fitting: a differentiable run of a dipolar film, forward and backward
        dict(_lattice(128, 128, 16, B=0.2, site_K=True), name="film128_adjoint_ddi", kind="adjoint", solver="depondt",
             steps=20, checkpoint=10, dt=5e-4, damping=0.3, ddi="fft", images=0, padding=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("gradient", "llg", "llg", "ddi", "ddi", "ddi", "minimise", "mc", "gneb", "ensemble", "adjoint"))
    if kind == "gradient":
        if rng.random() < 0.5:
            return dict(_lattice(_log(rng, 20, 700), _log(rng, 20, 700), 1, lattice=rng.choice(("sc", "hex2d")),
                                 bc=rng.choice(("110", "000")), D=6.0, chirality=2, K=0.2, B=2.0), kind=kind)
        return dict(_lattice(_log(rng, 8, 100), _log(rng, 8, 100), _log(rng, 4, 90),
                             lattice=rng.choice(("sc", "bcc", "fcc")), bc=rng.choice(("111", "000")),
                             shells=rng.randint(1, 3), K=0.1), kind=kind)
    dyn = dict(dt=5e-4, damping=round(rng.uniform(0.05, 0.5), 3))
    if kind == "llg":
        dyn.update(kind="llg", solver=rng.choice(sorted(SOLVERS)), T=rng.choice((0.0, 10.0)), ddi="none")
        if rng.random() < 0.5:
            na, nb = _log(rng, 24, 1000), _log(rng, 24, 1000)
            c = dict(_lattice(na, nb, 1, lattice=rng.choice(("sc", "hex2d")), bc=rng.choice(("110", "000", "100")),
                              shells=rng.randint(1, 3), D=3.0, chirality=2, K=0.2, B=1.0), **dyn)
        else:
            na, nb, nc = _log(rng, 12, 200), _log(rng, 12, 200), _log(rng, 4, 100)
            lattice, basis = rng.choice((("sc", 1), ("sc", 2), ("bcc", 1), ("fcc", 1)))
            c = dict(_lattice(na, nb, nc, lattice=lattice, basis=basis, bc=rng.choice(("111", "000", "110")), shells=rng.randint(1, 3),
                              D=rng.choice((0.0, 1.0)), K=0.1, site_K=rng.random() < 0.25), **dyn)
        c["steps"] = max(5, min(200, int(2.5e7 / (_nos(c) * EVALS[c["solver"]]))))
        return c
    # lengths whose padded double the transforms take (prime factors to 13), odd ones among them
    smooth = [n for n in range(10, 257) if _largest_prime(n) <= 13]

    def near(lo, hi):
        n = _log(rng, lo, hi)
        return min(smooth, key=lambda m: abs(m - n))

    if kind in ("ddi", "minimise", "adjoint"):
        shape = rng.random()
        if shape < 0.3:
            na, nb, nc = near(40, 256), near(40, 256), rng.choice((1, 1, 2, 3))
        elif shape < 0.7:
            na, nb, nc = near(24, 200), near(24, 200), rng.choice((4, 5, 6, 8, 10, 16, 21, 32))
        else:
            na, nb, nc = near(16, 110), near(16, 110), near(16, 110)
        bc = rng.choice(("000", "000", "110"))
        c = _lattice(na, nb, nc, bc=bc, K=0.05, basis=2 if kind == "ddi" and rng.random() < 0.15 else 1)
        c.update(ddi="fft", images=rng.choice((0, 2)) if bc == "110" else 0, padding=rng.random() < 0.8)
    if kind == "ddi":
        c.update(dyn, kind="llg", solver=rng.choice(sorted(SOLVERS)), T=rng.choice((0.0, 0.0, 10.0)))
        c["steps"] = max(5, min(60, int(1.5e7 / (_nos(c) * EVALS[c["solver"]]))))
    elif kind == "minimise":
        c.update(kind=kind, steps=max(6, min(60, int(1.5e7 / _nos(c)))), dt=1e-3)
    elif kind == "adjoint":
        c.update(dyn, kind=kind, solver=rng.choice(("depondt", "heun")), site_K=True, basis=1,
                 steps=max(4, min(24, int(5e6 / _nos(c)))))
        c["checkpoint"] = max(2, c["steps"] // 2)
    elif kind == "mc":
        bc = rng.choice(("111", "000"))
        even = 2 if bc == "111" else 1
        size = lambda lo, hi: max(even, _log(rng, lo, hi) // even * even)  # noqa: E731
        c = dict(_lattice(size(16, 200), size(16, 200), size(2, 80), bc=bc, K=0.05), kind=kind, T=rng.choice((1.0, 10.0, 50.0)))
        c["steps"] = max(5, min(100, int(5e7 / _nos(c))))
    elif kind == "gneb":
        n = _log(rng, 24, 160)
        c = dict(_lattice(n, _log(rng, 24, 160), 1, lattice=rng.choice(("sc", "hex2d")), bc="110", D=6.0, chirality=2,
                          K=0.4, B=3.0), kind=kind, images=rng.randint(5, 32), dt=1e-5)
        c["steps"] = rng.randint(40, 100)
    elif kind == "ensemble":
        c = dict(kind=kind, replicas=rng.randint(2, 48), smallest=rng.choice((24, 32, 48)), largest=rng.choice((64, 100, 200)),
                 steps=rng.randint(60, 200), dt=1e-3, damping=0.2, solver=rng.choice(("depondt", "heun")))
    return c


def _largest_prime(n):
    p, d = 1, 2
    while n > 1:
        while n % d == 0:
            n, p = n // d, d
        d += 1
    return p


def _nos(case):
    return case["na"] * case["nb"] * case["nc"] * case["basis"]


def _replicas(case):
    """(sides, fields [T], temperatures [K]) of an ensemble's replicas; the lattice sizes belong to the case."""
    rng = np.random.default_rng(case["replicas"])
    sides = np.unique(np.round(np.geomspace(case["smallest"], case["largest"], 7)).astype(int) // 2 * 2)
    return (rng.choice(sides, case["replicas"]), rng.uniform(0.0, 2.0, case["replicas"]),
            rng.uniform(1.0, 50.0, case["replicas"]))


def _padded(case):
    P = []
    for k, n in enumerate((case["na"], case["nb"], case["nc"])):
        pad = n > 1 and (case["bc"][k] == "0" or case["padding"])
        P.append(2 * n if pad else n)
    return P


def work(case):
    """Bytes: per step the vector fields FIELDS names (24 B a spin each), and per dipolar field evaluation one round trip
    of the spectrum of the c < Nc planes each way, the spins, the field and one read of the kernel spectrum of an octant;
    whatever a call brings to the host is written once.  Flops: 12 a pair and evaluation, 2.5 M log2 M a real transform."""
    if case["kind"] == "ensemble":
        sides, _, _ = _replicas(case)
        n = int((sides.astype(np.int64) ** 2).sum())
        return {"bytes": 24.0 * n * (FIELDS[case["solver"]] * case["steps"] + 2), "flops": 2.0 * case["steps"] * n * 150}
    n = _nos(case)
    pairs = len(_pairs(case)[0]) / case["basis"]
    dip_b = dip_f = 0.0
    if case.get("ddi") == "fft":
        Pa, Pb, Pc = _padded(case)
        Ha = Pa // 2 + 1
        M = float(Pa) * Pb * Pc
        kernel = 48.0 * case["basis"] ** 2 * Ha * (Pb // 2 + 1) * (Pc // 2 + 1)
        dip_b = 48.0 * n + 4 * 48.0 * case["basis"] * Ha * Pb * case["nc"] + kernel
        dip_f = 6 * case["basis"] * 2.5 * M * math.log2(max(M, 2.0)) + 15.0 * M * case["basis"] ** 2
    local_f = n * (12.0 * pairs + 60)
    kind = case["kind"]
    if kind == "gradient":
        return {"bytes": 48.0 * n, "flops": local_f}
    if kind == "llg":
        ev = EVALS[case["solver"]]
        return {"bytes": case["steps"] * (24.0 * n * FIELDS[case["solver"]] + ev * dip_b) + 48.0 * n,
                "flops": case["steps"] * ev * (local_f + dip_f)}
    if kind == "minimise":
        # spins, gradient, search direction and three pairs of the L-BFGS memory read, six fields written
        return {"bytes": case["steps"] * (24.0 * n * 15 + dip_b) + 48.0 * n, "flops": case["steps"] * (local_f + dip_f + 60.0 * n)}
    if kind == "mc":
        return {"bytes": 48.0 * n * case["steps"], "flops": case["steps"] * n * (24.0 * pairs + 200)}
    if kind == "gneb":
        n *= case["images"]
        return {"bytes": case["steps"] * 24.0 * n * 8, "flops": case["steps"] * n * (12.0 * pairs + 200)}
    # adjoint: the run, the run again with its tape, and the transposed steps, each two evaluations
    return {"bytes": case["steps"] * (3 * (24.0 * n * 7 + 2 * dip_b)) + 96.0 * n, "flops": case["steps"] * 6 * (local_f + dip_f)}


def tolerance(case):
    # all arithmetic is FP64: against `exact` the spins, fields and gradients differ by 1e-16 to 6e-15 over the declared ranges (sums
    # in another order, another factorisation of the transforms); the L-BFGS recursion and the band's springs and tangents divide by
    # small differences and amplify that a few hundred times over their iterations
    if case["kind"] in ("minimise", "gneb"):
        return {"rel": 1e-10, "max": 1e-7}
    if case["kind"] == "adjoint":
        return {"rel": 1e-12, "max": 1e-10}
    return {"rel": 1e-13, "max": 1e-10}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _random_spins(n, gen):
    """n directions, uniform on the sphere, on the GPU."""
    u = torch.rand((2, n), dtype=torch.float64, device="cuda", generator=gen)
    z = 2 * u[0] - 1
    phi = 2 * math.pi * u[1]
    r = torch.sqrt(torch.clamp(1 - z * z, min=0.0))
    return torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], dim=1)


def _inputs(case, seed):
    """What the case's arrays are, on the GPU: spins, per-site anisotropy, loss target."""
    gen = _generator(seed)
    if case["kind"] == "ensemble":
        sides, _, _ = _replicas(case)
        return {"spins": [_random_spins(int(L) * int(L), gen) for L in sides]}
    if case["kind"] == "gneb":
        return {"spins": _collapse_path(case, gen)}
    n = _nos(case)
    got = {"spins": _random_spins(n, gen)}
    if case["site_K"]:
        got["site_K"] = 0.02 + 0.08 * torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
    if case["kind"] == "adjoint":
        got["target"] = _random_spins(n, gen)
    return got


def _collapse_path(case, gen):
    """images x spins: a Neel skyrmion whose radius shrinks along the path to the ferromagnet, each inner image
    displaced a little, as after an interpolation with noise.  (The cases' small time step keeps the iteration of a
    dense band from amplifying rounding: at 1e-4 ps it multiplies a difference by 1e10 in 100 iterations, at 1e-5 ps by 1e3
    in 200.)"""
    a1, a2 = BRAVAIS[case["lattice"]][:2]
    ia = torch.arange(case["na"], dtype=torch.float64, device="cuda")[None, :]
    ib = torch.arange(case["nb"], dtype=torch.float64, device="cuda")[:, None]
    x = ((ia - case["na"] / 2) * a1[0] + (ib - case["nb"] / 2) * a2[0]).reshape(-1)
    y = ((ia - case["na"] / 2) * a1[1] + (ib - case["nb"] / 2) * a2[1]).reshape(-1)
    r, phi = torch.sqrt(x * x + y * y), torch.atan2(y, x)
    path = []
    for k in range(case["images"]):
        f = 1 - k / (case["images"] - 1)
        theta = f * 2 * torch.atan2(torch.sinh(torch.tensor(8.0 / 3.0, dtype=torch.float64, device="cuda")), torch.sinh(r / 3.0))
        s = torch.stack([torch.sin(theta) * torch.cos(phi), torch.sin(theta) * torch.sin(phi), torch.cos(theta)], dim=1)
        if 0 < k < case["images"] - 1:
            s = s + 0.02 * torch.randn(s.shape, dtype=torch.float64, device="cuda", generator=gen)
            s = s / s.norm(dim=1, keepdim=True)
        path.append(s)
    return path


def _config(case, seed, **more):
    """The engine's input keywords of the case."""
    images = [case["images"] if case["bc"][k] == "1" else 0 for k in range(3)] if case.get("ddi") == "fft" else [0, 0, 0]
    cfg = dict(bravais_lattice=case["lattice"], n_basis_cells=[case["na"], case["nb"], case["nc"]],
               boundary_conditions=[int(c) for c in case["bc"]], mu_s=[2.0] * case["basis"],
               external_field_magnitude=case["B"], external_field_normal=[0, 0, 1], anisotropy_magnitude=case["K"],
               anisotropy_normal=[0, 0, 1], n_shells_exchange=case["shells"], jij=list(SHELL_J[: case["shells"]]),
               n_shells_dmi=1 if case["D"] else 0, dij=[case["D"]] if case["D"] else [], dm_chirality=case["chirality"],
               ddi_method=case.get("ddi", "none"), ddi_n_periodic_images=images,
               ddi_pb_zero_padding=1 if case.get("padding", True) else 0, llg_dt=case.get("dt", 1e-3),
               llg_damping=case.get("damping", 0.3), llg_temperature=case.get("T", 0.0), llg_seed=_noise_seed(seed),
               llg_n_iterations=2000000000, llg_force_convergence=1e-14, gneb_force_convergence=1e-14,
               gneb_spring_constant=1.0)
    if case["basis"] == 2:
        cfg["basis"] = [[0, 0, 0], [0.5, 0.5, 0.5]]
    cfg.update(more)
    return cfg


def _noise_seed(seed):
    return int(seed) % 1000000 + 1


class _State:
    """What a user's program holds: the engine's state (deleted with this object) and device arrays."""

    def __init__(self, case):
        self.case, self.handles, self.session = case, [], None

    def add(self, cfg, extra=""):
        from spirit_amd import configs, state
        folder = tempfile.mkdtemp(prefix="spirit_case_")
        try:
            path = os.path.join(folder, "input.cfg")
            with open(path, "w") as f:
                f.write(configs.config_text(cfg) + extra)
            p = state.setup(path, True)
        finally:
            shutil.rmtree(folder, ignore_errors=True)
        if not p:
            raise RuntimeError("State_Setup failed")
        self.handles.append(p)
        return p

    def __del__(self):
        from spirit_amd import simulation, state
        if self.session is not None:
            self.session.close()
        for p in self.handles:
            if simulation.running_anywhere_on_chain(p):
                simulation.stop(p)
            state.delete(p)


class _View(np.ndarray):
    """One of the engine's host arrays, which lives as long as the state it belongs to: holds on to that."""

    state = None


def _spins(st, p, **where):
    from spirit_amd import system
    v = system.get_spin_directions(p, **where).view(_View)
    v.state = st
    return v


def _field(st, p):
    from spirit_amd import system
    v = system.get_effective_field(p).view(_View)
    v.state = st
    return v


def prepare(case, seed):
    from spirit_amd import adjoint, chain, hip, simulation, system
    from spirit_amd.parameters import gneb, mc
    st = _State(case)
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "ensemble":
        sides, fields, temps = _replicas(case)
        for k, (L, B, T) in enumerate(zip(sides, fields, temps)):
            rep = _lattice(int(L), int(L), 1, bc="110", D=3.0, chirality=2, K=0.1, B=float(B))
            p = st.add(_config(dict(rep, dt=case["dt"], damping=case["damping"], T=float(T)), seed + 1000 * k))
            system.get_spin_directions(p)[:] = inp["spins"][k].cpu().numpy()
        return st
    p = st.add(_config(case, seed), "mc_seed %d\n" % _noise_seed(seed) if kind == "mc" else "")
    if kind == "gneb":
        chain.image_to_clipboard(p)
        for _ in range(case["images"] - 1):
            chain.insert_image_after(p)
        for k, s in enumerate(inp["spins"]):
            system.get_spin_directions(p, idx_image=k)[:] = s.cpu().numpy()
        gneb.set_climbing_falling(p, 1, idx_image=_climbing(case))
        return st
    if case["site_K"]:
        hip.set_site_anisotropy(p, inp["site_K"].cpu().numpy(), (0.0, 0.0, 1.0))
    if kind == "gradient":
        st.spins = inp["spins"].contiguous()
        st.gradient = torch.empty_like(st.spins)
        st.energy = torch.empty(1, dtype=torch.float64, device="cuda")
        return st
    system.get_spin_directions(p)[:] = inp["spins"].cpu().numpy()
    if kind == "llg":
        simulation.start(p, simulation.METHOD_LLG, SOLVERS[case["solver"]], single_shot=True)
    elif kind == "minimise":
        simulation.start(p, simulation.METHOD_LLG, simulation.SOLVER_LBFGS_OSO, single_shot=True)
    elif kind == "mc":
        mc.set_iterations(p, 2000000000, 2000000000)
        mc.set_temperature(p, case["T"])
        mc.set_metropolis_cone(p, True, 30.0, True, 0.5)
        simulation.start(p, simulation.METHOD_MC, single_shot=True)
    elif kind == "adjoint":
        st.session = adjoint.Session(p, solver=SOLVERS[case["solver"]], n_steps=case["steps"],
                                     checkpoint_every=case["checkpoint"])
        st.spins, st.target = inp["spins"], inp["target"]
    return st


def _climbing(case):
    return case["images"] // 2


def run(st):
    from spirit_amd import hip, simulation
    case, kind = st.case, st.case["kind"]
    p = st.handles[0]
    if kind == "gradient":
        rc = hip.gradient_and_energy_noalloc(p, st.spins.data_ptr(), st.gradient.data_ptr(), st.energy.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError("Spirit_HIP_Gradient_and_Energy_NoAlloc failed")
        return {"gradient": st.gradient, "energy": st.energy}
    if kind in ("llg", "minimise"):
        simulation.n_shot(p, case["steps"])
        return {"spins": _spins(st, p), "field": _field(st, p)}
    if kind == "mc":
        simulation.n_shot(p, case["steps"])
        return {"spins": _spins(st, p)}
    if kind == "gneb":
        simulation.start(p, simulation.METHOD_GNEB, simulation.SOLVER_VP, n_iterations=case["steps"])
        return [_spins(st, p, idx_image=k) for k in range(case["images"])]
    if kind == "ensemble":
        hip.llg_start_batch(st.handles, SOLVERS[case["solver"]], n_iterations=case["steps"])
        return [_spins(st, q) for q in st.handles]
    sN = st.session.forward(st.spins)
    g = st.session.backward(2.0 * (sN - st.target) / sN.shape[0])
    return {"spins": sN, "d_spins": g["s0"], "d_J": g["J"], "d_D": g["D"], "d_B": g["B"], "d_K_site": g["K_site"]}


# ---------------------------------------------------------------------------
# the same in plain torch (FP64)
# ---------------------------------------------------------------------------
def _pairs(case):
    """(exchange pairs, DMI pairs) as (i, j, (ta, tb, tc), shell, unit vector i -> j): all neighbours of each basis
    atom in the case's shells, along the directions that hold more than one cell."""
    br = np.array(BRAVAIS[case["lattice"]])
    atoms = [np.zeros(3), np.full(3, 0.5)][: case["basis"]]
    n = (case["na"], case["nb"], case["nc"])
    reach = [min(case["shells"] + 2, m - 1) for m in n]
    found = []
    for i, pi in enumerate(atoms):
        for ta in range(-reach[0], reach[0] + 1):
            for tb in range(-reach[1], reach[1] + 1):
                for tc in range(-reach[2], reach[2] + 1):
                    for j, pj in enumerate(atoms):
                        if i == j and ta == tb == tc == 0:
                            continue
                        # shells are ordered by the distance with the basis offset in Cartesian units
                        d = pj - pi + ta * br[0] + tb * br[1] + tc * br[2]
                        real = (pj[0] - pi[0] + ta) * br[0] + (pj[1] - pi[1] + tb) * br[1] + (pj[2] - pi[2] + tc) * br[2]
                        found.append((float(np.linalg.norm(d)), i, j, (ta, tb, tc), real))
    radii = []
    for d in sorted(f[0] for f in found):
        if not radii or d - radii[-1] > 1e-3:
            radii.append(d)
    exch = [(i, j, t, s, r / np.linalg.norm(r)) for s in range(case["shells"])
            for d, i, j, t, r in found if abs(d - radii[s]) < 1e-3]
    dmi = [p for p in exch if p[3] == 0] if case["D"] else []
    return exch, dmi


def _dmi_normal(unit, chirality):
    return np.array(unit) if chirality == 1 else np.cross(unit, (0.0, 0.0, 1.0))


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=-1)


def _dot(a, b):
    return (a * b).sum(dim=-1, keepdim=True)


def _unit(a):
    return a / torch.sqrt(_dot(a, a))


class _Model:
    """Gradient and energy of the case's Hamiltonian on spins shaped (..., Nc, Nb, Na, basis, 3)."""

    def __init__(self, case, site_K=None, B=None):
        self.case = case
        self.shape = (case["nc"], case["nb"], case["na"], case["basis"], 3)
        self.exch, self.dmi = _pairs(case)
        self.J = [torch.tensor(v, dtype=torch.float64, device="cuda") for v in SHELL_J[: case["shells"]]]
        self.D = torch.tensor(float(case["D"]), dtype=torch.float64, device="cuda")
        self.B = torch.tensor(float(case["B"] if B is None else B), dtype=torch.float64, device="cuda")
        self.site_K = None if site_K is None else site_K.reshape(self.shape[:-1])
        self.mu = 2.0
        self.z = torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64, device="cuda")
        self.dipole = self._dipole() if case.get("ddi") == "fft" else None

    def neighbour(self, s, j, t):
        """Basis atom j of the cell shifted by t; zero beyond an open boundary."""
        x = s[..., j, :]
        for axis, shift, n, k in ((-2, t[0], self.case["na"], 0), (-3, t[1], self.case["nb"], 1),
                                  (-4, t[2], self.case["nc"], 2)):
            if shift == 0:
                continue
            x = torch.roll(x, -shift, dims=axis)
            if self.case["bc"][k] == "0":
                keep = torch.ones(n, dtype=torch.float64, device="cuda")
                if shift > 0:
                    keep[max(0, n - shift):] = 0
                else:
                    keep[: min(n, -shift)] = 0
                x = x * keep.reshape((n,) + (1,) * (-axis - 1))
        return x

    def _dipole(self):
        """Spectra of the dipole tensor, [b1][b2] -> six components on the half grid."""
        c = self.case
        P, N = _padded(c), (c["na"], c["nb"], c["nc"])
        img = [c["images"] if c["bc"][k] == "1" else 0 for k in range(3)]
        br = torch.tensor(BRAVAIS[c["lattice"]], dtype=torch.float64, device="cuda")
        mult = MU_0 * MU_B * MU_B / (4 * math.pi * 1e-30)
        idx = [torch.arange(P[k], device="cuda", dtype=torch.float64) for k in range(3)]
        idx = [torch.where(i < N[k], i, i - P[k]) for k, i in enumerate(idx)]
        out = {}
        for b1 in range(c["basis"]):
            for b2 in range(c["basis"]):
                off = 0.5 * (b1 - b2)
                comp = [torch.zeros((P[2], P[1], P[0]), dtype=torch.float64, device="cuda") for _ in range(6)]
                for pa in range(-img[0], img[0] + 1):
                    for pb in range(-img[1], img[1] + 1):
                        for pc in range(-img[2], img[2] + 1):
                            f = [(idx[0] + pa * N[0] + off)[None, None, :], (idx[1] + pb * N[1] + off)[None, :, None],
                                 (idx[2] + pc * N[2] + off)[:, None, None]]
                            r = [f[0] * br[0][q] + f[1] * br[1][q] + f[2] * br[2][q] for q in range(3)]
                            d2 = r[0] ** 2 + r[1] ** 2 + r[2] ** 2
                            ok = d2 > 1e-20
                            d2 = torch.where(ok, d2, torch.ones_like(d2))
                            i3 = torch.where(ok, mult / (d2 * torch.sqrt(d2)), torch.zeros_like(d2))
                            i5 = 3 * i3 / d2
                            k = 0
                            for q in range(3):
                                for w in range(q, 3):
                                    comp[k] += i5 * r[q] * r[w]
                                    if q == w:
                                        comp[k] -= i3
                                    k += 1
                out[b1, b2] = [torch.fft.rfftn(x) for x in comp]
        return out

    def dipolar(self, s):
        c = self.case
        P = _padded(c)
        size = (P[2], P[1], P[0])
        S = [[torch.fft.rfftn(self.mu * s[..., b, q], s=size, dim=(-3, -2, -1)) for q in range(3)] for b in range(c["basis"])]
        rows = ((0, 1, 2), (1, 3, 4), (2, 4, 5))
        h = []
        for b1 in range(c["basis"]):
            comp = []
            for q in range(3):
                X = sum(self.dipole[b1, b2][rows[q][w]] * S[b2][w] for b2 in range(c["basis"]) for w in range(3))
                comp.append(self.mu * torch.fft.irfftn(X, s=size, dim=(-3, -2, -1))[..., : c["nc"], : c["nb"], : c["na"]])
            h.append(torch.stack(comp, dim=-1))
        return torch.stack(h, dim=-2)

    def force(self, s, energy=False):
        """-dE/ds of spins (..., n, 3), and the energy of each configuration."""
        x = s.reshape(s.shape[:-2] + self.shape)
        f = [torch.zeros_like(x[..., 0, :]) for _ in range(self.case["basis"])]
        for i, j, t, shell, _ in self.exch:
            f[i] = f[i] + self.J[shell] * self.neighbour(x, j, t)
        for i, j, t, _, unit in self.dmi:
            n = torch.tensor(_dmi_normal(unit, self.case["chirality"]), dtype=torch.float64, device="cuda")
            y = self.neighbour(x, j, t)
            f[i] = f[i] + self.D * _cross(y, n.expand_as(y))
        f = torch.stack(f, dim=-2)
        if self.case["K"]:
            f = f + 2 * self.case["K"] * x[..., 2:3] * self.z
        if self.site_K is not None:
            f = f + 2 * (self.site_K * x[..., 2])[..., None] * self.z
        if self.dipole is not None:
            f = f + self.dipolar(x)
        e = None
        if energy:
            e = (-0.5 * (f * x)).sum(dim=(-1, -2, -3, -4, -5)) - (self.mu * self.B * MU_B) * x[..., 2].sum(dim=(-1, -2, -3, -4))
        f = f + self.mu * self.B * MU_B * self.z
        return f.reshape(s.shape), e


# Philox4x32-10 on int64 tensors, for the engine's counter-based random numbers
_M32 = 0xFFFFFFFF


def _philox(c, seed):
    k0, k1 = seed & _M32, (seed >> 32) & _M32
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & _M32) ^ c[1] ^ k0, p1 & _M32, ((p0 >> 32) & _M32) ^ c[3] ^ k1, p0 & _M32]
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return c


def _uniform(a, b):
    return ((a >> 5).double() * 67108864.0 + (b >> 6).double()) / 9007199254740992.0


def _uniforms(n, second, step, seed):
    """Four uniform numbers for each of n sites; `second` is the counter's second word."""
    i = torch.arange(n, device="cuda", dtype=torch.int64)
    w = torch.full_like(i, second)
    lo, hi = torch.full_like(i, step & _M32), torch.full_like(i, step >> 32)
    a, b = _philox([i, w, lo, hi], seed), _philox([i, w | 0x80000000, lo, hi], seed)
    return _uniform(a[0], a[1]), _uniform(a[2], a[3]), _uniform(b[0], b[1]), _uniform(b[2], b[3])


def _normals(n, step, seed):
    u1, u2, u3, u4 = _uniforms(n, 0, step, seed)
    r1, r2 = torch.sqrt(-2 * torch.log(1 - u1)), torch.sqrt(-2 * torch.log(1 - u3))
    return torch.stack([r1 * torch.cos(2 * math.pi * u2), r1 * torch.sin(2 * math.pi * u2), r2 * torch.cos(2 * math.pi * u4)], dim=-1)


def _rotate(s, v):
    angle = torch.sqrt(_dot(v, v))
    k = v / angle
    c, sn = torch.cos(angle), torch.sin(angle)
    return s * c + _cross(k, s) * sn + k * _dot(k, s) * (1 - c)


def _cayley(s, f):
    A = 0.5 * f
    a2 = s - _cross(s, A)
    return (a2 + A * _dot(A, a2) + _cross(A, a2)) / (1 + _dot(A, A))


def _llg(model, s, solver, steps, dt, damping, noise=None):
    """`steps` steps from s; noise(step) is the thermal field.  Returns the spins and the last step's first force."""
    dtg = dt * GAMMA / MU_B / (1 + damping * damping)
    F = None
    for n in range(steps):
        xi = noise(n) if noise else None

        def virtual(x):
            f, _ = model.force(x)
            v = dtg * (f + damping * _cross(x, f)) / model.mu
            if xi is not None:
                v = v + xi + damping * _cross(x, xi)
            return f, v

        F, v = virtual(s)
        if solver == "depondt":
            _, w = virtual(_rotate(s, v))
            s = _rotate(s, 0.5 * (v + w))
        elif solver == "heun":
            x = _unit(s - _cross(s, v))
            _, w = virtual(x)
            s = _unit(s - 0.5 * _cross(s, v) - 0.5 * _cross(x, w))
        elif solver == "sib":
            _, w = virtual(0.5 * (s + _cayley(s, v)))
            s = _cayley(s, w)
        else:
            k1 = -_cross(s, v)
            x = _unit(s + 0.5 * k1)
            k2 = -_cross(x, virtual(x)[1])
            x = _unit(s + 0.5 * k2)
            k3 = -_cross(x, virtual(x)[1])
            x = _unit(s + k3)
            k4 = -_cross(x, virtual(x)[1])
            s = _unit(s + k1 / 6 + k2 / 3 + k3 / 3 + k4 / 6)
    return s, F


def _thermal(case, T, seed, n, mu=2.0):
    if not T:
        return None
    a = case["damping"]
    eps = math.sqrt(2 * a * case["dt"] * GAMMA / MU_B * K_B) / (1 + a * a) * math.sqrt(T / mu)
    return lambda step: eps * _normals(n, step, seed)


def _lbfgs(model, s, steps):
    n = s.shape[0]
    mem = 3
    da, dg = [torch.zeros_like(s) for _ in range(mem)], [torch.zeros_like(s) for _ in range(mem)]
    rho, alpha = [0.0] * mem, [0.0] * mem
    it, sd, last, F = 0, None, None, None
    for _ in range(steps):
        F, _ = model.force(s)
        c = _cross(s, F)
        g = torch.stack([-c[:, 2], c[:, 1], -c[:, 0]], dim=1)
        descent = it == 0
        if not descent:
            m = it % mem
            da[m], dg[m] = sd, g - last
            curvature = float((dg[m] * da[m]).sum())
            if curvature > 1e-300:
                rho[m] = 1 / curvature
                first = [(k + it % mem + 1) % mem for k in range(mem)]
                order = list(range(mem)) if it < mem else first
                q = g
                for k in reversed(first):
                    alpha[k] = rho[k] * float((da[k] * q).sum())
                    q = q - alpha[k] * dg[k]
                d = q / (float((dg[m] * dg[m]).sum()) * rho[m])
                for k in order:
                    d = d + (alpha[k] - rho[k] * float((dg[k] * d).sum())) * da[k]
                d = -d
            else:
                descent, it = True, 0
        if descent:
            rho = [0.0] * mem
            da, dg = [torch.zeros_like(s) for _ in range(mem)], [torch.zeros_like(s) for _ in range(mem)]
            d = -g
        last = g
        rms = math.sqrt(float((d * d).sum()) / n)
        sd = d * (math.pi / 200 / rms if rms > math.pi / 200 else 1.0)
        it += 1
        # the rotation exp of the skew matrix of sd
        s = _rotate(s, torch.stack([sd[:, 2], -sd[:, 1], sd[:, 0]], dim=1))
    return s, F


def _metropolis(case, model, s, seed):
    n = s.shape[0]
    idx = torch.arange(n, device="cuda")
    a, rest = idx % case["na"], idx // case["na"]
    colour = (a + rest % case["nb"] + rest // case["nb"]) % 2
    z = model.z.expand_as(s)
    cone, rejected, kT = math.pi * 30.0 / 180.0, 0.0, K_B * case["T"]
    for step in range(case["steps"]):
        acc = 1 - rejected / n
        if acc < 0.5 and cone > 0.01:
            cone -= 0.01
        if acc > 0.5 and cone < math.pi - 0.01:
            cone += 0.01
        rejected = 0.0
        for col in range(2):
            u = _uniforms(n, col | 0x40000000, step, seed)
            flat = (s[:, 2:3] < 1 - 1e-10)
            x0 = _cross(s, z)
            x0 = x0 / torch.sqrt(torch.clamp(_dot(x0, x0), min=1e-300))
            e0 = torch.where(flat, x0, torch.tensor([1.0, 0.0, 0.0], dtype=torch.float64, device="cuda"))
            e1 = torch.where(flat, _cross(s, x0), torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64, device="cuda"))
            e2 = torch.where(flat, s, z)
            ct = (1 - (1 - math.cos(cone)) * u[0])[:, None]
            sn = torch.sqrt(1 - ct * ct)
            phi = (2 * math.pi * u[1])[:, None]
            trial = e0 * (sn * torch.cos(phi)) + e1 * (sn * torch.sin(phi)) + e2 * ct
            # the neighbours' field on each spin (its own anisotropy apart)
            f, _ = model.force(s)
            f = f - 2 * case["K"] * s[:, 2:3] * model.z
            dE = -_dot(f, trial - s)[:, 0] - case["K"] * (trial[:, 2] ** 2 - s[:, 2] ** 2)
            accept = (dE <= 1e-14) | (torch.exp(-dE / kT) >= u[2])
            mine = colour == col
            s = torch.where((accept & mine)[:, None], trial, s)
            rejected += float((~accept & mine).sum())
    return s


def _path(case, model, x, steps):
    """Nudged elastic band, velocity projection, one climbing image."""
    x = torch.stack(x)
    noi, dt = x.shape[0], case["dt"]
    v, last = torch.zeros_like(x), torch.zeros_like(x)
    for _ in range(steps):
        f, E = model.force(x, energy=True)
        angle = torch.acos(torch.clamp(_dot(x[1:], x[:-1]), -1, 1))
        dist = torch.sqrt((angle ** 2).sum(dim=(1, 2)))
        E = E.cpu()
        F = torch.zeros_like(x)
        for k in range(1, noi - 1):
            up, down = x[k + 1] - x[k], x[k] - x[k - 1]
            e, ep, em = float(E[k]), float(E[k + 1]), float(E[k - 1])
            if ep > e > em:
                t = up
            elif ep < e < em:
                t = down
            else:
                hi, lo = max(abs(ep - e), abs(em - e)), min(abs(ep - e), abs(em - e))
                if not ((ep < e and e > em) or (ep > e and e < em)):
                    hi = lo = 1.0
                t = (hi * up + lo * down) if ep > em else (lo * up + hi * down)
            t = t - _dot(t, x[k]) * x[k]
            t = t / torch.sqrt((t * t).sum())
            g = f[k] - _dot(f[k], x[k]) * x[k]
            along = (g * t).sum()
            if k == _climbing(case):
                F[k] = g - 2 * along * t
            else:
                F[k] = g - along * t + (dist[k] - dist[k - 1]) * t
        v = v + 0.5 * (last + F)
        power, norm = float((v * F).sum()), float((F * F).sum())
        v = F * (power / norm) if power > 0 else torch.zeros_like(F)
        x = _unit(x + dt * v + 0.5 * dt * F)
        last = F - _dot(F, x) * x
    return x


def exact(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "ensemble":
        return _exact_ensemble(case, inp["spins"], seed)
    model = _Model(case, inp.get("site_K"))
    if kind == "gradient":
        f, e = model.force(inp["spins"], energy=True)
        return {"gradient": -f, "energy": e.reshape(1)}
    if kind == "gneb":
        return [x.cpu().numpy() for x in _path(case, model, inp["spins"], case["steps"])]
    s = inp["spins"]
    if kind == "mc":
        return {"spins": _metropolis(case, model, s, _noise_seed(seed)).cpu().numpy()}
    if kind == "adjoint":
        return _exact_adjoint(case, model, s, inp["target"])
    if kind == "llg":
        s, F = _llg(model, s, case["solver"], case["steps"], case["dt"], case["damping"],
                    _thermal(case, case["T"], _noise_seed(seed), s.shape[0]))
    else:
        s, F = _lbfgs(model, s, case["steps"])
    return {"spins": s.cpu().numpy(), "field": (F - _dot(F, s) * s).cpu().numpy()}


def _exact_adjoint(case, model, s0, target):
    leaves = [s0.clone().requires_grad_(True), model.site_K.clone().requires_grad_(True)]
    leaves += [x.clone().requires_grad_(True) for x in (model.J[0], model.D, model.B)]
    s, model.site_K, model.J[0], model.D, model.B = leaves
    sN, _ = _llg(model, s, case["solver"], case["steps"], case["dt"], case["damping"])
    (((sN - target) ** 2).sum() / sN.shape[0]).backward()
    one = lambda x: x.grad.reshape(1).cpu().numpy()  # noqa: E731
    return {"spins": sN.detach(), "d_spins": s.grad, "d_J": one(model.J[0]), "d_D": one(model.D), "d_B": one(model.B),
            "d_K_site": model.site_K.grad.reshape(-1).cpu().numpy()}


def _exact_ensemble(case, spins, seed):
    sides, fields, temps = _replicas(case)
    out = []
    for k, (L, B, T) in enumerate(zip(sides, fields, temps)):
        rep = _lattice(int(L), int(L), 1, bc="110", D=3.0, chirality=2, K=0.1, B=float(B))
        s, _ = _llg(_Model(rep), spins[k], case["solver"], case["steps"], case["dt"], case["damping"],
                    _thermal(case, float(T), _noise_seed(seed + 1000 * k), int(L) * int(L)))
        out.append(s.cpu().numpy())
    return out
