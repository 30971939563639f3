"""Timed workloads of the polymer field theory on the GPU, with what each must compute.

Every case is one pass through the package's public entry points:

  eval      one evaluation of a melt: chain propagators, concentrations, partition functions and, with
            "stress", the box stress. "host" cases hand numpy fields in and take numpy concentrations out, as
            the SCFT driver does each iteration; the others keep the fields in device memory, as the L-FTS
            driver does.
  real      one evaluation with the real-space Crank-Nicolson solver (walls, a particle's mask, grafted chains).
  lfts      one Langevin step of an AB melt with the saddle points before and after it, stopped after a fixed
            number of iterations; with "replicas" > 1 independent runs advance together.
  train     Adam steps of the convolutional network that guesses a saddle point, forward and backward.

Numbers are drawn from the case's seed alone. exact() states the same results in plain torch, in 64 bits.
"""
import contextlib
import io
import math

import numpy as np
import torch

# ------------------------------------------------------------------------------------------------ cases


def listed():
    return [
        # SCFT of a lamellar phase in one dimension: the smallest calls, 100 contour steps of a few thousand bytes
        dict(name="lamella1d", kind="eval", nx="128", lx="3.6", model="continuous", n=100, chain="diblock", f=0.5,
             precision="hip", field="waves", sigma=10.0, stress=True, host=True),
        # SCFT of hexagonal cylinders in two dimensions: a rectangular cell of sides 1 : sqrt(3), box relaxation
        dict(name="cylinder2d", kind="eval", nx="60x104", lx="3.9x6.755", model="continuous", n=100, chain="diblock",
             f=0.3, precision="hip", field="waves", sigma=10.0, stress=True, host=True),
        # the reference's basic 3D evaluation: AB diblock, 32^3, random fields, with stress
        dict(name="cube32", kind="eval", nx="32x32x32", lx="4x4x4", model="continuous", n=100, chain="diblock", f=0.5,
             precision="hip", field="noise", sigma=1.0, stress=True, host=False),
        # SCFT iteration of a gyroid-forming diblock at 64^3 with box relaxation: host fields in, host fields out
        dict(name="gyroid64", kind="eval", nx="64x64x64", lx="3.3x3.3x3.3", model="continuous", n=100,
             chain="diblock", f=0.36, precision="hip", field="waves", sigma=10.0, stress=True, host=True),
        # branched polymers in a mixture: a 3-arm ABC star with an A homopolymer, different segment lengths
        dict(name="star64", kind="eval", nx="64x64x64", lx="4x4x4", model="continuous", n=100, chain="star", f=0.0,
             precision="hip", field="noise", sigma=1.0, stress=True, host=False),
        # an orthorhombic cell (the usual shape of cylinder and Fddd phases), 3D, FP64
        dict(name="box3d", kind="eval", nx="48x84x60", lx="3.9x6.755x4.8", model="continuous", n=100, chain="diblock",
             f=0.3, precision="hip", field="noise", sigma=3.0, stress=True, host=False),
        # discrete chains in FP32 on a large non-cubic grid, ragged last axis
        dict(name="box3d_fp32", kind="eval", nx="72x120x75", lx="4.5x7.5x4.7", model="discrete", n=64,
             chain="diblock", f=0.5, precision="hip-fp32", field="noise", sigma=6.0, stress=False, host=False),
        # a large melt in FP32 propagators: 128^3 with stress
        dict(name="melt128_fp32", kind="eval", nx="128x128x128", lx="6x6x6", model="continuous", n=100,
             chain="diblock", f=0.4, precision="hip-fp32", field="noise", sigma=2.0, stress=True, host=False),
        # chains grafted in a box with walls around a spherical particle (real-space steps)
        dict(name="particle3d", kind="real", nx="120x100x140", lx="4x5x6", n=100, bc="aarrrr", radius=1.0),
        # one L-FTS Langevin step of the discrete N=90 diblock at 64^3 (8 + 16 saddle iterations)
        dict(name="langevin64", kind="lfts", nx="64x64x64", lx="6x6x6", model="discrete", n=90, chi_n=17.0,
             nbar=1e4, dt=0.8, replicas=1, before=8, after=16),
        # 32 independent L-FTS replicas at 48^3 advancing together (4 + 8 saddle iterations)
        dict(name="replicas48", kind="lfts", nx="48x48x48", lx="4x4x4", model="discrete", n=64, chi_n=17.0,
             nbar=1e4, dt=0.8, replicas=32, before=4, after=8),
        # 8 training iterations of the learned guess at 64^3: forward, backward, Adam
        dict(name="train64", kind="train", nx="64x64x64", lx="6x6x6", iters=8, lr=5e-4),
    ]


def _smooth(lo, hi, most):
    """Lengths in lo..hi whose prime factors are at most `most` (what the FFT plans of that precision take)."""
    out = []
    for v in range(lo, hi + 1):
        m = v
        for p in (2, 3, 5, 7, 11, 13):
            if p <= most:
                while m % p == 0:
                    m //= p
        if m == 1:
            out.append(v)
    return out


def _log_pick(rng, values):
    """One of the values, evenly over their logarithm."""
    x = math.exp(rng.uniform(math.log(values[0]), math.log(values[-1])))
    return min(values, key=lambda v: abs(math.log(v / x)))


def _text(values, fmt="%g"):
    return "x".join(fmt % v for v in values)


def draw(rng):
    r = rng.random()
    if r < 0.72:   # evaluations
        precision = rng.choice(["hip", "hip", "hip", "hip-fp32"])
        most = 13 if precision == "hip" else 5
        dim = rng.choice([1, 2, 2, 3, 3, 3, 3, 3])
        model = rng.choice(["continuous", "continuous", "discrete"])
        n = _log_pick(rng, list(range(20, 121)))
        if dim == 1:
            nx = [_log_pick(rng, _smooth(24, 256, most))]
        elif dim == 2:
            nx = [_log_pick(rng, _smooth(20, 125, most)) for _ in range(2)]
        elif rng.random() < 0.4:
            nx = [rng.choice([32, 48, 64, 96, 128])] * 3
        else:
            nx = [_log_pick(rng, _smooth(18, 125, most)) for _ in range(3)]
        # no drawn evaluation moves more than the 128^3 FP32 one
        while int(np.prod(nx)) * n * (8 if precision == "hip" else 4) * (3 if model == "continuous" else 1) > \
                128 ** 3 * 100 * 12:
            n = max(20, n // 2)
            if n == 20:
                nx = [min(v, 96) for v in nx]
        dx = rng.uniform(0.04, 0.09)
        return dict(kind="eval", nx=_text(nx), lx=_text([v * dx for v in nx], "%.4f"), model=model, n=n,
                    chain=rng.choice(["diblock", "diblock", "triblock", "homopolymer", "star"]),
                    f=rng.choice([0.2, 0.3, 0.36, 0.5]), precision=precision, field=rng.choice(["waves", "noise"]),
                    sigma=rng.choice([1.0, 3.0, 6.0]), stress=rng.random() < 0.6, host=dim < 3 or rng.random() < 0.3)
    if r < 0.82:   # real-space evaluations
        dim = rng.choice([1, 2, 3, 3])
        nx = [rng.randint(30, 130) for _ in range(dim)]
        bc = "".join(2 * "p" if rng.random() < 0.4 else rng.choice("ra") + rng.choice("ra") for _ in range(dim))
        dx = rng.uniform(0.03, 0.07)
        return dict(kind="real", nx=_text(nx), lx=_text([v * dx for v in nx], "%.4f"),
                    n=rng.randint(20, 100 if dim == 3 else 200), bc=bc, radius=rng.choice([0.0, 0.25]) * min(nx) * dx)
    if r < 0.92:   # Langevin steps
        replicas = rng.choice([1, 1, 1, 4, 8])
        if rng.random() < 0.5:
            nx = [rng.choice([32, 48, 64])] * 3
        else:
            nx = [_log_pick(rng, _smooth(24, 72, 5)) for _ in range(3)]
        dx = rng.uniform(0.07, 0.1)
        return dict(kind="lfts", nx=_text(nx), lx=_text([v * dx for v in nx], "%.4f"), model="discrete",
                    n=10 * rng.randint(4, 9), chi_n=rng.choice([14.0, 17.0]), nbar=1e4, dt=0.8, replicas=replicas,
                    before=rng.randint(2, 5), after=rng.randint(4, 8))
    nx = [4 * rng.randint(6, 16), 4 * rng.randint(6, 16), 8 * rng.randint(3, 9)]
    return dict(kind="train", nx=_text(nx), lx=_text([v * 0.09375 for v in nx], "%.4f"), iters=rng.randint(2, 8),
                lr=5e-4)


# ------------------------------------------------------------------------------------------------ systems


def _nx(case):
    return [int(v) for v in case["nx"].split("x")]


def _lx(case):
    return [float(v) for v in case["lx"].split("x")]


def _bonds(chain):
    return {"A": 1.0, "B": 1.0, "C": 1.2} if chain == "star" else {"A": 1.0} if chain == "homopolymer" else \
        {"A": 1.0, "B": 1.0}


def _polymers(case):
    """[volume fraction, [[monomer, number of segments, v, u], ...]] of each polymer."""
    n = case["n"]
    if case["kind"] == "real" or case["chain"] == "homopolymer":
        return [[1.0, [["A", n, 0, 1]]]]
    f = case.get("f", 0.5)
    na = max(1, round(f * n))
    if case["chain"] == "diblock":
        return [[1.0, [["A", na, 0, 1], ["B", n - na, 1, 2]]]]
    if case["chain"] == "triblock":
        h = max(1, na // 2)
        return [[1.0, [["A", h, 0, 1], ["B", n - 2 * h, 1, 2], ["A", h, 2, 3]]]]
    a, b = max(1, round(0.3 * n)), max(1, round(0.4 * n))
    return [[0.8, [["A", a, 0, 1], ["B", a, 0, 2], ["C", b, 0, 3]]], [0.2, [["A", max(1, n // 2), 0, 1]]]]


def _unique_steps(case):
    """Contour steps that have to be computed: both directions of a chain, once for a symmetric one, and a leaf
    that two polymers share once."""
    n = case["n"]
    if case["kind"] == "real":
        return 2 * n
    if case["kind"] == "lfts" or case["chain"] == "diblock":
        return 2 * n
    if case["chain"] == "star":
        return 2 * n + n // 2 - round(0.3 * n)
    return n


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _fields(case, seed):
    """The monomer fields, [n_monomers, M] on the GPU: white noise, or a few plane waves with a little noise on them
    (an SCFT start)."""
    nx = _nx(case)
    M = int(np.prod(nx))
    S = len(_bonds(case["chain"]))
    g = _generator(seed)
    if case["field"] == "noise":
        return case["sigma"] * torch.randn(S, M, generator=g, device="cuda", dtype=torch.float64)
    rng = np.random.default_rng(seed)
    w = torch.zeros([S] + nx, device="cuda", dtype=torch.float64)
    axes = torch.meshgrid(*[torch.arange(v, device="cuda", dtype=torch.float64) / v for v in nx], indexing="ij")
    for s in range(S):
        for _ in range(6):
            k = rng.integers(-2, 3, len(nx))
            phase = sum(float(a) * x for a, x in zip(k, axes))
            w[s] += case["sigma"] / 4 * torch.cos(2 * math.pi * (phase + rng.random()))
    w = w.reshape(S, M) - w.reshape(S, M).mean(dim=1, keepdim=True)
    return w + 0.05 * torch.randn(S, M, generator=g, device="cuda", dtype=torch.float64)


_BC = {"p": "periodic", "r": "reflecting", "a": "absorbing"}


def _particle(case):
    """Mask of a sphere at the box centre and the grafting field: a plane across each axis, 1/dx high."""
    nx, lx = _nx(case), _lx(case)
    axes = np.meshgrid(*[np.linspace(-l / 2, l / 2, num=n, endpoint=False) for n, l in zip(nx, lx)], indexing="ij")
    mask = np.ones(nx)
    if case["radius"] > 0:
        mask[np.sqrt(sum(a ** 2 for a in axes)) < case["radius"]] = 0.0
    q0 = np.zeros(nx)
    for d, (n, l) in enumerate(zip(nx, lx)):
        at = [slice(None)] * len(nx)
        at[d] = n // 4
        q0[tuple(at)] = n / l
    return mask.ravel(), (q0 * mask).ravel()


def _sigma(case):
    """Amplitude of the Langevin noise."""
    return math.sqrt(2 * case["dt"] * np.prod(_nx(case)) / (np.prod(_lx(case)) * math.sqrt(case["nbar"])))


def _langevin_inputs(case, seed):
    """Auxiliary fields [R, 2, M] (exchange field at about its equilibrium deviation, pressure field zero, as at the
    start of a run), the previous and the current noise [R, M]."""
    R, M = case["replicas"], int(np.prod(_nx(case)))
    g = _generator(seed)
    w = torch.zeros(R, 2, M, device="cuda", dtype=torch.float64)
    amp = math.sqrt(M * case["chi_n"] / (2 * np.prod(_lx(case)) * math.sqrt(case["nbar"])))
    w[:, 0] = amp * torch.randn(R, M, generator=g, device="cuda", dtype=torch.float64)
    noise = _sigma(case) * torch.randn(2, R, M, generator=g, device="cuda", dtype=torch.float64)
    return w, noise[0], noise[1]


def _training_inputs(case, seed):
    """The exchange field, a pressure field that depends on it over a few grid points, and He-normal weights."""
    nx = _nx(case)
    g = _generator(seed)
    x = torch.randn(nx, generator=g, device="cuda", dtype=torch.float64)
    s = x * x - 1.0
    y = s.clone()
    for d in range(3):
        y += torch.roll(s, 1, d) + torch.roll(s, -1, d)
    rng = np.random.default_rng(seed)
    parts = [rng.normal(0.0, math.sqrt(2 / 27), 27 * 32), np.zeros(32)]
    for _ in range(4):
        parts += [rng.normal(0.0, math.sqrt(2 / (27 * 32)), 27 * 32 * 32), np.zeros(32)]
    parts += [rng.normal(0.0, math.sqrt(1 / (27 * 32)), 27 * 32), np.zeros(1)]
    return 10.0 * x.reshape(-1), 1.2 * y.reshape(-1), np.concatenate(parts).astype(np.float32)


# ------------------------------------------------------------------------------------------------ the package's part


def _solver(case):
    from langevin_fts_amd import langevinfts as lf

    real = case["kind"] == "real"
    factory = lf.PlatformSelector.create_factory("hip" if real else case["precision"], False)
    model = "continuous" if real else case["model"]
    if real:
        mask, q0 = _particle(case)
        cb = factory.create_computation_box(_nx(case), _lx(case), bc=[_BC[c] for c in case["bc"]], mask=mask)
    else:
        mask, q0 = None, None
        cb = factory.create_computation_box(_nx(case), _lx(case))
    ds = 1.0 / case["n"]
    mol = factory.create_molecules_information(model, ds, {"A": 1.0} if real else _bonds(case["chain"]))
    for vf, blocks in _polymers(case):
        blocks = [[m, k * ds, v, u] for m, k, v, u in blocks]
        if real:
            mol.add_polymer(vf, blocks, {0: "G"})
        else:
            mol.add_polymer(vf, blocks)
    analyzer = factory.create_propagator_analyzer(mol, not real)
    make = factory.create_realspace_solver if real else factory.create_pseudospectral_solver
    return make(cb, mol, analyzer), cb, mol, q0, factory


def _lfts(case, seed):
    from langevin_fts_amd.lfts import LFTS

    params = {
        "nx": _nx(case), "lx": _lx(case), "chain_model": case.get("model", "discrete"), "ds": 1.0 / case.get("n", 16),
        "segment_lengths": {"A": 1.0, "B": 1.0}, "chi_n": {"A,B": case.get("chi_n", 17.0)},
        "distinct_polymers": [{"volume_fraction": 1.0, "blocks": [{"type": "A", "length": 0.5},
                                                                 {"type": "B", "length": 0.5}]}],
        "langevin": {"max_step": 0, "dt": case.get("dt", 0.8), "nbar": case.get("nbar", 1e4)},
        "recording": {"dir": ".", "recording_period": 10 ** 9, "sf_computing_period": 10 ** 9,
                      "sf_recording_period": 10 ** 9},
        "saddle": {"max_iter": 100, "tolerance": 1e-4},
        "am": {"max_hist": 20, "start_error": 5e-1, "mix_min": 0.01, "mix_init": 0.01}, "verbose_level": 0}
    with contextlib.redirect_stdout(io.StringIO()):
        return LFTS(params, random_seed=seed, n_replicas=case.get("replicas", 1))


def prepare(case, seed):
    case = dict(case)
    state = {"case": case}
    if case["kind"] == "eval":
        w = _fields(case, seed)
        names = sorted(_bonds(case["chain"]))
        state["solver"], *state["keep"] = _solver(case)
        state["polymers"] = len(_polymers(case))
        if case["host"]:
            state["w"] = {m: w[i].cpu().numpy() for i, m in enumerate(names)}
        else:
            state["w"] = {m: w[i].contiguous() for i, m in enumerate(names)}
            state["phi"] = {m: torch.empty_like(w[i]) for i, m in enumerate(names)}
    elif case["kind"] == "real":
        M = int(np.prod(_nx(case)))
        state["solver"], *keep = _solver(case)
        state["keep"] = keep
        state["w"] = torch.randn(M, generator=_generator(seed), device="cuda", dtype=torch.float64)
        state["q0"] = torch.from_numpy(keep[2]).cuda()
        state["phi"] = torch.empty_like(state["w"])
    elif case["kind"] == "lfts":
        w, prev, cur = (t.cpu().numpy() for t in _langevin_inputs(case, seed))
        state.update(w=w, prev=prev, cur=cur, sim=_lfts(case, seed))
    else:
        from langevin_fts_amd import langevinfts as lf

        x, y, params = _training_inputs(case, seed)
        sim = _lfts(case, seed)
        sim.saddle_device.set_fields(torch.stack([x, y]).cpu().numpy())
        state.update(sim=sim, params=params, guess=lf.LearnedGuess(_nx(case), 10.0, 3.0))
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "eval":
        solver = state["solver"]
        if case["host"]:
            solver.compute_propagators(state["w"])
            solver.compute_concentrations()
            phi = [solver.get_total_concentration(m) for m in state["w"]]
        else:
            solver.compute_propagators_device({m: t.data_ptr() for m, t in state["w"].items()})
            solver.compute_concentrations()
            for m, t in state["phi"].items():
                solver.get_total_concentration_device(m, t.data_ptr())
            phi = list(state["phi"].values())
        out = {"phi": phi, "Q": np.array([solver.get_total_partition(p) for p in range(state["polymers"])])}
        if case["stress"]:
            solver.compute_stress()
            out["stress"] = np.array(solver.get_stress())
        return out
    if case["kind"] == "real":
        solver = state["solver"]
        solver.compute_propagators_device({"A": state["w"].data_ptr()}, {"G": state["q0"].data_ptr()})
        solver.compute_concentrations()
        solver.get_total_concentration_device("A", state["phi"].data_ptr())
        return {"phi": state["phi"], "Q": solver.get_total_partition(0)}
    if case["kind"] == "lfts":
        dev = state["sim"].saddle_device
        dev.set_fields(state["w"])
        dev.set_noise_prev(state["prev"])
        dev.find_saddle_point(1e-12, case["before"], 0)
        dev.backup()
        dev.langevin_update(state["cur"], case["dt"])
        _, error, hamiltonian, _ = dev.find_saddle_point(1e-12, case["after"], 0)
        out = {"w": dev.get_fields(), "error": np.array(error), "H": np.array(hamiltonian)}
        if case["replicas"] == 1:
            out["phi"] = [dev.get_concentration(i) for i in range(2)]
        return out
    guess = state["guess"]
    guess.set_params(state["params"])
    loss = state["sim"].saddle_device.train_guess(guess, case["lr"], case["iters"], 1)
    return {"loss": loss, "params": guess.get_params()}


# ------------------------------------------------------------------------------------------------ what it must do


def _eval_work(case, steps, monomers, stress_terms):
    nx = _nx(case)
    M = int(np.prod(nx))
    fft = 2.5 * M * math.log2(M)   # a real transform
    continuous = case.get("model") == "continuous"
    flops = steps * ((6 if continuous else 2) * fft + 2 * M) + stress_terms * 2 * fft
    return flops, 2 * 8.0 * monomers * M


def work(case):
    nx = _nx(case)
    M = int(np.prod(nx))
    if case["kind"] == "eval":
        flops, size = _eval_work(case, _unique_steps(case), len(_bonds(case["chain"])), case["n"] if case["stress"] else 0)
        return {"bytes": size, "flops": flops}
    if case["kind"] == "real":
        # per step: a 2 dim + 1 point stencil, and two multiply-adds each way for every axis' solve
        return {"bytes": 3 * 8.0 * M, "flops": _unique_steps(case) * M * (4.0 + 14.0 * len(nx))}
    if case["kind"] == "lfts":
        flops, _ = _eval_work(case, 2 * case["n"], 2, 0)
        its = case["before"] + case["after"]
        return {"bytes": case["replicas"] * 8.0 * M * 6, "flops": case["replicas"] * its * flops}
    # forward, data gradients and weight gradients of 4 hidden 32 -> 32 layers and the two 1-channel ends
    layer = 2.0 * 27 * M
    return {"bytes": 2 * 8.0 * M, "flops": case["iters"] * layer * (3 * 4 * 32 * 32 + 5 * 32)}


def tolerance(case):
    # about four times the errors measured against exact(): bf16 activations and Adam's quotients of small gradients
    # (1e-3), FP64 rounding carried through a search's mixing steps (1e-8 in the error level, 2e-10 in the fields),
    # FP32 propagators (1.3e-5: Q after 107 steps), FP64 (1e-13 over the longest chains)
    if case["kind"] == "train":
        return {"rel": 5e-3, "max": 0.3}
    if case["kind"] == "lfts":
        return {"rel": 2e-7}
    if case["kind"] == "eval" and case["precision"] == "hip-fp32":
        return {"rel": 5e-5, "max": 5e-4}
    return {"rel": 1e-12, "max": 1e-10}


# ------------------------------------------------------------------------------------------------ the same in plain torch


class _Melt:
    """Propagators of block copolymers on a periodic box in torch, FP64; fields have leading batch axes."""

    def __init__(self, nx, lx, model, ds, bonds, polymers):
        self.nx, self.lx, self.model, self.ds, self.bonds, self.polymers = nx, lx, model, ds, bonds, polymers
        self.dims = tuple(range(-len(nx), 0))
        k2 = []
        for d, (n, l) in enumerate(zip(nx, lx)):
            i = torch.arange(n // 2 + 1 if d == len(nx) - 1 else n, device="cuda", dtype=torch.float64)
            shape = [1] * len(nx)
            shape[d] = -1
            k2.append(((2 * math.pi / l * torch.minimum(i, n - i)) ** 2).reshape(shape))
        ksq = sum(k2)
        self.bond = {m: torch.exp(-b * b * ds / 6 * ksq) for m, b in bonds.items()}
        self.half = {m: torch.exp(-b * b * ds / 12 * ksq) for m, b in bonds.items()}
        kz = torch.arange(nx[-1] // 2 + 1, device="cuda")
        weight = torch.where((kz == 0) | (2 * kz == nx[-1]), 1.0, 2.0).to(torch.float64)
        self.basis = [k * weight + 0 * ksq for k in k2]

    def conv(self, table, q):
        return torch.fft.irfftn(table * torch.fft.rfftn(q, dim=self.dims), s=self.nx, dim=self.dims)

    def advance(self, m, n, start, leaf):
        """Slices 0..n of one direction of a block (slice 0 of a discrete block: the product at its start)."""
        if self.model == "continuous":
            e2, e4 = torch.exp(-self.w[m] * self.ds / 2), torch.exp(-self.w[m] * self.ds / 4)
            out = [start]
            for _ in range(n):
                q = out[-1]
                q1 = e2 * self.conv(self.bond[m], e2 * q)
                q2 = e4 * self.conv(self.half[m], e2 * self.conv(self.half[m], e4 * q))
                out.append((4 * q2 - q1) / 3)
            return out
        e = torch.exp(-self.w[m] * self.ds)
        out = [start, e.clone() if leaf else e * self.conv(self.half[m], start)]
        for _ in range(n - 1):
            out.append(e * self.conv(self.bond[m], out[-1]))
        return out

    def evaluate(self, w, stress=False):
        self.w = w
        one = torch.ones_like(next(iter(w.values())))
        phi = {m: torch.zeros_like(one) for m in self.bonds}
        Q, total = [], [0.0] * len(self.nx)
        for vf, blocks in self.polymers:
            alpha = sum(k for _, k, _, _ in blocks) * self.ds
            edges = {}
            for m, k, v, u in blocks:
                edges[(v, u)] = edges[(u, v)] = (m, k)
            done = {}

            def slices(v, u):
                if (v, u) not in done:
                    m, k = edges[(v, u)]
                    q, leaf = one, True
                    for (a, b) in edges:
                        if b == v and a != u:
                            end = slices(a, v)[-1]
                            q = q * (end if self.model == "continuous" else self.conv(self.half[edges[(a, v)][0]], end))
                            leaf = False
                    done[(v, u)] = self.advance(m, k, q, leaf)
                return done[(v, u)]

            partition = None
            force = [0.0] * len(self.nx)
            parts = []
            for m, k, v, u in blocks:
                left, right = slices(v, u), slices(u, v)
                if self.model == "continuous":
                    c = _simpson(k)
                    if partition is None:
                        partition = (left[k] * right[0]).mean(dim=self.dims)
                    parts.append((m, sum(c[n] * left[k - n] * right[n] for n in range(k + 1))))
                    pairs = [(left[k - n], right[n], c[n], 1.0, None) for n in range(k + 1)]
                else:
                    e = torch.exp(self.w[m] * self.ds)
                    if partition is None:
                        partition = (left[k] * right[1] * e).mean(dim=self.dims)
                    parts.append((m, e * sum(left[k - n + 1] * right[n] for n in range(1, k + 1))))
                    pairs = [(left[k - n], right[n], 1.0, 1.0, self.bond[m]) for n in range(1, k)]
                    if any(b == v and a != u for a, b in edges):
                        pairs.append((left[0], right[k], 1.0, 0.5, self.half[m]))
                    if any(b == u and a != v for a, b in edges):
                        pairs.append((left[k], right[0], 1.0, 0.5, self.half[m]))
                if stress:
                    for a, b, c, share, table in pairs:
                        x = torch.fft.rfftn(a, dim=self.dims) * torch.fft.rfftn(b, dim=self.dims).conj()
                        x = share * c * self.bonds[m] ** 2 * (x.real if table is None else x.real * table)
                        for d in range(len(self.nx)):
                            force[d] = force[d] + (x * self.basis[d]).sum()
            for m, s in parts:
                phi[m] = phi[m] + s * (self.ds * vf / alpha) / partition.reshape(partition.shape + (1,) * len(self.nx))
            Q.append(partition)
            if stress:
                M = float(np.prod(self.nx))
                for d in range(len(self.nx)):
                    total[d] = total[d] + force[d] * vf / alpha / partition / (-3.0 * self.lx[d] * M * M / self.ds)
        return phi, Q, total


def _simpson(N):
    """Weights of the 4th-order contour integral over N intervals (3/8 rule at the end for odd N)."""
    if N == 0:
        return [1.0]
    if N == 1:
        return [0.5, 0.5]
    c = [0.0] * (N + 1)
    even = N if N % 2 == 0 else N - 3
    for i in range(0, even, 2):
        c[i] += 1 / 3
        c[i + 1] += 4 / 3
        c[i + 2] += 1 / 3
    if N % 2:
        for k, v in enumerate((3 / 8, 9 / 8, 9 / 8, 3 / 8)):
            c[N - 3 + k] += v
    return c


class _Mixing:
    """Anderson mixing with a bounded history."""

    def __init__(self, most, start_error, least, first):
        self.most, self.start_error, self.least, self.mix = most, start_error, least, first
        self.w, self.d = [], []

    def step(self, w, d, old, new):
        if new < self.start_error or self.w:
            self.w, self.d = ([w.clone()] + self.w)[: self.most + 1], ([d.clone()] + self.d)[: self.most + 1]
        n = len(self.w) - 1
        if n <= 0:
            self.mix = max(self.mix * 0.7, self.least) if old < new else self.mix * 1.01
            return w + self.mix * d
        diff = torch.stack([self.d[0] - x for x in self.d[1:]])
        gram = (diff @ diff.T).cpu().numpy()
        a = np.linalg.solve(gram, (diff @ self.d[0]).cpu().numpy())
        out = self.w[0] + self.d[0]
        for k in range(n):
            out = out + a[k] * (self.w[k + 1] + self.d[k + 1] - self.w[0] - self.d[0])
        return out


def _exact_lfts(case, seed):
    nx, ds = _nx(case), 1.0 / case["n"]
    w, prev, cur = _langevin_inputs(case, seed)
    R, M = case["replicas"], int(np.prod(nx))
    k = case["n"] // 2
    melt = _Melt(nx, _lx(case), case["model"], ds, {"A": 1.0, "B": 1.0}, [[1.0, [["A", k, 0, 1], ["B", k, 1, 2]]]])

    def search(count):
        mix = [_Mixing(20, 0.5, 0.01, 0.01) for _ in range(R)]
        err = [1e20] * R
        for _ in range(count):
            f = {"A": w[:, 0] + w[:, 1], "B": w[:, 1] - w[:, 0]}
            phi, Q, _ = melt.evaluate({m: v.reshape([R] + nx) for m, v in f.items()})
            phi = {m: v.reshape(R, M) for m, v in phi.items()}
            h = phi["A"] + phi["B"] - 1
            H = -w[:, 1].mean(dim=1) + (w[:, 0] ** 2).mean(dim=1) / case["chi_n"] - torch.log(Q[0]) + case["chi_n"] / 4
            for r in range(R):
                old, err[r] = err[r], float(h[r].std(correction=0))
                w[r, 1] = mix[r].step(w[r, 1].clone(), h[r], old, err[r])
        w[:, 1] -= w[:, 1].mean(dim=1, keepdim=True)
        return phi, err, H

    phi, _, _ = search(case["before"])
    w[:, 0] += -case["dt"] * (2 * w[:, 0] / case["chi_n"] + phi["A"] - phi["B"]) + 0.5 * (prev + cur)
    phi, err, H = search(case["after"])
    out = {"w": w if R > 1 else w[0], "error": np.array(err if R > 1 else err[0]), "H": H if R > 1 else H[0]}
    if R == 1:
        out["phi"] = [phi["A"][0], phi["B"][0]]
    return out


def _exact_real(case, seed):
    nx, lx, ds = _nx(case), _lx(case), 1.0 / case["n"]
    D = len(nx)
    w = torch.randn(int(np.prod(nx)), generator=_generator(seed), device="cuda", dtype=torch.float64).reshape(nx)
    mask, q0 = (torch.from_numpy(a).cuda().reshape(nx) for a in _particle(case))
    implicit, inverse = [], []
    for d in range(D):
        n = nx[d]
        f = ds / ((lx[d] / n) ** 2 * 6)
        T = np.zeros((n, n))
        for i in range(n):
            T[i, i] += 1 + f
            for j, side in ((i - 1, case["bc"][2 * d]), (i + 1, case["bc"][2 * d + 1])):
                if 0 <= j < n or side == "p":
                    T[i, j % n] += -0.5 * f
                elif side == "r":
                    T[i, i] += -0.5 * f
        implicit.append(torch.from_numpy(T - np.eye(n)).cuda())
        inverse.append(torch.from_numpy(np.linalg.inv(T)).cuda())

    def along(matrix, q, d):
        return torch.movedim(torch.matmul(torch.movedim(q, d, -1), matrix.T.contiguous()), -1, d)

    e = torch.exp(-w * ds / 2)

    def advance(start):
        out = [start * mask]
        for _ in range(case["n"]):
            q = e * out[-1]
            b = [along(implicit[d], q, d) for d in range(D)]
            x = along(inverse[0], q - b[0] - 2 * sum(b[1:]), 0)
            for d in range(1, D):
                x = along(inverse[d], x + b[d], d)
            out.append(e * x * mask)
        return out

    left, right = advance(q0), advance(torch.ones_like(w))
    volume = float(np.prod(lx))
    n = case["n"]
    dv = volume / w.numel()
    Q = float((left[n] * right[0] * mask).sum()) * dv / volume
    phi = sum(c * left[n - i] * right[i] for i, c in enumerate(_simpson(n))) * ds / Q
    return {"phi": phi.reshape(-1), "Q": Q}


def _exact_train(case, seed):
    nx = _nx(case)
    M = int(np.prod(nx))
    x, y, params = _training_inputs(case, seed)
    x, y = (x / 10.0).reshape([1] + nx), (y / 3.0).reshape(M)
    p = torch.from_numpy(params.astype(np.float64)).cuda().requires_grad_()
    shapes = [(27, 32, 1), (32,)] + 4 * [(27, 32, 32), (32,)] + [(27, 1, 32), (1,)]
    sizes = [int(np.prod(s)) for s in shapes]

    def forward():
        at, h = 0, x
        parts = []
        for s, k in zip(shapes, sizes):
            parts.append(p[at:at + k].reshape(s))
            at += k
        for layer in range(6):
            W, b = parts[2 * layer], parts[2 * layer + 1]
            out = b[:, None].expand(-1, M)
            for t in range(27):
                shift = (-(t // 9 - 1), -(t // 3 % 3 - 1), -(t % 3 - 1))
                out = out + W[t] @ torch.roll(h, shift, (1, 2, 3)).reshape(h.shape[0], M)
            h = torch.relu(out) if layer < 5 else out
            h = h.reshape([-1] + nx)
        return h.reshape(M)

    m, v, first = torch.zeros_like(p), torch.zeros_like(p), None
    for i in range(case["iters"]):
        loss = ((forward() - y) ** 2).mean()
        first = float(loss) if first is None else first
        g, = torch.autograd.grad(loss, p)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        with torch.no_grad():
            p -= case["lr"] * (m / (1 - 0.9 ** (i + 1))) / (torch.sqrt(v / (1 - 0.999 ** (i + 1))) + 1e-8)
    return {"loss": first, "params": p.detach()}


def exact(case, seed):
    with torch.no_grad() if case["kind"] != "train" else contextlib.nullcontext():
        if case["kind"] == "lfts":
            return _exact_lfts(case, seed)
        if case["kind"] == "real":
            return _exact_real(case, seed)
        if case["kind"] == "train":
            return _exact_train(case, seed)
        bonds = _bonds(case["chain"])
        melt = _Melt(_nx(case), _lx(case), case["model"], 1.0 / case["n"], bonds, _polymers(case))
        w = _fields(case, seed)
        names = sorted(bonds)
        phi, Q, stress = melt.evaluate({m: w[i].reshape(_nx(case)) for i, m in enumerate(names)}, case["stress"])
        out = {"phi": [phi[m].reshape(-1) for m in names], "Q": torch.stack(Q)}
        if case["stress"]:
            out["stress"] = torch.stack(list(stress))
        # the 4th-order contour integral over an odd number of steps depends on which end takes the 3/8 rule, and on
        # the pieces that a block shared by several chain ends is cut into: no single value for those
        if case["model"] == "continuous" and any(k % 2 for _, blocks in _polymers(case) for _, k, _, _ in blocks):
            out["phi"] = [None] * len(names)
            out.pop("stress", None)
        return out
