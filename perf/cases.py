"""The work that a user of this package has it do, as cases that can be timed and compared.

Every case goes through the public entry points: event chains (DeviceChain.run, run_together),
batched replicas (DeviceBatch.run) and pair energies with their gradients (pair_energy).
``listed`` gives the fixed cases, ``draw`` one more of the ranges that they stand for,
``prepare`` what a program holds before the call, ``run`` one pass, ``work`` the bytes and
operations that the pass cannot do without and ``exact`` the result in plain 64-bit torch where
the outputs are computed numbers.  A chain's trajectory is a sequence of discrete choices that
plain torch cannot follow, so the chains and batches have no exact value.
"""
import math
import os

import numpy as np
import torch

from jellyfysh_amd.batch import DeviceBatch, lattice_positions
from jellyfysh_amd.chain import DeviceChain, make_desc, run_together
from jellyfysh_amd.config import RunConfig
from jellyfysh_amd.energy import pair_energy
from jellyfysh_amd.workloads import make_chain, soft_sphere_taggers

CONFIGS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jellyfysh_amd", "configs")
INVERSION_FLOPS = 60.0        # one pair inversion: three powers and a logarithm at 20, about 20 simple operations
MERGED_IMAGE = (3.45, 6, 2)   # alpha, Fourier cutoff, position cutoff
DIPOLE_DENSITY = 0.05         # dipoles per unit volume of flexible_dipoles.ini
CHUNK = 10000                 # legs per replica and step of the batched benchmark


def listed():
    return [
        # 256 hard disks at packing fraction 0.6 (hard_disks.ini): one chain, the cheapest leg there is
        dict(name="hard_disks_256", kind="chain", system="hard_disks", n=256, legs=4000, logged=False),
        # a short logged run of 256 Lennard-Jones units (lennard_jones.ini): the event log of a
        # test or an analysis, a call of a few milliseconds
        dict(name="lj_256_logged", kind="chain", system="lennard_jones", n=256, legs=64, logged=True),
        # the benchmark's plain chain: 4096 Lennard-Jones units, truncated at 2.5, 6 cells per side
        dict(name="lj_4096", kind="chain", system="lennard_jones_truncated", n=4096, legs=1000, logged=False),
        # 256 replicas of 512 charged soft spheres, far cells through the cell-bounding potential
        dict(name="charged_cell_bounding_256", kind="replicas", system="cell_bounding", n=512, replicas=256, legs=1000),
        # the same with the far cells through the cell veto
        dict(name="charged_cell_veto_256", kind="replicas", system="cell_veto", n=512, replicas=256, legs=1000),
        # 64 replicas of 500 flexible dipoles (flexible_dipoles.ini): factor-type maps, bonds, Coulomb, repulsion
        dict(name="dipoles_64", kind="replicas", system="dipoles", n=1000, replicas=64, legs=1000),
        # 256 replicas of two charges, each run to its next sampling event
        # (coulomb_atoms_cell_veto.ini): short launches, one read-out per sample
        dict(name="samples_256", kind="replicas", system="samples", n=2, replicas=256, legs=200000),
        # the headline: 4096 Lennard-Jones replicas of 64 to 2048 units, two steps, then the read-out
        dict(name="batch_4096", kind="batch", replicas=4096, n_min=64, n_max=2048, legs=2 * CHUNK),
        # the same for a few replicas: a small study, or one of many jobs on the card
        dict(name="batch_64", kind="batch", replicas=64, n_min=64, n_max=2048, legs=2000),
        # energy and gradients of a small Lennard-Jones system: a call per configuration
        dict(name="energy_lj_64", kind="energy", model="lennard_jones", n=64),
        # the same of an ordinary one
        dict(name="energy_lj_2048", kind="energy", model="lennard_jones", n=2048),
        # energy, forces and parameter gradients of 500 flexible dipoles (bond, Coulomb, repulsion)
        dict(name="energy_dipoles_1000", kind="energy", model="dipoles", n=1000),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    which = rng.choice(["disks", "lj", "charged", "dipoles", "samples", "batch", "batch", "energy", "energy"])
    if which == "disks":
        return dict(kind="chain", system="hard_disks", n=_log_uniform(rng, 64, 1024), legs=_log_uniform(rng, 50, 4000),
                    logged=rng.random() < 0.5)
    if which == "lj":
        return dict(kind="chain", system=rng.choice(["lennard_jones", "lennard_jones_truncated"]),
                    n=_log_uniform(rng, 108, 4096), legs=_log_uniform(rng, 50, 1000), logged=rng.random() < 0.5)
    if which == "charged":
        return dict(kind="replicas", system=rng.choice(["cell_bounding", "cell_veto"]), n=2 * rng.randint(32, 256),
                    replicas=_log_uniform(rng, 1, 256), legs=_log_uniform(rng, 50, 1000))
    if which == "dipoles":
        return dict(kind="replicas", system="dipoles", n=2 * _log_uniform(rng, 4, 500), replicas=_log_uniform(rng, 1, 64),
                    legs=_log_uniform(rng, 50, 1000))
    if which == "samples":
        return dict(kind="replicas", system="samples", n=2, replicas=rng.randint(1, 256), legs=200000)
    if which == "batch":
        n_min = _log_uniform(rng, 16, 512)
        return dict(kind="batch", replicas=_log_uniform(rng, 1, 2048), n_min=n_min,
                    n_max=_log_uniform(rng, n_min, 2048), legs=_log_uniform(rng, 100, CHUNK))
    if rng.random() < 0.5:
        return dict(kind="energy", model="lennard_jones", n=_log_uniform(rng, 16, 3000))
    return dict(kind="energy", model="dipoles", n=2 * _log_uniform(rng, 8, 600))


# ---- inputs ---------------------------------------------------------------------------------
def _config(name):
    return RunConfig.from_file(os.path.join(CONFIGS, name + ".ini"))


def _lj_length(n):
    return (n / 0.8) ** (1.0 / 3.0)


def _hard_disks(n, rng):
    """n disks of packing fraction 0.6 on sites of a square grid of the unit square, jittered by 1%."""
    m = int(math.ceil(math.sqrt(n)))
    sites = np.sort(rng.choice(m * m, size=n, replace=False))
    pos = (np.stack([sites % m, sites // m], axis=1) + 0.5 + rng.uniform(-0.01, 0.01, (n, 2))) / m
    return pos, math.sqrt(0.6 / (n * math.pi))


def _dipoles(n, length, rng):
    """n / 2 dipoles of bond length 0.9 to 1.1 and random direction, centres on a jittered grid."""
    centre = lattice_positions(n // 2, length, 0.05, rng)
    axis = rng.normal(size=(n // 2, 3))
    axis *= (rng.uniform(0.9, 1.1, (n // 2, 1)) / 2.0) / np.linalg.norm(axis, axis=1, keepdims=True)
    return np.mod(np.stack([centre + axis, centre - axis], axis=1).reshape(n, 3), length)


def _dipole_length(n):
    return (n / 2 / DIPOLE_DENSITY) ** (1.0 / 3.0)


def _chain(case, seed):
    n, rng = case["n"], np.random.default_rng(seed)
    cfg = _config(case["system"])
    if case["system"] == "hard_disks":
        pos, radius = _hard_disks(n, rng)
        taggers = [dict(t, params=[radius]) if t.get("potential") == "hard_sphere" else t for t in cfg.taggers]
        desc = make_desc(2, n, 1.0, cfg.beta, int(1.0 / (2.0 * radius)), taggers, seed, scheduler=cfg.scheduler)
    else:
        length = _lj_length(n)
        pos = lattice_positions(n, length, 0.01, rng)
        desc = make_desc(3, n, length, cfg.beta, max(3, int(length / 2.5)), cfg.taggers, seed, scheduler=cfg.scheduler)
    return DeviceChain(desc, pos)


def _replicas(case, seed):
    n, count, system = case["n"], case["replicas"], case["system"]
    chains = []
    if system in ("cell_bounding", "cell_veto"):
        length = n ** (1.0 / 3.0)
        taggers = soft_sphere_taggers(far=system)
        charges = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
        for i in range(count):
            pos = lattice_positions(n, length, 0.08, np.random.default_rng([seed, i]))
            chains.append(make_chain(dict(dim=3, n=n, system_length=length, beta=1.0, cells_per_side=int(length + 1e-9),
                                          seed=seed * 1000 + i, taggers=taggers, positions=pos, charges=charges,
                                          max_occupants=1)))
        return chains
    if system == "dipoles":
        cfg, length = _config("flexible_dipoles"), _dipole_length(n)
        charges = np.tile([0.5, -0.5], n // 2)
        for i in range(count):
            desc = make_desc(3, n, length, cfg.beta, 1, cfg.taggers, seed * 1000 + i, scheduler=cfg.scheduler,
                             leaves_per_root=2)
            chains.append(DeviceChain(desc, _dipoles(n, length, np.random.default_rng([seed, i])), charges))
        return chains
    cfg = _config("coulomb_atoms_cell_veto")
    sampling = [i for i, t in enumerate(cfg.taggers) if t["kind"] == "sampling"][0]
    for i in range(count):
        pos, charges, words = cfg.initial_state(seed * 1000 + i)
        chains.append(DeviceChain(cfg.desc(len(pos), seed * 1000 + i, rng_skip=words), pos, charges))
        chains[-1].set_stop_mask(1 << sampling)
    return chains


def _batch(case, seed):
    # the replicas' sizes and densities belong to the case, their starts to the seed
    size, start = np.random.default_rng(case["n_min"] + case["n_max"]), np.random.default_rng(seed)
    n = np.rint(np.exp(size.uniform(np.log(case["n_min"]), np.log(case["n_max"]), case["replicas"]))).astype(np.int32)
    lengths = (n / size.uniform(0.7, 0.9, case["replicas"])) ** (1.0 / 3.0)
    pos = [lattice_positions(int(k), float(v), 0.01, start) for k, v in zip(n, lengths)]
    return DeviceBatch(n, lengths, pos, seed=seed)


def _energy_inputs(case, seed):
    """The tensors of an energy case: positions and parameters (all differentiated), and what is fixed."""
    n, rng = case["n"], np.random.default_rng(seed)
    def t(v):
        return torch.tensor(v, dtype=torch.float64, device="cuda", requires_grad=True)
    if case["model"] == "lennard_jones":
        length = _lj_length(n)
        return dict(length=length, x=t(lattice_positions(n, length, 0.1, rng)), theta=[t([4.0, 1.0])])
    length = _dipole_length(n)
    return dict(length=length, x=t(_dipoles(n, length, rng)),
                theta=[t(400.0), t(1.0), t(0.5), t(1.0)],   # bond constant and length, charge, repulsion
                sign=torch.tensor(np.tile([1.0, -1.0], n // 2), device="cuda"),
                molecule=torch.arange(n, dtype=torch.int32, device="cuda") // 2)


def prepare(case, seed):
    state = dict(case)
    if case["kind"] == "chain":
        state["chain"] = _chain(case, seed)
    elif case["kind"] == "replicas":
        state["chains"] = _replicas(case, seed)
    elif case["kind"] == "batch":
        state["batch"] = _batch(case, seed)
    else:
        state.update(_energy_inputs(case, seed))
    return state


# ---- one pass -------------------------------------------------------------------------------
def run(state):
    return {"chain": _run_chain, "replicas": _run_replicas, "batch": _run_batch, "energy": _run_energy}[state["kind"]](state)


def _run_chain(state):
    chain = state["chain"]
    got = chain.run(state["legs"], log=state["logged"])
    active, direction, q, r, done = chain.active()
    out = dict(positions=chain.positions(), estimators=chain.estimators(), active=active, direction=direction,
               time=np.array([q, r]), words=chain.rng_words())
    if state["logged"]:
        out["log"] = {f: got[f] for f in got.dtype.names}
    else:
        out["legs"] = int(got)
    return out


def _run_replicas(state):
    chains = state["chains"]
    legs, _ = run_together(chains, state["legs"])
    return dict(legs=legs, positions=np.stack([c.positions() for c in chains]),
                estimators=np.stack([c.estimators() for c in chains]))


def _run_batch(state):
    batch, left = state["batch"], state["legs"]
    while left > 0:
        batch.run(min(CHUNK, left))
        left -= min(CHUNK, left)
    s = batch.states()
    return dict(active=s["active"], direction=s["direction"], chain_left=s["chain_left"], legs=s["legs"].astype(np.int64),
                estimators=s["est"], positions=np.concatenate(batch.positions()))


def _run_energy(state):
    x, theta, length = state["x"], state["theta"], state["length"]
    if state["model"] == "lennard_jones":
        terms = [pair_energy(x, theta[0], "lennard_jones", length)]
    else:
        k, r0, q, k12 = theta
        two, twelve = (torch.tensor(v, dtype=torch.float64, device=x.device) for v in (2.0, 12.0))
        mol = state["molecule"]
        terms = [pair_energy(x, torch.stack([r0, two, k / 2]), "displaced_even_power", length, molecule=mol, scope="intra"),
                 pair_energy(x, [float(v) for v in MERGED_IMAGE] + [1.0], "merged_image_coulomb", length,
                             charges=q * state["sign"], molecule=mol, scope="inter"),
                 pair_energy(x, torch.stack([twelve, k12]), "inverse_power", length, molecule=mol, scope="inter")]
    grads = torch.autograd.grad(sum(terms), [x] + theta)
    return dict(energies=[u.detach() for u in terms], grad_x=grads[0], grad_theta=list(grads[1:]))


# ---- what a pass cannot do without ----------------------------------------------------------
def _candidates(case):
    """Pair candidates per leg."""
    n, system = case["n"], case["system"]
    if system == "hard_disks":
        return n * 9.0 / int(1.0 / (2.0 * math.sqrt(0.6 / (n * math.pi)))) ** 2
    if system.startswith("lennard_jones"):
        return 2.0 * n * min(1.0, 27.0 / max(3, int(_lj_length(n) / 2.5)) ** 3)
    if system == "dipoles":
        return 2.0 * n
    if system == "samples":
        return 1.0
    return 2.0 * n if system == "cell_bounding" else 1.25 * n


def work(case):
    if case["kind"] == "energy":
        n = case["n"]
        pairs = n * (n - 1) / 2.0
        images, waves = (0, 0) if case["model"] == "lennard_jones" else (33, 900)
        # per pair about 40 operations a power pair and 60 a real-space image; per unit 20 a wave
        return dict(bytes=8.0 * (6 * n + 16), flops=pairs * (40.0 + 60.0 * images) + n * 20.0 * waves)
    if case["kind"] == "batch":
        # mean of a log-uniform size; 27 of the (L / 2.5)^3 cells, all units below three cells a side
        lo, hi = case["n_min"], case["n_max"]
        mean = lo if lo == hi else (hi - lo) / math.log(hi / lo)
        cands = min(mean, 350.0)
        legs = float(case["legs"]) * case["replicas"]
        return dict(bytes=case["replicas"] * (mean * 48.0 + 256.0), flops=legs * cands * 2 * INVERSION_FLOPS)
    dim = 2 if case["system"] == "hard_disks" else 3
    count = case.get("replicas", 1)
    legs = float(count) * (20.0 if case["system"] == "samples" else case["legs"])
    log = 64.0 * legs if case.get("logged") else 0.0
    return dict(bytes=count * case["n"] * (dim * 16.0 + 8.0) + log, flops=legs * _candidates(case) * INVERSION_FLOPS)


# ---- plain 64-bit values of the energy cases ------------------------------------------------
def _separations(x, rows, length):
    s = x[None, :, :] - x[rows][:, None, :] + length / 2
    return s - length * torch.floor(s.detach() / length) - length / 2


def _coulomb(s, length):
    """The merged-image Coulomb pair function for separations s (... x 3)."""
    alpha, fc, pc = MERGED_IMAGE
    a, psi = alpha / length, 0.0
    for i in range(-pc, pc + 1):
        for j in range(-pc, pc + 1):
            for k in range(-pc, pc + 1):
                if i * i + j * j + k * k <= pc * pc:
                    r = (s + length * torch.tensor([i, j, k], dtype=s.dtype, device=s.device)).norm(dim=-1)
                    psi = psi + torch.erfc(a * r) / r
    w = 2.0 * math.pi / length
    cos = [[torch.cos(w * m * s[..., d]) for m in range(fc + 1)] for d in range(3)]
    for i in range(fc + 1):
        for j in range(fc + 1):
            for k in range(fc + 1):
                n2 = i * i + j * j + k * k
                if 0 < n2 <= fc * fc:
                    weight = (2 if i else 1) * (2 if j else 1) * (2 if k else 1)
                    g = weight * math.exp(-math.pi ** 2 * n2 / alpha ** 2) / (math.pi * length * n2)
                    psi = psi + g * cos[0][i] * cos[1][j] * cos[2][k]
    return psi - math.pi / (alpha ** 2 * length)


def exact(case, seed):
    if case["kind"] != "energy":
        return None
    e = _energy_inputs(case, seed)
    x, theta, length, n = e["x"], e["theta"], e["length"], case["n"]
    grads = [torch.zeros_like(v) for v in [x] + theta]
    count = 1 if case["model"] == "lennard_jones" else 3
    energies = [0.0] * count
    for lo in range(0, n, 64):       # rows of pairs at a time: the graphs of all of them would not be small
        rows = torch.arange(lo, min(lo + 64, n), device=x.device)
        s = _separations(x, rows, length)
        other = rows[:, None] != torch.arange(n, device=x.device)[None, :]
        if case["model"] == "lennard_jones":
            r2 = (s ** 2).sum(-1)[other]
            x6 = (theta[0][1] ** 2 / r2) ** 3
            terms = [0.5 * (theta[0][0] * (x6 * x6 - x6)).sum()]
        else:
            k, r0, q, k12 = theta
            mol = e["molecule"]
            same = other & (mol[rows][:, None] == mol[None, :])
            apart = mol[rows][:, None] != mol[None, :]
            qq = ((q * e["sign"])[rows][:, None] * (q * e["sign"])[None, :])[apart]
            terms = [0.5 * (k / 2 * (s[same].norm(dim=-1) - r0) ** 2).sum(),
                     0.5 * (qq * _coulomb(s[apart], length)).sum(),
                     0.5 * (k12 / ((s ** 2).sum(-1)[apart]) ** 6).sum()]
        for i, u in enumerate(torch.autograd.grad(sum(terms), [x] + theta, allow_unused=True)):
            if u is not None:
                grads[i] += u
        energies = [a + u.detach() for a, u in zip(energies, terms)]
    return dict(energies=energies, grad_x=grads[0], grad_theta=grads[1:])
