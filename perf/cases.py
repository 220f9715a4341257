"""The work whose speed counts: what programs have this engine do, over the sizes they do it at.

Dynamics is most of it: a single engine advancing a fluid, a melt or a mixture, a whole script
through ``Simulation.execute()``, and batches of replicas. The rest is frame mode: forces at given
positions, force matching, position gradients and trajectory backprop through torch.

Systems start near equilibrium, as a run that has gone on for a while does. A periodic cell of
about a thousand beads is relaxed with plain torch in binary64 (once per process and kind),
repeated along the axes, shifted and jittered by the seed, and given Maxwell velocities; whole
molecules are left out for odd sizes. Batches start from their lattices, as the replica sets do.
"""

from __future__ import annotations

import functools
import math
import tempfile

import numpy as np
import torch

from beads_amd import workloads as W

DEVICE = "cuda"


def listed():
    return [
        # The reduced-unit fluid of 4,000 beads: a small system, bound by launches.
        {"name": "fluid-4k", "kind": "fluid", "base": 500, "cx": 2, "cy": 2, "cz": 2, "drop": 0,
         "steps": 100},
        # The same fluid as a whole script: builders, run, thermo rows and a snapshot read back.
        {"name": "script-4k", "kind": "script", "base": 500, "cx": 2, "cy": 2, "cz": 2, "drop": 3,
         "steps": 200},
        # An ordinary bead-spring melt with all listed terms, checked for rebuilds every step.
        {"name": "melt-48k", "kind": "melt", "beads": 50, "cx": 4, "cy": 4, "cz": 3, "drop": 7,
         "steps": 100, "precision": "single"},
        # The million-bead melt: the headline workload.
        {"name": "melt-1m", "kind": "melt", "beads": 50, "cx": 10, "cy": 10, "cz": 10, "drop": 0,
         "steps": 100, "precision": "single"},
        # A large four-type mixture without listed terms, thin skin, spatial sort by steps.
        {"name": "mixture-2m", "kind": "mixture", "cx": 13, "cy": 12, "cz": 13, "drop": 33,
         "steps": 100},
        # A melt on the binary64 build.
        {"name": "melt-80k-f64", "kind": "melt", "beads": 50, "cx": 5, "cy": 4, "cz": 4, "drop": 1,
         "steps": 50, "precision": "double"},
        # Sampling: independent fluids of uneven size advanced together.
        {"name": "replicas-64", "kind": "replicas", "count": 64, "n_min": 500, "n_max": 20000,
         "steps": 80},
        # The same for bead-spring melts.
        {"name": "melt-replicas-24", "kind": "melt_replicas", "count": 24, "side_min": 10,
         "side_max": 27, "steps": 100},
        # Forces and energy of one snapshot, then of the next: validation, analysis.
        {"name": "forces-100k", "kind": "forces", "cx": 5, "cy": 5, "cz": 4, "drop": 0,
         "frames": 2},
        # One force-matching training step over a few snapshots of a four-type system.
        {"name": "match-100k", "kind": "match", "cx": 5, "cy": 5, "cz": 4, "drop": 17,
         "frames": 4},
        # Position and parameter gradients of a loss of forces and energies, full force field.
        {"name": "gradient-300k", "kind": "gradient", "cx": 7, "cy": 6, "cz": 7, "drop": 11,
         "frames": 2},
        # Backprop through a short trajectory.
        {"name": "trajectory-18k", "kind": "trajectory", "cx": 3, "cy": 3, "cz": 2, "drop": 5,
         "steps": 20, "every": 10},
    ]


def _copies(rng, least, most):
    """Copies along three axes whose product is near a log-uniform total."""
    total = math.exp(rng.uniform(math.log(least), math.log(most)))
    a = max(1, round(total ** (1 / 3) * rng.uniform(0.8, 1.25)))
    b = max(1, round((total / a) ** 0.5 * rng.uniform(0.8, 1.25)))
    c = max(1, int(total / (a * b)))
    return {"cx": a, "cy": b, "cz": c}


def draw(rng):
    kind = rng.choice(["fluid", "script", "melt", "melt", "melt", "mixture", "mixture", "replicas",
                       "melt_replicas", "forces", "match", "gradient", "trajectory"])
    case = {"kind": kind}
    if kind in ("fluid", "script"):
        case |= {"base": rng.choice([500, 633, 847, 1000])} | _copies(rng, 1, 32)
        case |= {"drop": rng.randrange(0, 20),
                 "steps": 20 * rng.randrange(2, 6 if kind == "fluid" else 11)}
    elif kind == "melt":
        double = rng.random() < 0.25
        case |= {"beads": rng.choice([20, 25, 40, 50])} | _copies(rng, 2, 100 if double else 900)
        case |= {"drop": rng.randrange(0, 15), "steps": rng.randrange(30, 90),
                 "precision": "double" if double else "single"}
    elif kind == "mixture":
        case |= _copies(rng, 4, 1800) | {"drop": rng.randrange(0, 99),
                                         "steps": rng.randrange(30, 90)}
    elif kind == "replicas":
        case |= {"count": rng.randrange(8, 64), "n_min": 500,
                 "n_max": round(math.exp(rng.uniform(math.log(1000), math.log(20000)))),
                 "steps": rng.randrange(30, 81)}
    elif kind == "melt_replicas":
        case |= {"count": rng.randrange(4, 24), "side_min": 10, "side_max": rng.randrange(12, 28),
                 "steps": rng.randrange(40, 100)}
    elif kind == "trajectory":
        steps = rng.randrange(8, 21)
        case |= _copies(rng, 1, 18) | {"drop": rng.randrange(0, 9), "steps": steps,
                                       "every": rng.randrange(3, steps + 1)}
    else:
        case |= _copies(rng, 1, 260 if kind == "gradient" else 100)
        case |= {"drop": rng.randrange(0, 19)}
        case |= {"frames": rng.randrange(1, 3 if kind == "gradient" else 5)}
    return case


# ------------------------------------------------------------------------ systems


def _pair_force(x, box, eps24, sig2, rc, excluded, cap):
    """LJ forces of a small periodic cell, all pairs, capped per pair."""
    d = x[:, None, :] - x[None, :, :]
    d = d - box * torch.round(d / box)
    r2 = (d * d).sum(-1)
    u = torch.where((r2 < rc * rc) & ~excluded, 1.0 / r2.clamp_min(1e-12), torch.zeros_like(r2))
    s6 = (sig2 * u) ** 3
    s = eps24 * u * (2.0 * s6 * s6 - s6)
    return (s.clamp(-cap, cap)[:, :, None] * d).sum(1)


def _bonded_energy(x, w):
    """Harmonic bonds and angles of equal chains x [chains, beads, 3] (unwrapped)."""
    b = x[:, 1:] - x[:, :-1]
    r = (b * b).sum(-1).sqrt()
    e = 0.5 * float(w.bond_k[0]) * ((r - float(w.bond_r0[0])) ** 2).sum()
    if len(w.angles):
        p, q = -b[:, :-1], b[:, 1:]
        n = torch.linalg.cross(p, q)
        t = torch.atan2((n * n).sum(-1).clamp_min(1e-16).sqrt(), (p * q).sum(-1))
        e = e + 0.5 * float(w.angle_k[0]) * ((t - math.radians(float(w.angle_theta0[0]))) ** 2).sum()
    return e


@functools.lru_cache(maxsize=None)
def _cell(kind, base, beads):
    """A relaxed periodic cell: (workload of the cell, unwrapped positions [n, 3], chains)."""
    chains = 0
    if kind == "fluid":
        w = W.lj_box(base, 0.8442, 1.0, seed=base)
    elif kind == "melt":
        chains = 1000 // beads
        w = W.polymer_melt(n_chains=chains, beads_per_chain=beads, seed=beads)
    elif kind == "mixture":
        w = W.lj_mixture(n=1000)
    else:
        chains, beads = 5, 100
        w = W.polymer_solvent(n_chains=chains, beads_per_chain=beads, n_solvent=500)
    n = w.n
    f64 = functools.partial(torch.tensor, dtype=torch.float64, device=DEVICE)
    box = f64((w.box_bound[1] - w.box_bound[0]).astype(np.float64))
    x = w.positions.astype(np.float64)
    if chains:  # unwrap every chain along its bonds
        c = x[:chains * beads].reshape(chains, beads, 3)
        b = np.diff(c, axis=1)
        L = box.cpu().numpy()
        b -= L * np.round(b / L)
        c[:, 1:] = c[:, :1] + np.cumsum(b, axis=1)
    x, t = f64(x), torch.tensor(w.types.astype(np.int64) - 1, device=DEVICE)
    eps24 = 24.0 * f64(w.lj_epsilon)[t][:, t]
    sig2 = f64(w.lj_sigma)[t][:, t] ** 2
    at = torch.arange(n, device=DEVICE)
    excluded = at[:, None] == at[None, :]
    if chains:
        m = torch.where(at < chains * beads, at // beads, at + chains)
        excluded |= (m[:, None] == m[None, :]) & ((at[:, None] - at[None, :]).abs() <= 2)
    mass, kt = float(w.masses[0]), w.kb * w.temperature
    v = f64(W.maxwell_boltzmann(np.random.default_rng(1), w.masses, w.temperature, w.kb))
    dt, steps = w.dt, 500
    for k in range(steps):
        cap = 2000.0 if k < steps // 2 else 1e9
        f = _pair_force(x, box, eps24, sig2, float(w.cutoff), excluded, cap)
        if chains:
            c = x[:chains * beads].reshape(chains, beads, 3).clone().requires_grad_(True)
            g, = torch.autograd.grad(_bonded_energy(c, w), c)
            f = f.clone()
            f[:chains * beads] -= g.reshape(-1, 3)
        v = v + (dt / mass) * f.clamp(-1e4, 1e4)
        t_now = mass * (v * v).sum() / (3 * n - 3)
        v = v * (1.0 + 0.1 * (kt / t_now - 1.0)).clamp(0.25, 4.0).sqrt()
        x = x + dt * v
    x = x.cpu().numpy()
    if not np.isfinite(x).all():
        raise RuntimeError(f"the {kind} cell did not relax")
    return w, x, chains, beads


def _system(kind, case, rng, shuffle=False):
    """The cell repeated cx x cy x cz times, shifted and jittered, as a Workload. drop leaves out
    that many molecules (chains, or single beads where there are none). shuffle puts the molecules
    in random order, as a snapshot taken long after its set-up has them in space."""
    w, x, chains, beads = _cell(kind, case.get("base", 1000), case.get("beads", 50))
    L = (w.box_bound[1] - w.box_bound[0]).astype(np.float64)
    m = np.array([case["cx"], case["cy"], case["cz"]])
    offset = np.stack(np.meshgrid(*[np.arange(c) for c in m], indexing="ij"), -1).reshape(-1, 1, 3)
    pos = x[None] + offset * L
    copies, n0 = pos.shape[0], w.n
    nc = chains * beads
    box = L * m
    # molecules: every copy's chains, then every copy's single beads
    mols = [pos[:, :nc].reshape(-1, beads, 3)] if chains else []
    mol_types = [np.tile(w.types[:nc].reshape(chains, beads), (copies, 1))] if chains else []
    if nc < n0:
        mols.append(pos[:, nc:].reshape(-1, 1, 3))
        mol_types.append(np.tile(w.types[nc:].reshape(-1, 1), (copies, 1)))
    keep = []
    for k, q in enumerate(mols):
        drop = min(case["drop"], len(q) // 10) if k == len(mols) - 1 or not chains else 0
        if chains and k == 0 and nc == n0:
            drop = min(case["drop"], len(q) // 10)
        gone = rng.choice(len(q), size=drop, replace=False)
        order = np.delete(np.arange(len(q)), gone)
        keep.append(rng.permutation(order) if shuffle else order)
    mols = [q[k] for q, k in zip(mols, keep)]
    mol_types = [q[k] for q, k in zip(mol_types, keep)]
    p = np.concatenate([q.reshape(-1, 3) for q in mols])
    types = np.concatenate([q.reshape(-1) for q in mol_types])
    n = p.shape[0]
    spacing = float(np.cbrt(np.prod(box) / n))
    p = p + rng.uniform(0, 1, 3) * box + rng.uniform(-0.01, 0.01, p.shape) * spacing
    hi = box.astype(np.float32)
    p32 = np.mod(p, box).astype(np.float32)
    p32 = np.where(p32 >= hi, np.float32(0), p32)
    masses = np.full(n, w.masses[0], np.float32)
    out = dict(positions=p32, types=types, masses=masses, tags=None, images=None,
               box_bound=np.stack([np.zeros(3, np.float32), hi]),
               velocities=W.maxwell_boltzmann(rng, masses, w.temperature, w.kb))
    n_chains = len(mols[0]) if chains else 0
    tags = np.arange(1, n_chains * beads + 1, dtype=np.uint32).reshape(n_chains, beads if chains else 1)
    mol = np.repeat(np.arange(1, n_chains + 1, dtype=np.uint32), beads if chains else 0)
    out["molecule_ids"] = np.concatenate(
        [mol, np.arange(n_chains + 1, n_chains + 1 + n - mol.size, dtype=np.uint32)])

    def chain_terms(width):
        if not chains:
            return np.zeros((0, width + 1), np.uint32)
        cols = [tags[:, k:beads - (width - 1) + k] for k in range(width)]
        return np.stack(cols + [np.ones_like(cols[0])], -1).reshape(-1, width + 1)

    if chains:
        out["bonds"] = chain_terms(2)
    if len(w.angles):
        out["angles"] = chain_terms(3)
    if len(w.dihedrals):
        out["dihedrals"] = chain_terms(4)
    out["name"] = f"{kind}_{n}"
    if kind == "fluid":  # the fluid's run settings: constant energy, checked every tenth step
        out |= dict(rebuild_check_every=10, berendsen=False)
    elif kind in ("solvent", "mixture"):
        out |= dict(berendsen=False)
    return w.with_(**out)


def _replicas(case, rng):
    """The replicas of a batch: their sizes belong to the case, their beads to the seed."""
    sizes = np.random.default_rng(case["count"])
    count, out = case["count"], []
    for _ in range(count):
        seed = int(rng.integers(1 << 31))
        if case["kind"] == "replicas":
            n = round(math.exp(sizes.uniform(math.log(case["n_min"]), math.log(case["n_max"]))))
            out.append(W.lj_box(n, sizes.uniform(0.6, 0.9), sizes.uniform(0.8, 1.5), seed=seed,
                                berendsen=True, tau=0.5))
        else:
            side = round(math.exp(sizes.uniform(math.log(case["side_min"]),
                                                math.log(case["side_max"]))))
            beads = int(sizes.choice([20, 30, 40, 50]))
            chains = int(0.95 * side ** 3) // beads
            out.append(W.polymer_melt(n_chains=chains, beads_per_chain=beads,
                                      density=chains * beads / (0.48 * side) ** 3, seed=seed))
    return out


def _snapshots(w, count, rng):
    """Independent frames: the system shifted as a whole and jittered, wrapped into the box."""
    L = (w.box_bound[1] - w.box_bound[0]).astype(np.float64)
    hi = w.box_bound[1]
    out = []
    for _ in range(count):
        p = w.positions.astype(np.float64) + rng.uniform(0, 1, 3) * L
        p = np.mod(p + rng.uniform(-0.01, 0.01, p.shape), L).astype(np.float32)
        out.append(np.where(p >= hi, np.float32(0), p))
    return out


# ----------------------------------------------------------------------- the calls


def _frame_inputs(case, seed):
    """System, frames, targets or loss weights of a frame-mode case, from the seed alone."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    w = _system("melt" if kind == "gradient" else "solvent", case, rng, shuffle=True)
    frames = _snapshots(w, 1 if kind == "trajectory" else case["frames"], rng)
    noise = [(300.0 * rng.standard_normal(w.positions.shape)).astype(np.float32) for _ in frames]
    return w, frames, noise


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind in ("fluid", "melt", "mixture"):
        from beads_amd.capi import Engine
        precision = case.get("precision", "single")
        w = _system(kind, case, rng)
        engine = Engine(w.as_float64() if precision == "double" else w, precision)
        engine.initialize()
        return {"kind": kind, "engine": engine, "steps": case["steps"]}
    if kind == "script":
        return {"kind": kind, "workload": _system("fluid", case, rng).with_(steps=case["steps"]),
                "folder": tempfile.TemporaryDirectory()}
    if kind in ("replicas", "melt_replicas"):
        from beads_amd.capi import Batch
        batch = Batch(_replicas(case, rng))
        batch.autotune(5)
        return {"kind": kind, "batch": batch, "steps": case["steps"]}
    from beads_amd.adjoint import FrameModel
    w, frames, noise = _frame_inputs(case, seed)
    model = FrameModel(w)
    on = functools.partial(torch.tensor, device=DEVICE)
    state = {"kind": kind, "model": model, "params": model.initial_params(),
             "frames": [on(x) for x in frames], "noise": [on(x) for x in noise]}
    if kind == "trajectory":
        state |= {"velocities": on(w.velocities), "steps": case["steps"], "every": case["every"]}
    return state


def _by_tag(s):
    order = np.argsort(s["tags"])
    return {k: s[k][order] for k in ("positions", "velocities", "forces", "images")}


def run(state):
    kind = state["kind"]
    if kind in ("fluid", "melt", "mixture"):
        engine = state["engine"]
        engine.advance(state["steps"], observables_on_last=True)
        s, st = engine.state(), engine.stats()
        out = _by_tag(s) if kind == "fluid" else {
            k: s[k] for k in ("positions", "velocities", "forces", "images", "tags")}
        return out | {"pe": np.array(st.pe), "virial": np.array(st.virial), "ke": float(st.ke)}
    if kind == "script":
        from beads_amd.system import read_snapshot
        w, folder = state["workload"], state["folder"].name
        sim = w.to_simulation()
        sim.set_thermo(every=100, prefix=folder + "/run")
        sim.save_final_state(prefix=folder + "/run")
        sim.set_logging(echo="none")
        sim.execute()
        s = read_snapshot(folder + "/run.state.beadsbin")
        order = np.argsort(s["tags"])
        return {k: np.asarray(s[k])[order] for k in ("positions", "velocities", "images")}
    if kind in ("replicas", "melt_replicas"):
        batch = state["batch"]
        batch.run(state["steps"], observables_on_last=True)
        each = [batch.state(r) for r in range(len(batch.workloads))]
        stats = [batch.stats(r) for r in range(len(batch.workloads))]
        out = {k: np.concatenate([s[k] for s in each])
               for k in ("positions", "velocities", "forces", "images", "tags")}
        return out | {"pe": np.array([list(s.pe) for s in stats]),
                      "ke": np.array([s.ke for s in stats])}
    model, params = state["model"], state["params"]
    if kind == "forces":
        with torch.no_grad():
            got = [model.forces(x, params) for x in state["frames"]]
        return {"forces": [f for f, _ in got], "energy": [e for _, e in got]}
    for t in params.tensors():
        t.grad = None
    if kind == "match":
        from beads_amd.adjoint import force_matching_loss
        loss = force_matching_loss(model, state["frames"], state["noise"], params)
        loss.backward()
        return {"loss": loss.detach(), "params": [t.grad for t in params.tensors()]}
    xs = [x.clone().requires_grad_(True) for x in state["frames"]]
    if kind == "gradient":
        got = [model.forces(x, params) for x in xs]
        loss = sum((f * q).double().sum() * 1e-3 + e * 0.5
                   for (f, e), q in zip(got, state["noise"]))
        loss.backward()
        return {"forces": [f.detach() for f, _ in got], "energy": [e.detach() for _, e in got],
                "x": [x.grad for x in xs], "params": [t.grad for t in params.tensors()]}
    x = xs[0]
    v = state["velocities"].clone().requires_grad_(True)
    xT, vT = model.trajectory(x, v, params, steps=state["steps"], checkpoint_every=state["every"])
    loss = (xT.double() ** 2).sum() * 1e-3 + (vT.double() ** 2).sum()
    loss.backward()
    return {"xT": xT.detach(), "vT": vT.detach(), "x0": x.grad, "v0": v.grad,
            "params": [t.grad for t in params.tensors()]}


# ------------------------------------------------------------- what it cannot do without


def _beads(case):
    kind = case["kind"]
    if kind == "replicas":
        lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
        return case["count"] * (case["n_max"] - case["n_min"]) / max(hi - lo, 1e-9)
    if kind == "melt_replicas":
        a, b = case["side_min"], case["side_max"]
        return case["count"] * 0.95 * (b ** 3 - a ** 3) / (3 * math.log(b / a))
    return case.get("base", 1000) * case["cx"] * case["cy"] * case["cz"]


def work(case):
    """Positions and velocities in, positions, velocities and forces out once per step (once per
    pass for frames), the listed terms' partners; each pair inside the cut-off once per force
    evaluation at 40 operations, a listed term at 100."""
    kind, n = case["kind"], _beads(case)
    real = 8 if case.get("precision") == "double" else 4
    pairs = {"fluid": 27.6, "script": 27.6, "replicas": 24.5, "mixture": 23.7}.get(kind, 30.8)
    terms = {"melt": 3, "melt_replicas": 3, "gradient": 3, "forces": 0.5, "match": 0.5,
             "trajectory": 0.5}.get(kind, 0)
    evaluate = n * (40 * pairs + 100 * terms)
    if kind in ("forces", "match", "gradient"):
        passes = case.get("frames", 1)
        back = kind != "forces"
        return {"bytes": passes * n * (24 + 16 * terms + (36 if back else 0)),
                "flops": passes * evaluate * (3 if back else 1)}
    per_step = n * (15 * real + 12 * terms)
    if kind == "trajectory":
        return {"bytes": 3 * case["steps"] * per_step, "flops": 4 * case["steps"] * evaluate}
    return {"bytes": case["steps"] * per_step, "flops": case["steps"] * (evaluate + 30 * n)}


# ------------------------------------------------------------------ the same in 64 bits


def _pairs(x, w):
    """Ordered pairs (i, j) inside the cut-off, decided on binary32 displacements, less the bonded
    exclusions to distance 2; x [n, 3] binary64 holding binary32 values."""
    box = torch.tensor((w.box_bound[1] - w.box_bound[0]).astype(np.float64), device=DEVICE)
    rc = np.float32(w.cutoff)
    n = x.shape[0]
    grid = torch.clamp((box / (float(rc) * 1.0001)).floor().long(), min=1)
    cell = torch.minimum((x / box * grid).floor().long().clamp_min(0), grid - 1)
    flat = (cell[:, 2] * grid[1] + cell[:, 1]) * grid[0] + cell[:, 0]
    order = torch.argsort(flat, stable=True)
    count = torch.bincount(flat, minlength=int(grid.prod()))
    start = torch.cumsum(count, 0) - count
    mol = torch.tensor(w.molecule_ids.astype(np.int64), device=DEVICE)
    at = torch.arange(n, device=DEVICE)
    steps = [range(-1, 2) if int(g) >= 3 else range(int(g)) for g in grid]
    found = []
    for a in steps[0]:
        for b in steps[1]:
            for c in steps[2]:
                d = torch.tensor([a, b, c], device=DEVICE)
                q = torch.remainder(cell + d, grid)
                q = (q[:, 2] * grid[1] + q[:, 1]) * grid[0] + q[:, 0]
                m = count[q]
                i = torch.repeat_interleave(at, m)
                k = torch.arange(i.numel(), device=DEVICE) - torch.repeat_interleave(
                    torch.cumsum(m, 0) - m, m)
                j = order[start[q][i] + k]
                s = x[i] - x[j]
                s = (s - box * torch.round(s / box)).float()
                r2 = s[:, 0] * s[:, 0] + s[:, 1] * s[:, 1] + s[:, 2] * s[:, 2]
                ok = (r2 < float(rc * rc)) & (i != j)
                if len(w.bonds):
                    ok &= ~((mol[i] == mol[j]) & ((i - j).abs() <= 2))
                found.append(torch.stack([i[ok], j[ok]]))
    return torch.cat(found, 1)


def _lj_and_bonds(x, w, params, pairs):
    """Forces and energy of LJ pairs and harmonic bonds, differentiable in x and the parameters."""
    eps, sig, kb, r0 = params[:4]
    box = torch.tensor((w.box_bound[1] - w.box_bound[0]).astype(np.float64), device=DEVICE)
    t = torch.tensor(w.types.astype(np.int64) - 1, device=DEVICE)
    i, j = pairs
    d = x[i] - x[j]
    d = d - (box * torch.round(d / box)).detach()
    e, s2 = eps[t[i], t[j]], sig[t[i], t[j]] ** 2
    u = 1.0 / (d * d).sum(-1)
    s6 = (s2 * u) ** 3
    f = torch.zeros_like(x).index_add(
        0, i, (24.0 * e * u * (2.0 * s6 * s6 - s6))[:, None] * d)
    pot = 4.0 * e * (s6 * s6 - s6)
    if w.shift:
        c6 = (s2 / float(np.float32(w.cutoff)) ** 2) ** 3
        pot = pot - 4.0 * e * (c6 * c6 - c6)
    energy = 0.5 * pot.sum()
    if len(w.bonds):
        b = torch.tensor(w.bonds.astype(np.int64) - 1, device=DEVICE)
        d = x[b[:, 0]] - x[b[:, 1]]
        d = d - (box * torch.round(d / box)).detach()
        r = (d * d).sum(-1).sqrt()
        stretch = r - r0[b[:, 2]]
        energy = energy + 0.5 * (kb[b[:, 2]] * stretch ** 2).sum()
        p = (-kb[b[:, 2]] * stretch / r)[:, None] * d
        f = f.index_add(0, b[:, 0], p).index_add(0, b[:, 1], -p)
    return f, energy


def _angles_and_dihedrals(x, w, ka, th0, kd):
    box = torch.tensor((w.box_bound[1] - w.box_bound[0]).astype(np.float64), device=DEVICE)

    def disp(p, q):
        d = x[p] - x[q]
        return d - (box * torch.round(d / box)).detach()

    a = torch.tensor(w.angles.astype(np.int64) - 1, device=DEVICE)
    p, q = disp(a[:, 0], a[:, 1]), disp(a[:, 2], a[:, 1])
    n = torch.linalg.cross(p, q)
    th = torch.atan2((n * n).sum(-1).sqrt(), (p * q).sum(-1))
    e = 0.5 * (ka[a[:, 3]] * (th - th0[a[:, 3]] * (math.pi / 180.0)) ** 2).sum()
    b = torch.tensor(w.dihedrals.astype(np.int64) - 1, device=DEVICE)
    v0, v1, v2 = disp(b[:, 0], b[:, 1]), disp(b[:, 2], b[:, 1]), disp(b[:, 2], b[:, 3])
    c0, c1 = torch.linalg.cross(v0, v1), torch.linalg.cross(v1, v2)
    phi = torch.atan2((v1 * v1).sum(-1).sqrt() * (v0 * c1).sum(-1), (c0 * c1).sum(-1))
    d = torch.tensor(w.dihedral_d.astype(np.float64), device=DEVICE)[b[:, 4]]
    m = torch.tensor(w.dihedral_n.astype(np.float64), device=DEVICE)[b[:, 4]]
    return e + (kd[b[:, 4]] * (1.0 + d * torch.cos(m * phi))).sum()


def _params64(w, kind):
    names = ["lj_epsilon", "lj_sigma", "bond_k", "bond_r0"]
    if kind == "gradient":
        names += ["angle_k", "angle_theta0", "dihedral_k"]
    return [torch.tensor(getattr(w, k).astype(np.float64), device=DEVICE, requires_grad=True)
            for k in names]


def _fluid_run(w, steps):
    """Velocity Verlet of a small fluid in binary64, all pairs; velocities and forces by tag."""
    f64 = functools.partial(torch.tensor, dtype=torch.float64, device=DEVICE)
    x, v = f64(w.positions.astype(np.float64)), f64(w.velocities.astype(np.float64))
    box = f64((w.box_bound[1] - w.box_bound[0]).astype(np.float64))
    at = torch.arange(w.n, device=DEVICE)
    same = at[:, None] == at[None, :]
    dt = float(np.float32(w.dt))

    def force():
        return _pair_force(x, box, 24.0, 1.0, float(np.float32(w.cutoff)), same, math.inf)

    f = force()
    for _ in range(steps):
        v = v + 0.5 * dt * f
        x = x + dt * v
        f = force()
        v = v + 0.5 * dt * f
    return v, f


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fluid", "script"):
        w = _system("fluid", case, np.random.default_rng(seed))
        if w.n > 9000:
            return None
        v, f = _fluid_run(w, case["steps"])
        if kind == "script":
            return {"positions": None, "velocities": v, "images": None}
        return {"positions": None, "velocities": v, "forces": f, "images": None, "pe": None,
                "virial": None, "ke": None}
    if kind not in ("forces", "match", "gradient", "trajectory"):
        return None  # thousands of beads over many steps: no plain run of it is quick
    w, frames, noise = _frame_inputs(case, seed)
    xs = [torch.tensor(x.astype(np.float64), device=DEVICE) for x in frames]
    noise = [torch.tensor(x.astype(np.float64), device=DEVICE) for x in noise]
    params = _params64(w, kind)
    if kind == "forces":
        with torch.no_grad():
            got = [_lj_and_bonds(x, w, params, _pairs(x, w)) for x in xs]
        return {"forces": [f for f, _ in got], "energy": [e for _, e in got]}
    if kind == "match":
        scale, total = 1.0 / (len(xs) * w.n * 3), 0.0
        for x, target in zip(xs, noise):
            f, _ = _lj_and_bonds(x, w, params, _pairs(x, w))
            loss = ((f - target) ** 2).sum() * scale
            loss.backward()
            total = total + loss.detach()
        return {"loss": total, "params": [t.grad for t in params]}
    if kind == "gradient":
        out = {"forces": [], "energy": [], "x": []}
        for x, q in zip(xs, noise):
            x.requires_grad_(True)
            f, e = _lj_and_bonds(x, w, params, _pairs(x.detach(), w))
            u = _angles_and_dihedrals(x, w, *params[4:])
            g, = torch.autograd.grad(u, x, create_graph=True)
            f, e = f - g, e + u
            ((f * q).sum() * 1e-3 + e * 0.5).backward()
            for k, t in zip(("forces", "energy", "x"), (f.detach(), e.detach(), x.grad)):
                out[k].append(t)
        return out | {"params": [t.grad for t in params]}
    x = xs[0].clone().requires_grad_(True)
    v = torch.tensor(w.velocities.astype(np.float64), device=DEVICE, requires_grad=True)
    box = torch.tensor((w.box_bound[1] - w.box_bound[0]).astype(np.float64), device=DEVICE)
    dt, mass = float(w.dt), float(w.masses[0])

    def force(q):
        p = torch.remainder(q.detach(), box).float().double()
        return _lj_and_bonds(q, w, params, _pairs(p, w))[0]

    q, p, f = x, v, force(x)
    for _ in range(case["steps"]):
        p = p + (0.5 * dt / mass) * f
        q = q + dt * p
        f = force(q)
        p = p + (0.5 * dt / mass) * f
    loss = (q ** 2).sum() * 1e-3 + (p ** 2).sum()
    loss.backward()
    return {"xT": q.detach(), "vT": p.detach(), "x0": x.grad, "v0": v.grad,
            "params": [t.grad for t in params]}
