"""What a user of this engine has it do, as cases that can be timed and compared.

A case is one call pattern of the public surface (`GpuSimulation`, `Batch`) on
one system. `kind` says which:

- "run":      a stretch of molecular dynamics and the frame written after it
              (`run`, `read_state`), under the thermostat or thermostat and
              barostat;
- "batch":    the same for many replicas stepped together (`Batch.run`);
- "energy":   a single point, every energy term and the forces (`evaluate`);
- "forces":   the forces alone (`evaluate(energies=False)`);
- "minimise": steepest descent from a built structure (`set_state`,
              `minimise`, `read_positions`).

Systems are the seeded solvated-peptide builder's (alanine dipeptide and TIP3P
water, or water alone, at 1 g/cm^3) and the packaged truncated octahedron.
"""
import math

import numpy as np
import torch

import rainmd_amd as R

WATERS_PER_NM3 = 33.4      # liquid water at 1 g/cm^3
TEMPERATURE = 300.0


def _edge(waters):
    """The cube edge (nm) that holds `waters` at liquid density."""
    return round((waters / WATERS_PER_NM3) ** (1.0 / 3.0), 4)


def _single(name, kind, waters, edge=None, **more):
    case = {"name": name, "kind": kind, "waters": waters, "edge": edge or _edge(waters), "solute": True, "cutoff": 0.9,
            "barostat": False, "skin": 0.0, "flexible": False, "ewald": 5e-4, "grid": 0, "steps": 0}
    case.update(more)
    if name is None:
        del case["name"]
    return case


def listed():
    return [
        # the smallest production run: the solvated dipeptide at constant volume, a frame every 50 steps
        _single("nvt-1189", "run", 389, 2.2816, steps=50),
        # the engine's headline workload: 2854 atoms with the barostat, a move every 25 steps
        _single("npt-2854", "run", 944, 3.0539, steps=50, barostat=True),
        # a sheared (truncated octahedron) box, the usual choice for a globular solute
        {"name": "npt-octahedron-1315", "kind": "run", "file": "ala-oct", "cutoff": 0.9, "barostat": True, "skin": 0.0,
         "flexible": False, "ewald": 5e-4, "steps": 50},
        # an ordinary solvated system of about twelve thousand atoms
        _single("npt-12022", "run", 4000, steps=50, barostat=True),
        # twenty-four thousand atoms with the long cutoff some force fields ask for
        _single("nvt-24022-rc12", "run", 8000, steps=25, cutoff=1.2),
        # the large water box of this repository's benchmark, at its skin
        _single("nvt-100200", "run", 33400, 10.0, solute=False, cutoff=1.0, skin=0.15, grid=112, steps=25),
        # the same size at a tighter Ewald tolerance: a grid of twice the points per axis
        _single("nvt-100222-tight", "run", 33400, cutoff=0.9, ewald=5e-5, steps=25),
        # the largest: a solvated complex with the default skin
        _single("nvt-180022", "run", 60000, cutoff=1.0, steps=25),
        # an ensemble of uneven replicas (boxes of 2.2 to 5 nm), each with its own barostat
        {"name": "batch-64", "kind": "batch", "replicas": 64, "low": 2.2, "high": 5.0, "barostat": True, "cutoff": 0.9,
         "steps": 25},
        # single points: rescoring a frame with every term
        _single("energy-100200", "energy", 33400, 10.0, solute=False, cutoff=1.0, skin=0.15, grid=112),
        # forces alone, for a caller with an integrator of its own
        _single("forces-2854", "forces", 944, 3.0539),
        # relaxing a freshly built system before dynamics
        _single("minimise-2854", "minimise", 944, 3.0539, steps=50),
    ]


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "batch", "energy", "forces", "minimise"])
    if kind == "batch":
        low = round(rng.uniform(2.2, 3.2), 2)
        return {"kind": "batch", "replicas": rng.randrange(3, 49), "low": low, "high": round(low + rng.uniform(0.1, 1.8), 2),
                "barostat": rng.random() < 0.5, "cutoff": 0.9, "steps": 25}
    cutoff = rng.choice([0.8, 0.9, 0.9, 1.0, 1.0, 1.2])
    smallest = WATERS_PER_NM3 * (2.0 * cutoff + 0.45) ** 3
    largest = {"run": 40000, "energy": 40000, "forces": 40000, "minimise": 12000}[kind]
    waters = int(round(math.exp(rng.uniform(math.log(smallest), math.log(largest)))))
    if waters > 20000:
        cutoff = min(cutoff, 1.0)
    return _single(None, kind, waters, solute=rng.random() < 0.7, cutoff=cutoff,
                   barostat=kind == "run" and rng.random() < 0.5, skin=rng.choice([0.0, 0.0, 0.15]),
                   flexible=rng.random() < 0.2, ewald=rng.choice([5e-4, 5e-4, 5e-4, 1e-4]),
                   steps={"run": 50 if waters < 8000 and rng.random() < 0.5 else 25,
                          "minimise": rng.randrange(20, 51)}.get(kind, 0))


# ---- what a user's program has in hand --------------------------------------

def _system(case, seed):
    if case.get("file"):
        topology = R.Topology.load(case["file"] + ".prmtop")
        return R.System.build(topology, R.Coordinates.load(case["file"] + ".inpcrd"), cutoff=case["cutoff"])
    rigid = not case["flexible"]
    return R.System.solvated(case["waters"], case["edge"], seed, include_solute=case["solute"], cutoff=case["cutoff"],
                             constraints="HBonds" if rigid else "none", rigid_water=rigid)


def _options(case):
    o = {"temperature": TEMPERATURE}
    if case["barostat"]:
        o.update(pressure=1.0, barostat_interval=25)
    if case.get("flexible"):
        o["timestep"] = 0.0005  # unconstrained bonds to hydrogen
    if case.get("ewald"):
        o["ewald_tolerance"] = case["ewald"]
    if case.get("grid"):
        o["grid"] = [case["grid"]] * 3
    if case.get("skin"):
        o["skin"] = case["skin"]
    return o


def _relax(sim, system, seed):
    """Minimise and give velocities, at more than the target temperature, as
    half of it goes into the potential energy of the relaxed structure."""
    sim.minimise(max_iterations=150, force_tolerance=1000.0)
    sim.set_state(sim.read_positions().astype(np.float64), R.maxwell_boltzmann(system, 1.5 * TEMPERATURE, seed), step=0)


def prepare(case, seed):
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    system = _system(case, seed)
    sim = R.GpuSimulation(system, seed=seed, **_options(case))
    if case["kind"] == "minimise":
        return {"case": case, "sim": sim, "system": system, "start": system.positions.copy()}
    _relax(sim, system, seed)
    sim.run(200 if system.atom_count < 30000 else 100, 25)
    return {"case": case, "sim": sim, "system": system}


def _replicas(case):
    """(waters, edge) of each replica: edges spread evenly over [low, high]."""
    n = case["replicas"]
    edges = [case["low"] + (case["high"] - case["low"]) * (r + 0.5) / n for r in range(n)]
    return [(int(WATERS_PER_NM3 * e ** 3) - 8, e) for e in edges]


def _prepare_batch(case, seed):
    shapes = _replicas(case)
    seeds = [(seed * 1000 + r) % (1 << 31) for r in range(len(shapes))]
    systems = [R.System.solvated(w, e, s, cutoff=case["cutoff"]) for (w, e), s in zip(shapes, seeds)]
    batch = R.Batch(systems, seeds=seeds, **_options(case))
    sims = [batch.replica(r) for r in range(len(systems))]
    for sim, system, s in zip(sims, systems, seeds):
        _relax(sim, system, s)
    batch.run(50, 25)
    return {"case": case, "batch": batch, "sims": sims, "system": systems}


# ---- one pass ----------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        state["sim"].run(case["steps"], 25)
        return state["sim"].read_state()
    if kind == "batch":
        state["batch"].run(case["steps"], 25)
        frames = [sim.read_state() for sim in state["sims"]]
        return {"positions": np.concatenate([f["positions"] for f in frames]),
                "velocities": np.concatenate([f["velocities"] for f in frames]),
                "volumes": np.array([f["volume"] for f in frames])}
    if kind == "minimise":
        state["sim"].set_state(state["start"])
        result = state["sim"].minimise(max_iterations=case["steps"], force_tolerance=100.0)
        return {"positions": state["sim"].read_positions(), "potential": result["potential"]}
    if kind == "energy":
        terms, forces = state["sim"].evaluate()
        return {"forces": forces, "terms": np.array([terms[name] for name in TERMS])}
    return {"forces": state["sim"].evaluate(energies=False)[1]}


TERMS = ("bonded", "lennard_jones", "coulomb_direct", "coulomb_reciprocal", "potential")


# ---- the work a pass cannot do without ---------------------------------------

def _evaluation_flops(atoms, volume, cutoff):
    """Unique pairs within the cutoff at 78 operations each (distance, both
    LJ powers and the screened Coulomb force), order-5 spread and gather (10
    operations at each of 125 points) and two real transforms of the grid
    (points of about 0.1 nm)."""
    pairs = 0.5 * atoms * (atoms / volume) * 4.0 / 3.0 * math.pi * cutoff ** 3
    points = volume * 1000.0
    return 78.0 * pairs + 1250.0 * atoms + 2 * 2.5 * points * math.log2(points)


def work(case):
    if case["kind"] == "batch":
        shapes = [(3 * w + 22, e ** 3) for w, e in _replicas(case)]
    elif case.get("file"):
        shapes = [(1315, 16.9)]
    else:
        shapes = [(3 * case["waters"] + (22 if case["solute"] else 0), case["edge"] ** 3)]
    atoms = sum(n for n, _ in shapes)
    flops = sum(_evaluation_flops(n, v, case["cutoff"]) for n, v in shapes)
    if case["kind"] in ("run", "batch"):  # positions and velocities read and written each step
        return {"bytes": 48.0 * atoms * case["steps"], "flops": flops * case["steps"]}
    if case["kind"] == "minimise":
        return {"bytes": 24.0 * atoms * case["steps"], "flops": flops * case["steps"]}
    return {"bytes": 36.0 * atoms, "flops": flops}


def tolerance(case):
    """Positions and velocities are stored in 32 bits and a step's forces carry
    about 2e-6 of relative error (their 2-norm against 64 bits), so two
    correct single points are that close. Along a trajectory the difference
    grows about tenfold in 100 fs: with the reciprocal sum's transforms in
    another order, or the starting positions moved by one rounding, the
    velocities after two stretches of 50 steps were 3e-4 apart (2-norm; the
    worst atom 3e-2), after minimising the positions 1.3e-7."""
    if case["kind"] in ("energy", "forces"):
        return {"rel": 1e-5}
    if case["kind"] == "minimise":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1.5e-3, "max": 0.15}


# ---- the same values in 64 bits ----------------------------------------------

COULOMB = 138.935456  # kJ nm / (mol e^2)


def exact(case, seed):
    """Single points in plain torch, 64 bits, at the positions the pass
    evaluates. Trajectories and descents have no such value: each step rounds
    the stored positions to 32 bits, and a volume move or a trial step is a
    decision; their forces are the single points'."""
    if case["kind"] not in ("energy", "forces"):
        return None
    state = prepare(case, seed)
    sim, system = state["sim"], state["system"]
    frame, plan = sim.read_state(), sim.diagnostics()
    device = torch.device("cuda")
    x = torch.tensor(frame["positions"].reshape(-1, 3), dtype=torch.float64, device=device)
    box = torch.tensor(frame["box_vectors"].reshape(3, 3), dtype=torch.float64, device=device)
    alpha, grid = plan["pme_alpha"], list(plan["pme_grid"])
    charges = torch.tensor(system.charges, dtype=torch.float64, device=device)
    terms, forces = {}, torch.zeros_like(x)

    bonded, f = _gradient(lambda p: _bonded(p, system, device), x)
    forces += f
    terms["bonded"] = bonded
    reciprocal, f = _gradient(lambda p: _reciprocal(p, charges, box, alpha, grid), x)
    forces += f
    terms["coulomb_reciprocal"] = reciprocal
    lj, coulomb, f = _direct(x, charges, box, alpha, system, device)
    forces += f
    (lj14, coulomb14), f = _gradient(lambda p: _exceptions(p, box, alpha, system, device), x)
    forces += f
    terms["lennard_jones"], terms["coulomb_direct"] = lj + lj14, coulomb + coulomb14
    volume = float(torch.linalg.det(box))
    own = -COULOMB * alpha / math.sqrt(math.pi) * float((charges ** 2).sum())
    net = -COULOMB * math.pi / (2 * volume * alpha ** 2) * float(charges.sum()) ** 2
    tail = _tail(system, volume)
    terms["potential"] = sum(terms.values()) + own + net + tail
    out = {"forces": forces.cpu().numpy()}
    if case["kind"] == "energy":
        out["terms"] = np.array([terms[name] for name in TERMS])
    return out


def _gradient(energy, x):
    """(energy or tuple of energies, the forces of their sum)."""
    p = x.detach().clone().requires_grad_(True)
    e = energy(p)
    parts = e if isinstance(e, tuple) else (e,)
    total = sum(parts)
    f = -torch.autograd.grad(total, p)[0] if total.requires_grad else torch.zeros_like(x)
    values = tuple(float(v) for v in parts)
    return (values if isinstance(e, tuple) else values[0]), f


def _on(device, *arrays):
    return [torch.as_tensor(np.asarray(a), device=device).to(torch.float64 if np.asarray(a).dtype.kind == "f" else torch.int64)
            for a in arrays]


def _bonded(p, s, device):
    a, b, k, r0 = _on(device, s.bond_a, s.bond_b, s.bond_k, s.bond_r0)
    total = (0.5 * k * ((p[a] - p[b]).norm(dim=1) - r0) ** 2).sum()
    a, b, c, k, t0 = _on(device, s.angle_a, s.angle_b, s.angle_c, s.angle_k, s.angle_theta0)
    u, v = p[a] - p[b], p[c] - p[b]
    theta = torch.atan2(torch.linalg.cross(u, v).norm(dim=1), (u * v).sum(1))
    total = total + (0.5 * k * (theta - t0) ** 2).sum()
    a, b, c, d, k, n, phase = _on(device, s.torsion_a, s.torsion_b, s.torsion_c, s.torsion_d, s.torsion_k,
                                  s.torsion_periodicity, s.torsion_phase)
    b1, b2, b3 = p[b] - p[a], p[c] - p[b], p[d] - p[c]
    n1, n2 = torch.linalg.cross(b1, b2), torch.linalg.cross(b2, b3)
    phi = torch.atan2((torch.linalg.cross(n1, n2) * b2).sum(1) / b2.norm(dim=1), (n1 * n2).sum(1))
    return total + (k * (1 + torch.cos(n * phi - phase))).sum()


def _image(d, box):
    for axis in (2, 1, 0):
        d = d - torch.round(d[..., axis:axis + 1] / box[axis, axis]) * box[axis]
    return d


def _exceptions(p, box, alpha, s, device):
    """1-4 pairs at their scaled parameters, and what the reciprocal sum counts of every excluded pair taken back."""
    a, b, qq, A, B = _on(device, s.exception_a, s.exception_b, s.exception_charge_product, s.exception_lj_a,
                         s.exception_lj_b)
    charges = torch.as_tensor(s.charges, device=device)
    r = _image(p[a] - p[b], box).norm(dim=1)
    lj = (A / r ** 12 - B / r ** 6).sum()
    full = COULOMB * charges[a] * charges[b]
    return lj, (COULOMB * qq / r - full * torch.erf(alpha * r) / r).sum()


def _direct(x, charges, box, alpha, s, device):
    n = len(x)
    types, A, B = _on(device, s.atom_types, s.lj_a.reshape(s.type_count, -1), s.lj_b.reshape(s.type_count, -1))
    start = np.asarray(s.exclusion_start)
    of, partner = _on(device, np.repeat(np.arange(n), np.diff(start)), s.exclusion_partners)
    excluded = torch.unique(of * n + partner)
    lj = coulomb = 0.0
    forces = torch.zeros_like(x)
    rows = max(1, min(n, 40_000_000 // n))
    for first in range(0, n, rows):
        d = _image(x[first:first + rows, None] - x[None], box)
        i, j = torch.nonzero((d * d).sum(-1) <= s.cutoff ** 2, as_tuple=True)
        d = d[i, j]
        i = i + first
        key = i * n + j
        at = torch.searchsorted(excluded, key).clamp(max=max(0, len(excluded) - 1))
        keep = (i != j) & ((excluded[at] != key) if len(excluded) else True)
        i, j, d = i[keep], j[keep], d[keep]
        r2 = (d * d).sum(1)
        r = r2.sqrt()
        a, b = A[types[i], types[j]], B[types[i], types[j]]
        i6 = 1 / r2 ** 3
        qq = COULOMB * charges[i] * charges[j]
        screened = torch.erfc(alpha * r) / r
        lj += 0.5 * float(((a * i6 - b) * i6).sum())
        coulomb += 0.5 * float((qq * screened).sum())
        scalar = (12 * a * i6 - 6 * b) * i6 / r2
        scalar += qq * (screened + 2 * alpha / math.sqrt(math.pi) * torch.exp(-alpha ** 2 * r2)) / r2
        forces.index_add_(0, i, scalar[:, None] * d)
    return lj, coulomb, forces


def _spline(w):
    """Order-5 cardinal B-spline weights at offsets w in [0, 1): entry k is the weight of grid point floor(u) - 4 + k."""
    v = [w, 1 - w]  # v[j] = M_n(w + j), raised from n = 2 to 5
    for n in range(3, 6):
        lower = [0.0] + v + [0.0]
        v = [((w + j) * lower[j + 1] + (n - w - j) * lower[j]) / (n - 1) for j in range(n)]
    return torch.stack(v[::-1], dim=-1)


def _reciprocal(p, charges, box, alpha, grid):
    inverse = torch.linalg.inv(box)  # columns are the reciprocal vectors
    volume = torch.linalg.det(box)
    u = p @ inverse
    u = (u - torch.floor(u.detach())) * torch.tensor(grid, dtype=p.dtype, device=p.device)
    base = torch.floor(u.detach())
    weights = _spline(u - base)  # atoms, axis, 5
    base = base.to(torch.int64)
    ks = torch.arange(5, device=p.device) - 4
    index = [torch.remainder(base[:, a:a + 1] + ks, grid[a]) for a in range(3)]
    flat = ((index[0][:, :, None, None] * grid[1] + index[1][:, None, :, None]) * grid[2] + index[2][:, None, None, :])
    value = (charges[:, None, None, None] * weights[:, 0, :, None, None] * weights[:, 1, None, :, None]
             * weights[:, 2, None, None, :])
    q = torch.zeros(grid[0] * grid[1] * grid[2], dtype=p.dtype, device=p.device)
    q = q.index_add(0, flat.reshape(-1), value.reshape(-1)).reshape(grid)
    s = torch.fft.rfftn(q)
    m, moduli = [], []
    at = torch.arange(5, dtype=p.dtype, device=p.device)
    knots = _spline(torch.zeros(1, dtype=p.dtype, device=p.device))[0]
    for a in range(3):
        k = torch.fft.fftfreq(grid[a], 1.0 / grid[a], device=p.device, dtype=p.dtype)
        b = (knots * torch.exp(2j * math.pi * k[:, None] * at / grid[a])).sum(1).abs() ** 2
        for z in (b < 1e-7).nonzero().flatten().tolist():  # an odd order's Nyquist point: its neighbours' mean
            b[z] = 0.5 * (b[z - 1] + b[(z + 1) % grid[a]])
        if a == 2:
            k, b = k[: grid[2] // 2 + 1].abs(), b[: grid[2] // 2 + 1]
        m.append(k)
        moduli.append(b)
    wave = (m[0][:, None, None, None] * inverse[:, 0] + m[1][None, :, None, None] * inverse[:, 1]
            + m[2][None, None, :, None] * inverse[:, 2])
    m2 = (wave * wave).sum(-1)
    m2[0, 0, 0] = 1.0
    g = torch.exp(-math.pi ** 2 * m2 / alpha ** 2) / (
        m2 * moduli[0][:, None, None] * moduli[1][None, :, None] * moduli[2][None, None, :])
    g[0, 0, 0] = 0.0
    twice = torch.full((grid[2] // 2 + 1,), 2.0, dtype=p.dtype, device=p.device)
    twice[0] = 1.0
    if grid[2] % 2 == 0:
        twice[-1] = 1.0
    return COULOMB / (2 * math.pi * volume) * (twice * g * (s.real ** 2 + s.imag ** 2)).sum()


def _tail(s, volume):
    """The mean LJ energy beyond the cutoff, over ordered pairs of types (an atom paired with its own kind N(N+1)/2 times)."""
    count = np.bincount(s.atom_types, minlength=s.type_count).astype(np.float64)
    pairs = (np.outer(count, count) + np.diag(count)) * len(s.atom_types) / (len(s.atom_types) + 1)
    mean = [float((pairs * t.reshape(s.type_count, -1)).sum()) for t in (s.lj_a, s.lj_b)]
    return 2.0 * math.pi / volume * (mean[0] / (9 * s.cutoff ** 9) - mean[1] / (3 * s.cutoff ** 3))
