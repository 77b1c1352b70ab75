"""The work users have this library do, as cases that can be timed and compared.

A case names one kind of call through the public entry points (the Python
binding, or the C ABI where the binding has no wrapper) and its sizes:

  step      an MD context advances and hands over a frame
  batch     replicas advance together and hand over the energies that an exchange decides on
  npt       the same under a Monte Carlo barostat
  evaluate  energy and forces of conformations in host memory
  resident  forces only, positions and forces in device memory
  charges   the charge mesh of a constant-potential solver, host buffers
  noalloc   its allocation-free form, device buffers

Systems are boxes of 3-site water at about liquid density, as in the repository's
tests and benchmark.  In mixed precision, forces come from FP32 arithmetic: what
depends on them is handed over in single precision, as trajectory files, FP32
consumers of the forces and exchange criteria hold it.  Energies of the evaluation
calls (FP64 sums in either precision) and all results of the plain FP64 form stay FP64.
"""
import ctypes
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openmm-rs_amd"))

import ommhip  # noqa: E402

DENSITY = 33.4  # molecules / nm^3
TOLERANCE = 5e-4
ONE_4PI_EPS0 = 138.93545764438198


def listed():
    return [
        # The smallest box the tests use: a step is launch latency.
        {"name": "step-900", "kind": "step", "molecules": 300, "edge": 2.1, "cutoff": 0.9, "steps": 50},
        # The benchmark's headline system.
        {"name": "step-23550", "kind": "step", "molecules": 7850, "edge": 6.17, "cutoff": 0.9, "steps": 50},
        # The benchmark's large system, where the arithmetic counts.
        {"name": "step-300000", "kind": "step", "molecules": 100000, "edge": 14.42, "cutoff": 1.0, "steps": 20},
        # Rigid water (three constraints a molecule) of an ordinary box, at the tolerance that
        # drift-sensitive runs set.
        {"name": "step-rigid-6000", "kind": "step", "molecules": 2000, "edge": 3.92, "cutoff": 0.9, "steps": 50,
         "rigid": True},
        # The benchmark's 64 uneven replicas between two exchanges.
        {"name": "batch-64", "kind": "batch", "replicas": 64, "lo": 500, "hi": 6000, "steps": 20},
        # Small replicas at constant pressure, two barostat moves a pass.
        {"name": "npt-24", "kind": "npt", "replicas": 24, "lo": 300, "hi": 2000, "steps": 50},
        # Two unrelated conformations of the smallest box: a call from an outer program.
        {"name": "evaluate-900", "kind": "evaluate", "molecules": 300, "edge": 2.1, "cutoff": 0.9,
         "method": "PME", "double": False},
        # The tests' 9,000-atom box.
        {"name": "evaluate-9000", "kind": "evaluate", "molecules": 3000, "edge": 4.48, "cutoff": 0.9,
         "method": "PME", "double": False},
        # The same in plain FP64, as references are made.
        {"name": "evaluate-9000-fp64", "kind": "evaluate", "molecules": 3000, "edge": 4.48, "cutoff": 0.9,
         "method": "PME", "double": True},
        # Forces for an integrator that lives outside the library, on the same device.
        {"name": "resident-23550", "kind": "resident", "molecules": 7850, "edge": 6.17, "cutoff": 0.9,
         "method": "PME"},
        # One solver iteration and the final evaluation of a constant-potential cell.
        {"name": "charges-3000", "kind": "charges", "atoms": 3000, "edge": 3.1, "electrode": 400},
        # The same iteration under graph capture rules, smallest grid in use.
        {"name": "noalloc-900", "kind": "noalloc", "atoms": 900, "edge": 2.1, "electrode": 100},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(case, lo, hi):
        m = log_int(lo, hi)
        edge = round((m / rng.uniform(31.0, 34.0)) ** (1.0 / 3.0), 3)
        case.update(molecules=m, edge=edge, cutoff=rng.choice([c for c in (0.9, 1.0, 1.2) if 2.1 * c <= edge]))
        return case

    kind = rng.choice(["step", "step", "step", "batch", "npt", "evaluate", "evaluate", "resident", "charges",
                       "noalloc"])
    if kind == "step":
        c = box({"kind": kind}, 300, 60000)
        c["steps"] = rng.choice([20, 30, 50]) if c["molecules"] < 20000 else 20
        if rng.random() < 0.25:
            c["rigid"] = True
        return c
    if kind == "batch":
        return {"kind": kind, "replicas": rng.randint(4, 40), "lo": 300, "hi": log_int(600, 5000),
                "steps": rng.choice([20, 30])}
    if kind == "npt":
        return {"kind": kind, "replicas": rng.randint(2, 24), "lo": 300, "hi": log_int(600, 3000), "steps": 50}
    if kind == "evaluate":
        c = box({"kind": kind}, 300, 8000)
        c.update(method=rng.choice(["PME", "PME", "LJPME", "CutoffPeriodic"]), double=rng.random() < 0.35,
                 tilt=rng.random() < 0.2)
        return c
    if kind == "resident":
        c = box({"kind": kind}, 300, 40000)
        c["method"] = rng.choice(["PME", "PME", "CutoffPeriodic"])
        return c
    atoms = log_int(200, 12000 if kind == "charges" else 6000)
    return {"kind": kind, "atoms": atoms, "edge": round(rng.uniform(1.9, 6.5), 3), "electrode": max(1, atoms // rng.randint(3, 12))}


# ---------------------------------------------------------------------------
# Inputs


def water_positions(molecules, box, rng, spread):
    """Hydrogen-bonded columns of water on a lattice that fills the box (rows of `box`), in
    alternating directions, displaced and turned by about `spread` (nm, 10 rad/nm)."""
    n = math.ceil(molecules ** (1.0 / 3.0) - 1e-9)
    site = np.sort(rng.choice(n**3, molecules, replace=False))
    i = np.stack(np.unravel_index(site, (n, n, n)), 1)
    o = ((i + 0.5) / n) @ np.asarray(box, float) + rng.normal(scale=spread, size=(molecules, 3))
    s = np.where((i[:, 1] + i[:, 2]) % 2 == 0, 1.0, -1.0)
    t = s * np.where((i[:, 0] + i[:, 1]) % 2 == 0, 1.0, -1.0)
    flat = i[:, 2] % 2 == 0
    w = ommhip.WATER
    c, h = math.cos(w["theta0"]), math.sin(w["theta0"])
    arms = [np.stack([s, 0 * s, 0 * s], 1), np.stack([s * c, np.where(flat, t * h, 0.0), np.where(flat, 0.0, t * h)], 1)]
    turn = rng.normal(scale=10.0 * spread, size=(molecules, 3))
    angle = np.linalg.norm(turn, axis=1, keepdims=True)
    k = turn / angle
    out = [o]
    for d in arms:
        out.append(o + w["r_oh"] * (d * np.cos(angle) + np.cross(k, d) * np.sin(angle)
                                    + k * (k * d).sum(1, keepdims=True) * (1.0 - np.cos(angle))))
    return np.stack(out, 1).reshape(-1, 3)


def velocities(masses, rng):
    # The lattice gives up potential energy as it melts, so the atoms start cold.
    return rng.normal(size=(len(masses), 3)) * np.sqrt(0.00831446261815324 * 100.0 / masses)[:, None]


def box_of(case):
    box = np.diag([case["edge"]] * 3).astype(float)
    if case.get("tilt"):
        box[1, 0], box[2, 0], box[2, 1] = 0.21 * case["edge"], -0.13 * case["edge"], 0.17 * case["edge"]
    return box


@functools.lru_cache(maxsize=None)
def topology(molecules, edge, cutoff, method="PME", rigid=False):
    """The water system of a size (its coordinates are replaced by each preparation's own)."""
    s = ommhip.water_system(molecules, edge, 1, cutoff=cutoff, tolerance=TOLERANCE, method=method)
    if rigid:
        w = ommhip.WATER
        hh = 2.0 * w["r_oh"] * math.sin(0.5 * w["theta0"])
        s.constraints = [c for o in range(0, 3 * molecules, 3)
                         for c in ((o, o + 1, w["r_oh"]), (o, o + 2, w["r_oh"]), (o + 1, o + 2, hh))]
        s.constraint_tolerance = 1e-6
        s.bonds, s.bond_params = np.zeros((0, 2), np.int32), np.zeros((0, 2))
        s.angles, s.angle_params = np.zeros((0, 3), np.int32), np.zeros((0, 2))
    return s


def replica_sizes(case):
    """Log-uniform replica sizes, the largest first (fixed by the case, not by the seed)."""
    rng = np.random.default_rng(4096)
    m = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), size=case["replicas"]))
    return sorted((int(x) for x in np.rint(m)), reverse=True)


def conformations(case, seed):
    """Two conformations with thermal bond lengths, as frames of a trajectory far apart."""
    rng = np.random.default_rng(seed)
    box = box_of(case)
    return [water_positions(case["molecules"], box, rng, 0.012) + rng.normal(scale=0.003, size=(3 * case["molecules"], 3))
            for _ in range(2)]


def cell(case, seed):
    """Charges and positions of a constant-potential cell: an ion mixture and electrode atoms."""
    rng = np.random.default_rng(seed)
    n, edge = case["atoms"], case["edge"]
    pos = rng.uniform(-0.2 * edge, 1.2 * edge, size=(n, 3))
    q = rng.normal(scale=0.4, size=n)
    q[::5] = 0.0
    q[1::5] -= q.sum() / max(1, len(q[1::5]))
    idx = np.sort(rng.choice(n, case["electrode"], replace=False)).astype(np.int32)
    return pos, q, idx, np.diag([edge] * 3).astype(float), *pme_rule(0.9, edge)


def pme_rule(cutoff, edge):
    alpha = math.sqrt(-math.log(2.0 * TOLERANCE)) / cutoff
    n = max(6, math.ceil(2.0 * alpha * edge / (3.0 * TOLERANCE**0.2)))
    return alpha, (n, n, n)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "step":
        s = topology(case["molecules"], case["edge"], case["cutoff"], "PME", case.get("rigid", False))
        s = dataclasses.replace(s, positions=water_positions(case["molecules"], s.box, rng, 0.004))
        ctx = ommhip.Context(s, temperature=300.0, friction=1.0, step_size=0.001, seed=seed % 100003 + 1)
        v = velocities(s.masses, rng)
        if case.get("rigid"):
            v = np.repeat(v[::3], 3, axis=0)  # molecules translate; the constraints hold
        ctx.set_velocities(v)
        return {"kind": kind, "ctx": ctx, "steps": case["steps"]}
    if kind in ("batch", "npt"):
        systems, vels = [], []
        for m in replica_sizes(case):
            s = topology(m, float((m / DENSITY) ** (1.0 / 3.0)), 0.9)
            systems.append(dataclasses.replace(s, positions=water_positions(m, s.box, rng, 0.004)))
            vels.append(velocities(s.masses, rng))
        b = ommhip.Batch(systems, temperature=300.0, friction=1.0, step_size=0.001,
                         seeds=[seed % 100003 + 1 + r for r in range(len(systems))])
        for r, v in enumerate(vels):
            b.set_velocities(r, v)
        if kind == "npt":
            b.set_barostat(1.0, 300.0, 25, seed=seed % 100003 + 7)
        return {"kind": kind, "batch": b, "steps": case["steps"], "report": len(systems) - 1}
    if kind in ("evaluate", "resident"):
        s = topology(case["molecules"], case["edge"], case["cutoff"], case["method"])
        double = case.get("double", False)
        op = ommhip.GpuNonbondedForce(s.nonbonded, ommhip.PRECISION_DOUBLE if double else ommhip.PRECISION_MIXED)
        box = box_of(case)
        op.initialize(box)
        frames = conformations(case, seed)
        state = {"kind": kind, "op": op, "box": box, "double": double, "frames": frames}
        if kind == "resident":
            # Successive steps of an outer integrator: atoms move by about 0.002 nm.
            state["frames"] = [torch.from_numpy(frames[0] + k * rng.normal(scale=0.002, size=frames[0].shape)).cuda()
                               for k in range(2)]
            state["forces"] = [torch.zeros(frames[0].shape, dtype=torch.float64, device="cuda") for _ in range(2)]
        return state
    pos, q, idx, box, alpha, grid = cell(case, seed)
    if kind == "charges":
        return {"kind": kind, "mesh": ommhip.PmeCache(), "args": (pos, q, box, (alpha, grid)), "idx": idx}
    dev = [torch.from_numpy(x).cuda() for x in (pos, q, idx)]
    return {"kind": kind, "dev": dev, "out": torch.zeros(len(idx), dtype=torch.float64, device="cuda"),
            "box": np.ascontiguousarray(box).reshape(9), "alpha": alpha, "grid": (ctypes.c_int32 * 3)(*grid)}


# ---------------------------------------------------------------------------
# One pass


def run(state):
    kind = state["kind"]
    if kind == "step":
        ctx = state["ctx"]
        ctx.step(state["steps"])
        f = ctx.get_state()
        return {"positions": f["positions"].astype(np.float32), "velocities": f["velocities"].astype(np.float32),
                "energy": np.float32(f["potential_energy"])}
    if kind in ("batch", "npt"):
        b = state["batch"]
        b.step(state["steps"])
        e = b.energies()
        f = b.get_state(state["report"])
        return {"energies": e.astype(np.float32), "positions": f["positions"].astype(np.float32),
                "velocities": f["velocities"].astype(np.float32), "box": f["box"].astype(np.float32)}
    if kind == "evaluate":
        out = []
        for p in state["frames"]:
            f, e = state["op"].calc_forces_and_energy(p, state["box"])
            out.append({"forces": f if state["double"] else f.astype(np.float32), "energy": np.float64(e)})
        return out
    if kind == "resident":
        op, stream = state["op"], torch.cuda.current_stream().cuda_stream
        out = []
        for p, f in zip(state["frames"], state["forces"]):
            op.calc_forces_and_energy_device(p.data_ptr(), state["box"], f.data_ptr(), stream=stream, energy=False)
            out.append(f.float())
        return out
    if kind == "charges":
        mesh, args = state["mesh"], state["args"]
        d = np.zeros(len(state["idx"]))
        mesh.charge_derivatives(*args, state["idx"], d)
        f = np.zeros((len(args[1]), 3))
        e = mesh.evaluate_charges(*args, f)
        return {"derivatives": d, "energy": np.float64(e), "forces": f}
    pos, q, idx = state["dev"]
    out = state["out"].zero_()
    lib = ommhip.library()
    st = lib.omm_pme_charge_derivatives_noalloc(
        len(q), ctypes.c_void_p(pos.data_ptr()), ctypes.c_void_p(q.data_ptr()),
        state["box"].ctypes.data_as(ctypes.c_void_p), ctypes.c_double(state["alpha"]), state["grid"],
        ctypes.c_void_p(idx.data_ptr()), len(idx), ctypes.c_void_p(out.data_ptr()),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if st != 0:
        raise ommhip.OmmError(st, lib.omm_last_error().decode())
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without


def work(case):
    kind = case["kind"]

    def system(m, edge, cutoff, mesh=True, energy=False):
        n = 3 * m
        pairs = 0.5 * n * n * (4.0 / 3.0) * math.pi * cutoff**3 / edge**3
        g = pme_rule(cutoff, edge)[1][0] ** 3 if mesh else 0
        # 75 FLOP a pair, spread and gather, five-fold n log n of the two transforms.
        return pairs * 75.0 + mesh * (1730.0 * n + 10.0 * g * math.log2(max(g, 2)))

    if kind == "step":
        n, per = 3 * case["molecules"], system(case["molecules"], case["edge"], case["cutoff"])
        return {"bytes": case["steps"] * 96.0 * n + 96.0 * n, "flops": (case["steps"] + 1) * per}
    if kind in ("batch", "npt"):
        sizes = replica_sizes(case)
        per = sum(system(m, (m / DENSITY) ** (1.0 / 3.0), 0.9) for m in sizes)
        n = 3 * sum(sizes)
        return {"bytes": (case["steps"] + 1) * 96.0 * n, "flops": (case["steps"] + 2) * per}
    if kind in ("evaluate", "resident"):
        n = 3 * case["molecules"]
        per = system(case["molecules"], case["edge"], case["cutoff"], case["method"] != "CutoffPeriodic")
        return {"bytes": 2 * 48.0 * n, "flops": 2 * per}
    g = pme_rule(0.9, case["edge"])[1][0] ** 3
    n, calls = case["atoms"], 2 if kind == "charges" else 1
    return {"bytes": calls * (32.0 * n + 12.0 * case["electrode"]) + (24.0 * n if kind == "charges" else 0.0),
            "flops": calls * (600.0 * n + 10.0 * g * math.log2(g) + 500.0 * case["electrode"])}


# ---------------------------------------------------------------------------
# The same outputs in plain FP64


def min_image(d, box):
    for k in (2, 1, 0):
        s = torch.round(d[..., k] / box[k, k])
        d = d - s[..., None] * box[k]
    return d


def splines(x):
    """Order-5 cardinal B-spline weights and derivatives at fractions x, [n, 5] each."""
    w = [1.0 - x, x]
    for order in range(3, 6):
        if order == 5:
            d = [-w[0]] + [w[k - 1] - w[k] for k in range(1, 4)] + [w[3]]
        div = 1.0 / (order - 1)
        new = [div * (1.0 - x) * w[0]]
        for k in range(1, order - 1):
            new.append(div * ((x + (order - 1 - k)) * w[k - 1] + ((k + 1) - x) * w[k]))
        new.append(div * x * w[order - 2])
        w = new
    return torch.stack(w, 1), torch.stack(d, 1)


def moduli(n, dev):
    m5 = torch.tensor([1.0, 11.0, 11.0, 1.0], dtype=torch.float64, device=dev) / 24.0
    t = 2.0 * math.pi * torch.outer(torch.arange(n, dtype=torch.float64, device=dev),
                                    torch.arange(4, dtype=torch.float64, device=dev)) / n
    v = (torch.cos(t) @ m5) ** 2 + (torch.sin(t) @ m5) ** 2
    return torch.where(v < 1e-7, 0.5 * (torch.roll(v, 1) + torch.roll(v, -1)), v)


def mesh(pos, amp, box, alpha, grid, dispersion=False):
    """Energy, forces and potential at the particles of the smooth-PME mesh."""
    dev = pos.device
    recip = torch.linalg.inv(box)  # columns: reciprocal vectors
    vol = float(torch.det(box))
    f = pos @ recip
    c = (f - torch.floor(f)) * torch.tensor(grid, dtype=torch.float64, device=dev)
    base = torch.floor(c).long()
    wd = [splines(c[:, a] - torch.floor(c[:, a])) for a in range(3)]
    idx = [(base[:, a, None] + torch.arange(5, device=dev)) % grid[a] for a in range(3)]
    flat = (idx[0][:, :, None, None] * grid[1] + idx[1][:, None, :, None]) * grid[2] + idx[2][:, None, None, :]
    q = torch.zeros(grid[0] * grid[1] * grid[2], dtype=torch.float64, device=dev)
    weight = torch.einsum("ni,nj,nk->nijk", wd[0][0], wd[1][0], wd[2][0])
    q.index_add_(0, flat.reshape(-1), (amp[:, None, None, None] * weight).reshape(-1))
    s = torch.fft.fftn(q.reshape(grid))
    m = [torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=dev) for n in grid]
    k = (m[0][:, None, None, None] * recip[:, 0] + m[1][None, :, None, None] * recip[:, 1]
         + m[2][None, None, :, None] * recip[:, 2])
    k2 = (k * k).sum(-1)
    b = [moduli(n, dev) for n in grid]
    bk = b[0][:, None, None] * b[1][None, :, None] * b[2][None, None, :]
    if dispersion:
        kk = torch.sqrt(k2)
        x = math.pi * kk / alpha
        infl = -(math.pi**1.5) / (3.0 * vol * bk) * (
            2.0 * math.pi**3.5 * torch.erfc(x) * kk**3
            + torch.exp(-x * x) * (alpha**3 - 2.0 * alpha * math.pi**2 * k2))
    else:
        k2[0, 0, 0] = 1.0
        infl = ONE_4PI_EPS0 / (math.pi * vol) * torch.exp(-((math.pi / alpha) ** 2) * k2) / (k2 * bk)
        infl[0, 0, 0] = 0.0
    energy = 0.5 * float((infl * (s.real**2 + s.imag**2)).sum())
    phi = torch.fft.ifftn(infl * s).real.reshape(-1) * q.numel()
    p = phi[flat]
    grads = []
    for a in range(3):
        ws = [wd[x][1 if x == a else 0] for x in range(3)]
        grads.append(torch.einsum("nijk,ni,nj,nk->n", p, *ws) * grid[a])
    force = -amp[:, None] * (torch.stack(grads, 1) @ recip.T)
    return energy, force, (p * weight).sum((1, 2, 3))


def water_energy_forces(case, pos):
    """Nonbonded energy and forces of a water box in FP64."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    w, method, rc, n = ommhip.WATER, case["method"], case["cutoff"], 3 * case["molecules"]
    box = torch.from_numpy(box_of(case)).to(dev)
    x = torch.from_numpy(pos).to(dev)
    q = torch.tensor([w["q_o"], w["q_h"], w["q_h"]], dtype=torch.float64, device=dev).repeat(case["molecules"])
    mol = torch.arange(n, device=dev) // 3
    oxygen = torch.arange(n, device=dev) % 3 == 0
    vol = float(torch.det(box))
    sig, eps = w["sigma_o"], w["eps_o"]
    alpha, grid = pme_rule(rc, case["edge"])
    krf, crf = (78.3 - 1.0) / (2.0 * 78.3 + 1.0) / rc**3, 3.0 * 78.3 / (2.0 * 78.3 + 1.0) / rc
    s6c, c6 = (sig / rc) ** 6, 4.0 * eps * sig**6

    def complement(r2):  # C6 / r^6 (1 - e^-x (1 + x + x^2 / 2)) and dE/dr^2
        y = alpha * alpha * r2
        e = torch.exp(-y)
        v = c6 / r2**3 * (1.0 - e * (1.0 + y + 0.5 * y * y))
        return v, -3.0 * v / r2 + c6 / r2**3 * e * 0.5 * y * y * alpha * alpha

    energy, force = 0.0, torch.zeros_like(x)
    rows = max(1, 24_000_000 // n)
    for a in range(0, n, rows):
        i = torch.arange(a, min(n, a + rows), device=dev)
        d = min_image(x[None, :, :] - x[i][:, None, :], box)
        r2 = (d * d).sum(-1)
        near = torch.nonzero((r2 < rc * rc) & (mol[i][:, None] != mol[None, :]))
        ii, jj, d, r2 = i[near[:, 0]], near[:, 1], d[near[:, 0], near[:, 1]], r2[near[:, 0], near[:, 1]]
        r, qq = torch.sqrt(r2), ONE_4PI_EPS0 * q[ii] * q[jj]
        if method == "CutoffPeriodic":
            e = qq * (1.0 / r + krf * r2 - crf)
            de = qq * (2.0 * krf * r - 1.0 / r2)
        else:
            ec = qq * torch.erfc(alpha * r) / r
            e = ec.clone()
            de = -(ec + qq * 2.0 * alpha / math.sqrt(math.pi) * torch.exp(-(alpha * alpha) * r2)) / r
        oo = oxygen[ii] & oxygen[jj]
        s6 = (sig * sig / r2) ** 3
        lj = 4.0 * eps * (s6 * s6 - s6)
        dlj = 4.0 * eps * (6.0 * s6 - 12.0 * s6 * s6) / r
        if method == "LJPME":
            v, dv = complement(r2)
            vc, _ = complement(torch.tensor(rc * rc, dtype=torch.float64, device=dev))
            lj = lj + v - (4.0 * eps * (s6c * s6c - s6c) + vc)
            dlj = dlj + dv * 2.0 * r
        e = e + torch.where(oo, lj, torch.zeros_like(lj))
        de = de + torch.where(oo, dlj, torch.zeros_like(dlj))
        energy += 0.5 * float(e.sum())
        force.index_add_(0, ii, (de / r)[:, None] * d)
    if method != "CutoffPeriodic":
        em, fm, _ = mesh(x, q, box, alpha, grid)
        energy += em - ONE_4PI_EPS0 * alpha / math.sqrt(math.pi) * float((q * q).sum())
        energy -= ONE_4PI_EPS0 * math.pi * float(q.sum()) ** 2 / (2.0 * alpha * alpha * vol)
        force += fm
        for a, b in ((0, 1), (0, 2), (1, 2)):  # excluded pairs of each molecule
            d = x[b::3] - x[a::3]
            r = d.norm(dim=1)
            qq = ONE_4PI_EPS0 * q[a] * q[b]
            erf = torch.erf(alpha * r) / r
            energy -= float((qq * erf).sum())
            g = -qq * (2.0 * alpha / math.sqrt(math.pi) * torch.exp(-(alpha * r) ** 2) - erf) / r
            force[a::3] += (g / r)[:, None] * d
            force[b::3] -= (g / r)[:, None] * d
    if method == "LJPME":
        half = tuple(max(6, math.ceil(alpha * case["edge"] / (3.0 * TOLERANCE**0.2))) for _ in range(3))
        amp = torch.where(oxygen, 2.0 * math.sqrt(eps) * sig**3, 0.0).double()
        ed, fd, _ = mesh(x, amp, box, alpha, half, dispersion=True)
        energy += ed + alpha**6 / 3.0 * case["molecules"] * eps * sig**6
        force += fd
    else:
        m = case["molecules"]
        tail = eps * (m * m + m) * (sig**12 * rc**-9 / 9.0 - sig**6 * rc**-3 / 3.0)
        energy += 8.0 * math.pi * n / (n + 1.0) * tail / vol
    return energy, force


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "batch", "npt"):
        return None  # the noise is the library's own random stream
    if kind == "evaluate":
        out = []
        for p in conformations(case, seed):
            e, f = water_energy_forces(case, p)
            out.append({"forces": f, "energy": torch.tensor(e, dtype=torch.float64)})
        return out
    if kind == "resident":
        rng = np.random.default_rng(seed)
        p = conformations(case, seed)[0]
        return [water_energy_forces(case, p + k * rng.normal(scale=0.002, size=p.shape))[1] for k in range(2)]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    pos, q, idx, box, alpha, grid = cell(case, seed)
    e, f, p = mesh(torch.from_numpy(pos).to(dev), torch.from_numpy(q).to(dev), torch.from_numpy(box).to(dev), alpha, grid)
    d = p[torch.from_numpy(idx).long().to(dev)]
    if kind == "noalloc":
        return d
    return {"derivatives": d, "energy": torch.tensor(e, dtype=torch.float64), "forces": f}
