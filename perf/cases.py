"""The work that is timed: whole calls through the Python interface.

Five kinds of case, each a program that a user of the library writes:

* ``step``    a particle simulation in given fields: some full particle steps
              (push, migration, J and mass-matrix deposit) in one call, then
              its output: J, or J and M, or (large runs) the particle number
              of every cell with the particle energy and CFL.
* ``move``    test particles: steps of the mover alone, then the population.
* ``cycle``   one cycle of the self-consistent ECSIM simulation on a
              single-level mesh: mover, deposit and field step with E and B
              in host arrays.
* ``scan``    a cutoff-rigidity map: every (location, direction) pair's
              rigidity grid, traced whole, downward or inside a bracket.
* ``train``, ``predict``  the cutoff surrogate network.

Particles cross ``cfl`` of the smallest cell per step at the electrons'
thermal speed, the regime an implicit particle-in-cell run is set up for.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from amps_amd import _lib as L
from amps_amd import cutoff as CU
from amps_amd import mesh as M
from amps_amd import surrogate as SG
from amps_amd.pic import PicState, Species

VTH = (0.05, 0.005)      # electrons, ions (mass ratio 100)
DRIFT = (0.01, 0.0, 0.0)
CHARGE, MASS = (-1.0, 1.0), (0.01, 1.0)


def listed():
    return [
        # a small run on a coarse box, where launches and latency count; J and M to the host
        {"name": "step small", "kind": "step", "mesh": "uniform1", "per_species": 8192, "precision": "fp64",
         "steps": 10, "cfl": 0.1, "copy": "JM"},
        # the two-level mesh with 16 particles per cell and species
        {"name": "step two-level", "kind": "step", "mesh": "octant", "per_species": 16 * 120 * 512,
         "precision": "fp64", "steps": 4, "cfl": 0.2, "copy": "J"},
        # the particle step at scale: 2^27 particles on the three-level mesh
        {"name": "step 2^27", "kind": "step", "mesh": "three", "per_species": 1 << 26, "precision": "fp64",
         "steps": 8, "cfl": 0.1, "copy": "diag"},
        # the FP32 mode on a single-level box, a particle count that divides nothing
        {"name": "step fp32", "kind": "step", "mesh": "uniform3", "per_species": 7654321, "precision": "fp32",
         "steps": 4, "cfl": 0.1, "copy": "diag"},
        # 2^20 test protons, Boris mover: steps of MoveParticles, then the particles
        {"name": "move 2^20 boris", "kind": "move", "mesh": "uniform2", "n": 1 << 20, "steps": 20, "cfl": 0.05},
        # the self-consistent cycle on a small and on a large single-level box
        {"name": "cycle 33^3", "kind": "cycle", "level": 2, "per_species": 8 * 64 * 512, "cfl": 0.1, "tol": 1e-8},
        {"name": "cycle 129^3", "kind": "cycle", "level": 4, "per_species": 16 * 4096 * 512, "cfl": 0.1, "tol": 1e-8},
        # the cutoff map: 64 x 32 points, 8 directions, 48 rigidities, every bin traced
        {"name": "map fp64", "kind": "scan", "mode": "full", "nlon": 64, "nlat": 32, "ndir": 8, "nr": 48,
         "precision": "fp64"},
        # a time series of maps with a bracket from the dipole formula, the rest rescanned in the same launch
        {"name": "map bracketed", "kind": "scan", "mode": "bracketed", "nlon": 64, "nlat": 32, "ndir": 16, "nr": 48,
         "precision": "fp64"},
        # the surrogate's training set: downward scans of random pairs in the FP32 mode
        {"name": "map upper fp32", "kind": "scan", "mode": "upper", "nlon": 331, "nlat": 199, "ndir": 2, "nr": 48,
         "precision": "fp32"},
        # the surrogate: Adam steps of 4096 samples, and inference for a fine map
        {"name": "train", "kind": "train", "n": 1 << 17, "batch": 4096, "steps": 64},
        {"name": "predict", "kind": "predict", "n": 1 << 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "move", "cycle", "cycle", "scan", "scan", "train", "predict"])
    cfl = rng.choice([0.02, 0.05, 0.1, 0.2, 0.3])
    if kind == "step":
        mesh = rng.choice(["uniform1", "uniform2", "octant", "uniform3"])
        ncell = 512 * {"uniform1": 8, "uniform2": 64, "octant": 120, "uniform3": 512}[mesh]
        return {"kind": kind, "mesh": mesh, "per_species": _log(rng, ncell // 4, 48 * ncell),
                "precision": rng.choice(["fp64", "fp64", "fp32"]), "steps": rng.randint(1, 12), "cfl": cfl,
                "copy": {"uniform1": "JM", "uniform3": "diag"}.get(mesh, "J")}
    if kind == "move":
        return {"kind": kind, "mesh": rng.choice(["uniform1", "uniform2", "octant"]), "n": _log(rng, 1000, 1 << 20),
                "steps": rng.randint(2, 40), "cfl": cfl}
    if kind == "cycle":
        level = rng.choice([1, 2, 2, 3])
        return {"kind": kind, "level": level, "per_species": _log(rng, 2 * 512 * 8 ** level, 24 * 512 * 8 ** level),
                "cfl": cfl, "tol": rng.choice([1e-8, 1e-10])}
    if kind == "scan":
        return {"kind": kind, "mode": rng.choice(["full", "bracketed", "upper"]), "nlon": _log(rng, 3, 72),
                "nlat": _log(rng, 2, 36), "ndir": rng.randint(1, 5), "nr": rng.choice([24, 37, 48]),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "train":
        batch = rng.choice([1024, 2048, 4096, 8192])
        return {"kind": kind, "n": batch * rng.randint(3, 16), "batch": batch, "steps": rng.randint(16, 64)}
    return {"kind": kind, "n": _log(rng, 60, 1 << 20)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _mesh(name):
    """Mesh and corner fields: a weak dipole and uniform Bz, so that the
    electrons' gyration over a step stays below a radian away from the origin."""
    if name == "octant":
        m = M.central_octant_mesh()
    elif name == "three":
        m = M.three_level_mesh()
    else:
        m = M.uniform_mesh(int(name[len("uniform"):]))
    E, B = M.corner_fields(m, E0=(1e-3, 0.0, 0.0), moment=1.5e-4, bz0=0.05)
    return m, E, B


def _dt(mesh, cfl):
    return cfl * float(mesh.cell_size().min()) / VTH[0]


def _species(mesh, case):
    """Electrons and ions; the particle weight puts omega_pe dt near one."""
    dt = _dt(mesh, case["cfl"])
    vol = float(np.prod(mesh.cell_size().max(axis=0)))
    ppc = max(1.0, case["per_species"] / mesh.ncells)
    w = vol * MASS[0] / (4.0 * math.pi * ppc * dt * dt)
    return Species(list(CHARGE), list(MASS), [dt, dt], w), dt


def _scan_inputs(case, seed):
    """Points, arrival directions (seeded) and, for the bracketed mode, the
    bracket of four bins around the dipole (Stoermer) cutoff."""
    pts, lat, lon = CU.config2_points(case["nlon"], case["nlat"])
    zen, az = CU.config2_directions(case["ndir"] + 1, seed=1000 + seed)
    zen, az = zen[1:], az[1:]  # the first is vertical for every seed
    dirs = CU.arrival_dirs(pts, zen, az).reshape(-1, 3)
    x0 = np.repeat(pts, len(zen), axis=0)
    grid = CU.build_search_grid(0.1, 20.0, case["nr"])
    lo = hi = None
    if case["mode"] == "bracketed":
        P = CU.config2_params()
        m = np.array([P.m_hat[0], P.m_hat[1], P.m_hat[2]])
        r = np.linalg.norm(x0, axis=1) / CU.RE_DIPOLE
        u = x0 / np.linalg.norm(x0, axis=1)[:, None]
        cosl2 = 1.0 - (u @ m) ** 2
        east = np.cross(m, u)
        east /= np.maximum(np.linalg.norm(east, axis=1), 1e-12)[:, None]
        cosg = np.einsum("ij,ij->i", -dirs, east)
        rc = 59.6 / r ** 2 * cosl2 ** 2 / (1.0 + np.sqrt(np.maximum(1.0 + cosg * cosl2 ** 1.5, 0.0))) ** 2
        b = np.searchsorted(np.log(grid), np.log(np.maximum(rc, 1e-3)))
        lo, hi = SG.bracket_bins(np.clip(b, 0, len(grid) - 1), len(grid), half=4)
    return x0, dirs, grid, lo, hi


def _surrogate_data(n, seed):
    """Features of random pairs and the log10 dipole cutoff as target."""
    rng = np.random.default_rng(100 + seed)
    lat = np.degrees(np.arcsin(rng.uniform(-1, 1, n)))
    lon, az = rng.uniform(0, 360, n), rng.uniform(0, 360, n)
    zen = np.degrees(np.arccos(rng.uniform(0.5, 1.0, n)))
    c4 = np.cos(np.radians(lat)) ** 4
    t = np.log10(np.maximum(14.9 * c4 * (1.0 + 0.2 * np.sin(np.radians(zen)) * np.sin(np.radians(az))), 0.1))
    return SG.features(lat, lon, zen, az), t.astype(np.float32)


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case}
    if k in ("step", "move", "cycle"):
        name = "uniform%d" % case["level"] if k == "cycle" else case["mesh"]
        mesh, E, B = _mesh(name)
        if k == "move":
            dt = _dt(mesh, case["cfl"])
            st = PicState(mesh, E, B, Species([1.0], [1.0], [dt]))
            st.set_particles(M.uniform_particles(mesh, case["n"], VTH[0], seed_x=2 * seed + 1, seed_v=2 * seed + 2))
        else:
            sp, dt = _species(mesh, case)
            st = PicState(mesh, E, B, sp)
            st.generate_particles(case["per_species"], VTH, drift=DRIFT, seed=seed + 11,
                                  precision=L.FP32 if case.get("precision") == "fp32" else L.FP64)
        s.update(st=st, dt=dt)
        if k == "cycle":
            rng = np.random.default_rng(seed)
            dx = float(mesh.cell_size()[0][0])
            s["params"] = st.ecsim_params(dt, theta=0.5, cDt=dt)
            s["E"] = 1e-3 * rng.normal(size=(st.nnodes, 3))
            s["B"] = (M.interior_center_fields(mesh, lambda x: M.dipole_field(x, moment=1.5e-4, bz0=0.05))
                      .reshape(-1, 3) + 1e-3 * rng.normal(size=(mesh.ncells, 3)))
            s["dx"] = dx
    elif k == "scan":
        s["ctx"] = L.Context(0)
        s["params"] = CU.config2_params()
        s["x0"], s["dirs"], s["grid"], s["lo"], s["hi"] = _scan_inputs(case, seed)
    elif k == "train":
        s["ctx"] = L.Context(0)
        s["sur"] = SG.Surrogate(s["ctx"], seed=seed)
        s["sur"].set_data(*_surrogate_data(case["n"], seed))
    else:
        s["ctx"] = L.Context(0)
        s["sur"] = SG.Surrogate(s["ctx"], seed=seed)
        s["X"] = _surrogate_data(case["n"], seed)[0]
    return s


def _counts(st):
    """The particle number of every cell (ParticleNumberTable of a restart file)."""
    counts, n = np.zeros((st.mesh.nblocks, 512), np.int32), ctypes.c_int64()
    L.check(st.lib.amps_gpu_get_particles_restart(st.ctx.h, ctypes.byref(L.aos_layout_aligned()),
                                                  L._ptr(counts, ctypes.c_int32), None, 0, ctypes.byref(n)), "counts")
    return counts


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "step":
        s["st"].run_steps(case["steps"], s["dt"])
        if case["copy"] == "diag":
            energy, cfl = s["st"].ParticleEnergyCfl(s["dt"])
            return {"energy": np.float64(energy), "cfl": cfl, "counts": _counts(s["st"])}
        J, Mm = s["st"].UpdateJMassMatrix(s["dt"], copy_out=True if case["copy"] == "JM" else "J")
        return {"J": J} if Mm is None else {"J": J, "M": Mm}
    if k == "move":
        for _ in range(case["steps"]):
            s["st"].MoveParticles(mover=L.MOVER_BORIS, bc_mode=L.BC_REFLECT, r_sphere=0.0)
        p, code = s["st"].get_particles()
        return {"x": p.x, "v": p.v, "blk": p.blk, "cell": p.cell, "id": p.id, "code": code}
    if k == "cycle":
        s["st"].MoveParticles()
        s["st"].UpdateJMassMatrix(s["dt"], copy_out=False)
        E, Eth, B, _, _ = s["st"].EcsimTimeStep(s["params"], s["E"], s["B"], tol=case["tol"], max_iter=400, restart=40)
        return {"E": E, "E_theta": Eth, "B": B}
    if k == "scan":
        mode = {"full": CU.SCAN_FULL, "upper": CU.SCAN_UPPER, "bracketed": CU.SCAN_BRACKETED}[case["mode"]]
        states, bins, _ = CU.cutoff_scan(s["ctx"], s["params"], s["x0"], s["dirs"], s["grid"], mode=mode, lo=s["lo"],
                                         hi=s["hi"], precision=L.FP32 if case["precision"] == "fp32" else L.FP64)
        return {"states": states, "bins": bins}
    if k == "train":
        s["sur"].train(case["steps"], batch=case["batch"], lr=1e-3)
        theta, n = s["sur"].params()
        return {"theta": theta, "adam_steps": n}
    return s["sur"].predict(s["X"])


def work(case):
    """Bytes: particle state read and written per step, node rows written
    once per deposit, host arrays once.  Flops: about 300 per push and 780 per
    deposited particle; a Boris trace step about 120 (a full map takes some
    13,000 steps per trajectory, a downward scan 2,000 per traced bin of
    about half the grid); the network's multiply-adds."""
    k = case["kind"]
    if k in ("step", "move", "cycle"):
        mesh = _mesh("uniform%d" % case["level"] if k == "cycle" else case["mesh"])[0]
        nodes = mesh.ncells + 3 * mesh.ncells ** (2 / 3)
        fields = mesh.nblocks * 729 * 6 * 8
    if k == "step":
        n = 2 * case["per_species"]
        pb = 102 if case["precision"] == "fp64" else 78
        per = n * (pb + 48) + fields + nodes * 1968
        out = {"JM": nodes * 1968, "J": nodes * 24, "diag": mesh.ncells * 4}[case["copy"]]
        return {"bytes": case["steps"] * per + out, "flops": case["steps"] * n * 1080.0}
    if k == "move":
        return {"bytes": case["steps"] * (case["n"] * 102.0 + fields) + case["n"] * 68.0,
                "flops": case["steps"] * case["n"] * 300.0}
    if k == "cycle":
        n = 2 * case["per_species"]
        its = (5 + 150 * case["cfl"]) * (1.0 if case["tol"] >= 1e-8 else 1.25)  # Arnoldi steps taken, about
        return {"bytes": n * 150.0 + fields + nodes * 1968 + its * nodes * 2127 + nodes * 72 + mesh.ncells * 48.0,
                "flops": n * 1080.0 + its * nodes * 500.0}
    if k == "scan":
        traj = case["nlon"] * case["nlat"] * case["ndir"]
        steps = {"full": 13000.0 * case["nr"], "bracketed": 60000.0, "upper": 22000.0}[case["mode"]]
        return {"bytes": traj * (48.0 + case["nr"]), "flops": traj * steps * 120.0}
    fwd = 2.0 * (6 * 128 + 128 * 128 + 128)
    if k == "train":
        return {"bytes": case["steps"] * case["batch"] * 28.0 + 17537 * 12.0,
                "flops": 3 * fwd * case["batch"] * case["steps"]}
    return {"bytes": case["n"] * 28.0, "flops": fwd * case["n"]}


def tolerance(case):
    k = case["kind"]
    if k == "step":
        # four times what up to 12 steps show against 64 bits; the FP32 mode carries its increments' rounding
        return {"rel": 1e-12, "max": 5e-11} if case["precision"] == "fp64" else {"rel": 8e-5, "max": 1e-2}
    if k == "move":
        return {"rel": 1e-14, "max": 1e-12}
    if k == "cycle":
        # the solver stops at a relative residual of tol; E is then up to 11 tol off, single nodes up to 300 tol
        return {"rel": 40 * case["tol"], "max": 1200 * case["tol"]}
    if k == "scan":
        # states and bins are whole numbers of trajectories that a change of rounding alters
        return "exact"
    # BF16 operands
    return {"rel": 1.6e-3, "max": 0.05} if k == "train" else {"rel": 1.8e-2, "max": 0.1}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
DEV = "cuda"


def _geometry(mesh):
    lv = torch.as_tensor(mesh.level.astype(np.int64), device=DEV)
    return (torch.as_tensor(mesh.blk_xmin, device=DEV), torch.as_tensor(mesh.blk_xmax, device=DEV), lv,
            torch.as_tensor(mesh.leaf.astype(np.int64), device=DEV))


def _stencil(geo, x, blk):
    """Lower corner index [n, 3] and offsets f [n, 3] of points x [n, 3] in their blocks."""
    lo, hi = geo[0][blk], geo[1][blk]
    dx = (hi - lo) / 8
    t = (x - lo) / dx
    i = t.floor().clamp(0, 7)
    return i.long(), t - i


CORNERS = [(a, b, c) for c in (0, 1) for b in (0, 1) for a in (0, 1)]


def _weights(f):
    return [(f[:, 0] if a else 1 - f[:, 0]) * (f[:, 1] if b else 1 - f[:, 1]) * (f[:, 2] if c else 1 - f[:, 2])
            for a, b, c in CORNERS]


def _at_corners(F, i, f, blk):
    out = 0.0
    for (a, b, c), w in zip(CORNERS, _weights(f)):
        idx = blk * 729 + (i[:, 0] + a) + 9 * ((i[:, 1] + b) + 9 * (i[:, 2] + c))
        out = out + w[:, None] * F[idx]
    return out


def _rotation(B, g):
    """alpha of the Lapenta mover for g = q dt / 2m, [n, 3, 3]."""
    b = g[:, None] * B
    c0 = 1.0 / (1.0 + (b * b).sum(1))
    a = b[:, :, None] * b[:, None, :]
    eye = torch.eye(3, device=DEV, dtype=torch.float64)
    z = torch.zeros_like(b[:, 0])
    eps = torch.stack([z, b[:, 2], -b[:, 1], -b[:, 2], z, b[:, 0], b[:, 1], -b[:, 0], z], 1).reshape(-1, 3, 3)
    return c0[:, None, None] * (eye + eps + a)


def _push(mesh, geo, E, B, x, v, blk, qm, dt, boris=False):
    """One step with reflection at the box [-1, 1]^3; returns x, v, blk and whether it was reflected."""
    i, f = _stencil(geo, x, blk)
    Ep, Bp = _at_corners(E, i, f, blk), _at_corners(B, i, f, blk)
    g = 0.5 * qm * dt
    if boris:
        u = v + g[:, None] * Ep
        h = g[:, None] * Bp
        h2, uh = (h * h).sum(1, keepdim=True), (u * h).sum(1, keepdim=True)
        v1 = ((1 - h2) * u + 2 * (torch.linalg.cross(u, h) + uh * h)) / (1 + h2) + g[:, None] * Ep
    else:
        al = _rotation(Bp, g)
        v1 = 2.0 * torch.einsum("nij,nj->ni", al, v + g[:, None] * Ep) - v
    x1 = x + dt * v1
    out = ((x1 < -1) | (x1 >= 1)).any(1)
    if bool(out.any()):
        eps = 0.0001 * 2.0 / 8 / (1 << mesh.lmax)
        xo, vo, v1o = x[out], v[out], v1[out]
        vm = 0.5 * (vo + v1o)
        t = torch.where(vm > 0, (1 - xo) / vm, torch.where(vm < 0, (-1 - xo) / vm, torch.inf))
        tm, ax = t.min(1)
        n = torch.zeros_like(xo).scatter_(1, ax[:, None], vm.gather(1, ax[:, None]).sign())
        xr = xo + tm[:, None] * vm - eps * n
        vr = vo + (tm / dt).clamp(max=1)[:, None] * (v1o - vo)
        vr = vr - 2 * (vr * n).sum(1, keepdim=True) * n
        x1[out], v1[out] = xr, vr
    nf = 1 << mesh.lf
    c = ((x1 + 1) / 2 * nf).floor().long().clamp(0, nf - 1)
    return x1, v1, geo[3][c[:, 2], c[:, 1], c[:, 0]], out


def _start(st):
    p, _ = st.get_particles()
    t = lambda a: torch.as_tensor(a, device=DEV)  # noqa: E731
    return (t(p.x).T.contiguous(), t(p.v).T.contiguous(), t(p.spec.astype(np.int64)), t(p.blk.astype(np.int64)),
            t(p.cell.astype(np.int64)), t(p.id))


def _deposit(st, mesh, geo, B, x, v, spec, blk, dt, with_m):
    """J [nodes, 3] and M [nodes, 243] of the particles."""
    noc, _ = st.node_map()
    noc = torch.as_tensor(noc.astype(np.int64), device=DEV)
    w = torch.tensor(st.species.weight, device=DEV)[spec]
    q = torch.tensor(CHARGE, dtype=torch.float64, device=DEV)[spec] * w
    g = 0.5 * dt * q / (torch.tensor(MASS, dtype=torch.float64, device=DEV)[spec] * w)
    vol = ((geo[1] - geo[0]) / 8).prod(1)[blk]
    J = torch.zeros(st.nnodes, 3, dtype=torch.float64, device=DEV)
    Mm = torch.zeros(st.nnodes, 27, 9, dtype=torch.float64, device=DEV) if with_m else None
    step = 1 << 21
    for a in range(0, len(x), step):
        s = slice(a, a + step)
        i, f = _stencil(geo, x[s], blk[s])
        al = _rotation(_at_corners(B, i, f, blk[s]), g[s])
        qv = (q[s] / vol[s])[:, None] * torch.einsum("nij,nj->ni", al, v[s])
        W = _weights(f)
        nd = [noc[blk[s] * 729 + (i[:, 0] + p) + 9 * ((i[:, 1] + r) + 9 * (i[:, 2] + t))] for p, r, t in CORNERS]
        for c in range(8):
            J.index_add_(0, nd[c], W[c][:, None] * qv)
        if not with_m:
            continue
        ma = (q[s] * g[s] / vol[s])[:, None] * al.reshape(-1, 9)
        flat = Mm.reshape(-1, 9)
        for c, (p, r, t) in enumerate(CORNERS):
            for d, (p2, r2, t2) in enumerate(CORNERS):
                slot = [0, 2, 1][p2 - p] + 3 * [0, 2, 1][r2 - r] + 9 * [0, 2, 1][t2 - t]
                flat.index_add_(0, nd[c] * 27 + slot, (W[c] * W[d])[:, None] * ma)
    return J, None if Mm is None else Mm.reshape(-1, 243)


def _diag(mesh, geo, species, x, v, spec, blk, dt):
    """Particle energy, the largest mean CFL of a cell per species, the cells' particle numbers."""
    w = torch.tensor(species.weight * species.mass, device=DEV)[spec]
    i, _ = _stencil(geo, x, blk)
    cell = blk * 512 + 64 * i[:, 0] + 8 * i[:, 1] + i[:, 2]
    counts = torch.bincount(cell, minlength=mesh.ncells)
    speed = (v * v).sum(1).sqrt()
    diag = ((geo[1] - geo[0]) / 8).norm(dim=1)
    cfl = []
    for s in range(len(CHARGE)):
        at = spec == s
        num = torch.zeros(mesh.ncells, dtype=torch.float64, device=DEV).index_add_(0, cell[at], speed[at] * dt)
        den = torch.bincount(cell[at], minlength=mesh.ncells)
        cfl.append(float((num / den.clamp(min=1) / diag.repeat_interleave(512)).max()))
    return {"energy": np.float64((0.5 * w * speed ** 2).sum().item()), "cfl": np.array(cfl),
            "counts": counts.int().reshape(-1, 512).cpu()}


def _conv(u, axis, w):
    """Three-point weights w = (minus, centre, plus) along an axis of u, zero outside."""
    p = torch.zeros_like(u)
    n = u.shape[axis]
    p.narrow(axis, 1, n - 1).add_(w[0] * u.narrow(axis, 0, n - 1))
    p.add_(w[1] * u)
    p.narrow(axis, 0, n - 1).add_(w[2] * u.narrow(axis, 1, n - 1))
    return p


def _curlcurl(u, c):
    """(grad-div minus Laplacian) of a node field [z, y, x, 3], c = c dt theta / dx per axis."""
    S, D, T = (0.25, 0.5, 0.25), (-0.5, 0.0, 0.5), (1.0, -2.0, 1.0)
    ax = [2, 1, 0]

    def op(f, kinds):
        for d in range(3):
            f = _conv(f, ax[d], kinds[d])
        return f

    out = torch.zeros_like(u)
    for i in range(3):
        for j in range(3):
            second = [T if d == j else S for d in range(3)]
            out[..., i] -= c[j] * c[j] * op(u[..., i], second)
            mixed = [S, S, S]
            if i == j:
                mixed[i] = T
            else:
                mixed[i] = mixed[j] = D
            out[..., i] += c[i] * c[j] * op(u[..., j], mixed)
    return out


def _mass(Mm, u):
    """The mass-matrix product over the 27 neighbours, u [z, y, x, 3]."""
    n = u.shape[0]
    out = torch.zeros_like(u)
    off = [0, -1, 1]
    pad = torch.nn.functional.pad(u, (0, 0, 1, 1, 1, 1, 1, 1))
    M5 = Mm.reshape(n, n, n, 27, 3, 3)
    for s in range(27):
        dx, dy, dz = off[s % 3], off[(s // 3) % 3], off[s // 9]
        nb = pad[1 + dz:1 + dz + n, 1 + dy:1 + dy + n, 1 + dx:1 + dx + n]
        out += torch.einsum("zyxij,zyxj->zyxi", M5[..., s, :, :], nb)
    return out


def _field_step(s, J, Mm):
    st, p, mesh = s["st"], s["params"], s["st"].mesh
    n = round(st.nnodes ** (1 / 3))
    nb = 1 << s["case"]["level"]
    c = [p.cDt * p.theta / s["dx"]] * 3
    E0 = torch.as_tensor(s["E"], device=DEV).reshape(n, n, n, 3)
    fp = 4 * math.pi * p.dt * p.theta
    # cell-centred B on the cell lattice [z, y, x, 3]
    k = torch.as_tensor(mesh.ijk, device=DEV)
    blk_of = torch.empty(nb, nb, nb, dtype=torch.long, device=DEV)
    blk_of[k[:, 2], k[:, 1], k[:, 0]] = torch.arange(mesh.nblocks, device=DEV)
    g = torch.arange(8 * nb, device=DEV)
    Z, Y, X = torch.meshgrid(g, g, g, indexing="ij")
    cid = blk_of[Z // 8, Y // 8, X // 8] * 512 + X % 8 + 8 * (Y % 8) + 64 * (Z % 8)
    Bc = torch.as_tensor(s["B"], device=DEV)[cid.reshape(-1)].reshape(*cid.shape, 3)

    def face(u, d):  # difference along axis d, averages along the others, cells to interior nodes or nodes to cells
        for a, axis in enumerate((2, 1, 0)):
            m = u.shape[axis] - 1
            lo, hi = u.narrow(axis, 0, m), u.narrow(axis, 1, m)
            u = hi - lo if a == d else 0.5 * (hi + lo)
        return u

    def curl(u):
        return torch.stack([face(u[..., 2], 1) - face(u[..., 1], 2), face(u[..., 0], 2) - face(u[..., 2], 0),
                            face(u[..., 1], 0) - face(u[..., 0], 1)], -1)

    inner = torch.zeros(n, n, n, 1, dtype=torch.float64, device=DEV)
    inner[1:-1, 1:-1, 1:-1] = 1.0
    rhs = -_curlcurl(E0, c) - fp * _mass(Mm, E0) - fp * J.reshape(n, n, n, 3)
    rhs[1:-1, 1:-1, 1:-1] += c[0] * curl(Bc)
    rhs = rhs * inner

    def A(u):
        ui = u * inner
        return (ui + _curlcurl(ui, c) + fp * _mass(Mm, ui)) * inner

    # GMRES(60) with two passes of Gram-Schmidt, to 1e-13
    x = torch.zeros_like(rhs)
    bn = rhs.norm()
    for _ in range(8):
        r = rhs - A(x)
        beta = r.norm()
        if beta <= 1e-13 * bn:
            break
        V, H = [(r / beta).reshape(-1)], torch.zeros(61, 60, dtype=torch.float64)
        for j in range(60):
            w = A(V[-1].reshape(x.shape)).reshape(-1)
            for _ in range(2):
                for q, vq in enumerate(V):
                    h = torch.dot(w, vq)
                    w = w - h * vq
                    H[q, j] += float(h)
            H[j + 1, j] = float(w.norm())
            V.append(w / w.norm())
        e = torch.zeros(61, 1, dtype=torch.float64)
        e[0] = float(beta)
        y = torch.linalg.lstsq(H, e).solution[:, 0]
        for q in range(60):
            x = x + float(y[q]) * V[q].reshape(x.shape)
    Eth = x + E0
    E1 = (Eth - (1 - p.theta) * E0) / p.theta
    B1 = Bc - p.cDt / s["dx"] * curl(Eth)
    Bout = torch.empty(mesh.ncells, 3, dtype=torch.float64, device=DEV)
    Bout[cid.reshape(-1)] = B1.reshape(-1, 3)
    return {"E": E1.reshape(-1, 3).cpu(), "E_theta": Eth.reshape(-1, 3).cpu(), "B": Bout.cpu()}


def exact(case, seed):
    k = case["kind"]
    if k == "scan" or (k == "step" and case["per_species"] * case["steps"] > 1 << 26) or \
            (k == "cycle" and case["level"] > 3):
        return None
    s = prepare(case, seed)
    if k in ("step", "move", "cycle"):
        st, dt = s["st"], s["dt"]
        mesh, E, B = _mesh("uniform%d" % case["level"] if k == "cycle" else case["mesh"])
        geo = _geometry(mesh)
        E = torch.as_tensor(E, device=DEV).reshape(-1, 3)
        B = torch.as_tensor(B, device=DEV).reshape(-1, 3)
        x, v, spec, blk, cell, pid = _start(st)
    if k == "move":
        code = torch.full_like(cell, 3)
        for _ in range(case["steps"]):
            old = blk * 512 + cell
            x, v, blk, _ = _push(mesh, geo, E, B, x, v, blk, torch.ones_like(x[:, 0]), dt, boris=True)
            i, _ = _stencil(geo, x, blk)
            cell = i[:, 0] + 8 * (i[:, 1] + 8 * i[:, 2])
            key = blk * 512 + cell
            # per cell the particles that stayed, then those that came, each in array order
            order = torch.argsort((2 * key + (key != old)), stable=True)
            x, v, blk, cell, pid = x[order], v[order], blk[order], cell[order], pid[order]
            code = torch.full_like(cell, 3)
        return {"x": x.T.contiguous().cpu(), "v": v.T.contiguous().cpu(), "blk": blk.int().cpu(),
                "cell": cell.int().cpu(), "id": pid.cpu(), "code": code.int().cpu()}
    if k in ("step", "cycle"):
        qm = (torch.tensor(CHARGE, dtype=torch.float64, device=DEV) / torch.tensor(MASS, dtype=torch.float64, device=DEV))
        for _ in range(case["steps"] if k == "step" else 1):
            x, v, blk, _ = _push(mesh, geo, E, B, x, v, blk, qm[spec], dt)
        if case.get("copy") == "diag":
            return _diag(mesh, geo, st.species, x, v, spec, blk, dt)
        J, Mm = _deposit(st, mesh, geo, B, x, v, spec, blk, dt, k == "cycle" or case["copy"] == "JM")
        if k == "cycle":
            return _field_step(s, J, Mm)
        return {"J": J.cpu()} if Mm is None else {"J": J.cpu(), "M": Mm.cpu()}
    # the network in 64 bits
    th = torch.as_tensor(s["sur"].params()[0].astype(np.float64), device=DEV)
    sizes = [768, 128, 16384, 128, 128, 1]
    shapes = [(128, 6), (128,), (128, 128), (128,), (128,), (1,)]

    def forward(par, X):
        W1, b1, W2, b2, w3, b3 = [t.reshape(sh) for t, sh in zip(torch.split(par, sizes), shapes)]
        gelu = torch.nn.functional.gelu
        return gelu(gelu(X @ W1.T + b1) @ W2.T + b2) @ w3 + b3

    if k == "predict":
        X = torch.as_tensor(s["X"].astype(np.float64), device=DEV)
        return torch.cat([forward(th, X[a:a + 65536]) for a in range(0, len(X), 65536)]).cpu()
    X, T = _surrogate_data(case["n"], seed)
    X, T = torch.as_tensor(X.astype(np.float64), device=DEV), torch.as_tensor(T.astype(np.float64), device=DEV)
    m, v2 = torch.zeros_like(th), torch.zeros_like(th)
    b, at = case["batch"], 0
    for t in range(1, case["steps"] + 1):
        par = th.clone().requires_grad_(True)
        loss = ((forward(par, X[at:at + b]) - T[at:at + b]) ** 2).mean()
        g, = torch.autograd.grad(loss, par)
        m, v2 = 0.9 * m + 0.1 * g, 0.999 * v2 + 0.001 * g * g
        th = th - 1e-3 * (m / (1 - 0.9 ** t)) / ((v2 / (1 - 0.999 ** t)).sqrt() + 1e-8)
        at = (at + b) % len(X)
    return {"theta": th.cpu(), "adam_steps": case["steps"]}
