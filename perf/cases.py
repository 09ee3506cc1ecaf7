"""The work whose speed is measured: time steps of whole simulations and the
blocks a program calls on their own, through the package's public entry points.

A case is a dict of plain values with a `kind`:

  steps     `Simulation.step(n)` and the fields a caller reads back after it
  density   NEIGHBOR + PNUM: the neighbour lists and the particle number density
  pressure  PRESSURECALC: PPE assembly, solve and clamp (Jacobi-CG or the
            learned preconditioner; FP64 or mixed precision)
  slot      vox_cgm_slot on device arrays in the reference's slot layout
  grad      loss and gradient of the learned preconditioner on a stored PPE

`wx, wy, wz` is the water column in particles (wz = 0: 2D); tanks follow the
proportions of the dam breaks of voxarmps_amd.cases.
"""
import ctypes as C
import functools
import math
import os

import numpy as np
import torch

import voxarmps_amd as vx

FIELDS_2D = ("X", "Y", "U", "V", "P", "N")
FIELDS_3D = ("X", "Y", "Z", "U", "V", "W", "P", "N")
WEIGHTS = os.path.join(os.path.dirname(vx.__file__), "data", "lpc_weights.npy")


def _c(name, kind, wx, wy, wz=0, l0=0.01, **more):
    return {"name": name, "kind": kind, "wx": wx, "wy": wy, "wz": wz, "l0": l0, **more}


def listed():
    return [
        # the 2D dam break of the framework's first configuration: a small run,
        # bound by launches and host waits
        _c("dam2d_small", "steps", 25, 50, model="plain", precision="fp64", n=10),
        # a two-phase 2D run with SPS-LES and a Bingham fluid, all in FP64
        _c("dam2d_two_phase", "steps", 173, 131, model="two_phase", precision="fp64", n=5),
        # the weakly compressible model: cubic kernel, one radius, no PPE
        _c("dam2d_weakly_compressible", "steps", 311, 207, l0=0.004, model="wc", precision="fp64",
           n=5),
        # the 3D dam break at half the benchmark's linear size
        _c("dam3d_half", "steps", 50, 50, 40, l0=0.005, model="plain", precision="fp64", n=4),
        # the benchmark: 1,175,450 particles, FP64 and mixed precision
        _c("dam3d_full", "steps", 100, 100, 80, l0=0.005, model="plain", precision="fp64", n=4),
        _c("dam3d_full_mixed", "steps", 100, 100, 80, l0=0.005, model="plain", precision="mixed",
           n=4),
        # 64 uneven two-phase 2D dam breaks batched in one context
        _c("ensemble64", "steps", 0, 0, l0=0.01, model="ensemble", precision="mixed", n=4,
           scenarios=64),
        # density evaluation on the reference's own single 3D radius, ragged sizes
        _c("density3d", "density", 67, 59, 41, l0=0.01, radii="one"),
        # one pressure solve of a mid-sized ragged 3D system
        _c("pressure3d", "pressure", 75, 71, 53, l0=0.005, solver="jacobi", precision="fp64"),
        # the solve on a caller's own device arrays (the reference's CUDA layout)
        _c("slot3d", "slot", 31, 29, 23, l0=0.005),
        # a pressure solve with the learned preconditioner
        _c("pressure3d_learned", "pressure", 50, 50, 40, l0=0.005, solver="learned",
           precision="fp64"),
        # training of the preconditioner: one gradient on a stored 3D system
        _c("lpc_grad3d", "grad", 25, 25, 20, l0=0.005),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "density", "pressure", "pressure", "slot", "grad"])

    def box3(lo, hi):
        n = _log_int(rng, lo, hi)             # particles in the column
        a, b = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
        e = (n / (a * b)) ** (1.0 / 3.0)
        return {"wx": max(8, int(e * a)), "wy": max(8, int(e * b)), "wz": max(8, int(e))}

    def box2(lo, hi):
        n = _log_int(rng, lo, hi)
        a = rng.uniform(0.5, 2.0)
        return {"wx": max(10, int(math.sqrt(n * a))), "wy": max(10, int(math.sqrt(n / a))), "wz": 0}

    if kind == "steps":
        if rng.random() < 0.5:
            return {"kind": kind, **box3(4000, 700000), "l0": 0.005, "model": "plain",
                    "precision": rng.choice(["fp64", "fp64", "mixed"]), "n": rng.randint(2, 4)}
        model = rng.choice(["plain", "two_phase", "wc", "ensemble"])
        if model == "ensemble":
            return {"kind": kind, "wx": 0, "wy": 0, "wz": 0, "l0": 0.01, "model": model,
                    "precision": "mixed", "n": rng.randint(2, 4), "scenarios": rng.randint(4, 64)}
        return {"kind": kind, **box2(1000, 200000), "l0": 0.004 if model == "wc" else 0.01,
                "model": model, "precision": rng.choice(["fp64", "fp64", "mixed"]),
                "n": rng.randint(3, 8)}
    if kind == "density":
        if rng.random() < 0.6:
            return {"kind": kind, **box3(4000, 500000), "l0": 0.01,
                    "radii": rng.choice(["one", "two"])}
        return {"kind": kind, **box2(1000, 300000), "l0": 0.01, "radii": rng.choice(["one", "two"])}
    if kind == "pressure":
        solver, precision = rng.choice([("jacobi", "fp64"), ("jacobi", "mixed"), ("learned", "fp64")])
        if rng.random() < 0.6:
            return {"kind": kind, **box3(4000, 300000), "l0": 0.005, "solver": solver,
                    "precision": precision}
        return {"kind": kind, **box2(1000, 100000), "l0": 0.01, "solver": solver,
                "precision": precision}
    if kind == "slot":
        if rng.random() < 0.6:
            return {"kind": kind, **box3(4000, 60000), "l0": 0.005}
        return {"kind": kind, **box2(1000, 60000), "l0": 0.01}
    if rng.random() < 0.5:
        return {"kind": kind, **box3(4000, 40000), "l0": 0.005}
    return {"kind": kind, **box2(1000, 60000), "l0": 0.01}


# ---- geometry ---------------------------------------------------------------------------
def _dim(case):
    return 3 if case["wz"] else 2


def _tank(case):
    wx, wy, wz = case["wx"], case["wy"], case["wz"]
    if wz:
        return (16 * wx // 5, max(6 * wy // 5, wy + 4), wz + 1)
    return (4 * wx, wy + 20)


@functools.lru_cache(maxsize=2)
def _lattice(wx, wy, wz, l0, tank):
    if wz:
        return vx.dam_break(3, l0, (wx, wy, wz), tank)
    return vx.dam_break(2, l0, (wx, wy), tank)


@functools.lru_cache(maxsize=1)
def _ensemble(scenarios, l0):
    return vx.ensemble_c4(scenarios, seed=scenarios, l0=l0)


def _set_motion(cs, rng, height, speed):
    """A divergence-free initial velocity of a few random modes, as a run that
    is under way has, and a slight disorder of the lattice."""
    f = cs.ptype > 0
    x, y = cs.x[f] / height, cs.y[f] / height
    u, v = np.zeros(x.shape), np.zeros(x.shape)
    for _ in range(4):
        kx, ky, ph = rng.uniform(1, 6), rng.uniform(1, 6), rng.uniform(0, 2 * math.pi)
        a = speed * rng.uniform(0.3, 1.0) / math.hypot(kx, ky)
        c = np.cos(kx * x + ky * y + ph)
        u += a * ky * c
        v -= a * kx * c
    cs.u[f], cs.v[f] = u, v
    for q in (cs.x, cs.y) + ((cs.z,) if cs.dim == 3 else ()):
        q[f] += rng.uniform(-1e-4, 1e-4, x.shape[0]) * cs.l0


def _lattice_sum(dim, k):
    """Particle number density of a full lattice: radius k spacings, kernel k/r - 1."""
    m = int(math.ceil(k)) + 1
    g = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * dim, indexing="ij"), -1).reshape(-1, dim)
    r = np.sqrt((g.astype(np.float64) ** 2).sum(1))
    r = r[(r > 0) & (r < k)]
    return float(np.sum(k / r - 1.0))


def _block_inputs(case, seed):
    """Positions, types, PND and free-surface flags of a filled tank in
    disorder, and the densities of its lattice: what the density, pressure,
    slot and grad kinds start from."""
    d = _dim(case)
    base = _lattice(case["wx"], case["wy"], case["wz"], case["l0"], _tank(case))
    cs = vx.jitter(base, 0.05 * base.l0, seed=seed)
    rng = np.random.default_rng(seed)
    n0s, n0l = _lattice_sum(d, 2.1), _lattice_sum(d, 4.0)
    l0, fluid = base.l0, base.ptype > 0
    top = base.y[fluid].max()
    right = base.x[fluid].max()
    near = (base.x < right + 1.5 * l0) & (base.y < top - 0.5 * l0)
    bcon = np.where(base.ptype < 0, -1, np.where(near, 0, 1)).astype(np.int32)
    ph = rng.uniform(0, 2 * math.pi, 3)
    wave = (2.0 + np.sin(7 * cs.x / right + ph[0]) * np.cos(5 * cs.y / top + ph[1])
            + 0.2 * rng.uniform(-1, 1, cs.tp))
    pnd = n0s * (1.0 + 1e-6 * wave)
    return cs, pnd, bcon, n0s, n0l


def _block_params(cs):
    return vx.dam3d_params(cs) if cs.dim == 3 else vx.dam2d_params(cs, tol=1e-8)


def _block_sim(case, seed, **options):
    cs, pnd, bcon, n0s, n0l = _block_inputs(case, seed)
    p = _block_params(cs)
    for k, v in options.items():
        setattr(p, k, v)
    sim = vx.Simulation(p, cs)
    sim.init()
    sim.set_n0(n0s, n0l)
    sim.set("N", pnd)
    sim.set("BCON", bcon)
    return sim


# ---- prepare ------------------------------------------------------------------------------
def _prepare_steps(case, seed):
    rng = np.random.default_rng(seed)
    mixed = case["precision"] == "mixed"
    regions = None
    if case["model"] == "ensemble":
        base, reg, boxes, _ = _ensemble(case["scenarios"], case["l0"])
        cs, regions = base.copy(), (reg, boxes)
        p = vx.ensemble_params(base)
        height, speed = 2.0, 0.1
    else:
        base = _lattice(case["wx"], case["wy"], case["wz"], case["l0"], _tank(case))
        cs = base.copy()
        height, speed = float(base.y[base.ptype > 0].max()), 0.1
        if case["model"] == "two_phase":
            cs = vx.two_phase(cs)
            p = vx.ensemble_params(base)
        elif case["model"] == "wc":
            p = vx.wc_params(base)
        else:
            p = vx.dam3d_params(base) if base.dim == 3 else vx.dam2d_params(base)
    p.precision = vx._abi.PREC_MIXED if mixed else vx._abi.PREC_FP64
    _set_motion(cs, rng, height, speed)
    sim = vx.Simulation(p, cs)
    if regions is not None:
        sim.set_regions(*regions)
    sim.init()
    for k in ("U", "V"):                       # what the SPS stage reads in the first step
        sim.set(k + "NEW", getattr(cs, k.lower()))
    sim.step(2)
    return {"sim": sim, "n": case["n"], "fields": FIELDS_3D if cs.dim == 3 else FIELDS_2D}


def _prepare_density(case, seed):
    base = _lattice(case["wx"], case["wy"], case["wz"], case["l0"], _tank(case))
    cs = vx.jitter(base, 0.1 * base.l0, seed=seed)
    p = _block_params(cs) if case["radii"] == "two" else vx.set_box(
        vx.default_params(cs.dim, cs.l0), cs)
    return {"sim": vx.Simulation(p, cs)}


def _prepare_pressure(case, seed):
    learned = case["solver"] == "learned"
    sim = _block_sim(case, seed,
                     solver=vx._abi.SOLVER_LEARNED_FCG if learned else vx._abi.SOLVER_JACOBI_CG,
                     precision=vx._abi.PREC_MIXED if case["precision"] == "mixed"
                     else vx._abi.PREC_FP64)
    net = None
    if learned:
        net = vx.LearnedPreconditioner()
        net.set_weights(np.load(WEIGHTS, allow_pickle=False))
        sim.attach_lpc(net)
        sim.PRESSURECALC()                     # the Jacobi-CG solve that fixes the baseline
    return {"sim": sim, "net": net}


def _prepare_slot(case, seed):
    s = _system(case, seed)
    tp, i, j, val = s["tp"], s["i"], s["j"], s["val"]
    dev = val.device
    cnt = torch.bincount(i, minlength=tp)
    stride = int(cnt.max()) + 2
    first = torch.cumsum(cnt, 0) - cnt
    slot = torch.arange(i.numel(), device=dev) - first[i] + 2
    at = (i + 1) * stride + slot
    neighb = torch.zeros((tp + 1) * stride, dtype=torch.int32, device=dev)
    poiss = torch.zeros((tp + 1) * stride, dtype=torch.float64, device=dev)
    head = (torch.arange(tp, device=dev) + 1) * stride + 1
    neighb[head] = (cnt + 1).to(torch.int32)
    neighb[at] = (j + 1).to(torch.int32)
    poiss[head] = s["diag"]
    poiss[at] = -val
    source = torch.zeros(tp + 1, dtype=torch.float64, device=dev)
    source[1:] = s["rhs"]
    bcon = torch.zeros(tp + 1, dtype=torch.int32, device=dev)
    bcon[1:] = s["bcon"].to(torch.int32)
    f = vx.hip_backend().lib.vox_cgm_slot
    f.restype = C.c_int
    f.argtypes = [C.c_int, C.c_int] + [C.c_void_p] * 5 + [C.c_double, C.c_int,
                                                          C.POINTER(vx._abi.VoxSolveInfo)]
    return {"f": f, "tp": tp, "stride": stride, "arrays": (neighb, poiss, source, bcon),
            "x": torch.zeros(tp + 1, dtype=torch.float64, device=dev)}


def _prepare_grad(case, seed):
    sim = _block_sim(case, seed)
    sim.MATRIX()
    net = vx.LearnedPreconditioner()
    net.set_weights(np.load(WEIGHTS, allow_pickle=False))
    index = net.dump(sim)
    sim.close()
    return {"net": net, "index": index}


def prepare(case, seed):
    return {**{"steps": _prepare_steps, "density": _prepare_density, "pressure": _prepare_pressure,
               "slot": _prepare_slot, "grad": _prepare_grad}[case["kind"]](case, seed),
            "kind": case["kind"]}


# ---- run ----------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "steps":
        sim = state["sim"]
        sim.step(state["n"])
        return {k: sim.get(k) for k in state["fields"]}
    if kind == "density":
        sim = state["sim"]
        sim.NEIGHBOR()
        sim.PNUM()
        return {"N": sim.get("N")}
    if kind == "pressure":
        sim = state["sim"]
        sim.PRESSURECALC()
        return {"PNEW": sim.get("PNEW"), "SOURCE": sim.get("SOURCE")}
    if kind == "slot":
        info = vx._abi.VoxSolveInfo()
        x = state["x"]
        rc = state["f"](state["tp"], state["stride"], *(a.data_ptr() for a in state["arrays"]),
                        x.data_ptr(), 1e-8, 500, C.byref(info))
        if rc != 0:
            raise RuntimeError(f"vox_cgm_slot: {rc}")
        return {"pnew": x}
    loss, grad = state["net"].loss_grad(state["index"], 12345)
    return {"loss": np.array([loss]), "grad": grad}


# ---- work ---------------------------------------------------------------------------------
def _count(case):
    """(particles, fluid particles) of a case."""
    if case["kind"] == "steps" and case["model"] == "ensemble":
        base = _ensemble(case["scenarios"], case["l0"])[0]
        return base.tp, base.fp
    wx, wy, wz = case["wx"], case["wy"], case["wz"]
    t = _tank(case)
    shell = (t[0] + 5) * (t[1] + 3) * ((t[2] + 5) if wz else 1)
    inside = (t[0] - 1) * t[1] * ((t[2] - 1) if wz else 1)
    fluid = wx * wy * (wz or 1)
    return shell - inside + fluid, fluid


def _ball(dim, k):
    m = int(math.ceil(k)) + 1
    g = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * dim, indexing="ij"), -1).reshape(-1, dim)
    r2 = (g ** 2).sum(1)
    return int(np.count_nonzero((r2 > 0) & (r2 < k * k)))


def work(case):
    """Bytes: each array of a pass read once and written once - the fields, the
    neighbour lists (4 bytes an entry, written once per search and read once
    by every stage that walks them), the matrix (a column of at least 2 bytes
    and a value of 4 or 8) once per assembly and per product. Flops: the terms of
    the sums that these stand for."""
    d = 2 if case["kind"] == "steps" and case["model"] == "ensemble" else _dim(case)
    n, f = _count(case)
    if case["kind"] == "density":
        one = case["radii"] == "one"
        es = _ball(d, (3.2 if d == 3 else 4.0) if one else 2.1)
        el = 0 if one else _ball(d, 4.0)
        return {"bytes": n * (d * 8 + 8) * 2 + 4 * n * (2 * es + el), "flops": n * (es * 20 + el * 8)}
    es, el = _ball(d, 2.1), _ball(d, 4.0)
    wc = case["kind"] == "steps" and case["model"] == "wc"
    if wc:
        es = el = _ball(d, 4.0)
    vb = 4 if case.get("precision") == "mixed" else 8
    nu = f
    product = nu * (el * (2 + vb) + 4 * 8)
    assemble = nu * (4 * el + el * (2 + vb) + 3 * 8) + n * (d * 8 + 4)
    iters = {"learned": 10}.get(case.get("solver"), 15)
    solve = iters * (product + 9 * 8 * nu)
    if case["kind"] == "pressure":
        return {"bytes": assemble + solve + 2 * 8 * n, "flops": nu * el * (25 + 2 * iters)}
    if case["kind"] == "slot":
        return {"bytes": iters * nu * (el * 12 + 9 * 8), "flops": nu * el * 2 * iters}
    if case["kind"] == "grad":
        dense = 8 * 64 + 3 * (64 * 64 + 2 * 64 * 16) + 2 * 64
        # forward and backward: the graph's 3 aggregations each way, 4 probes
        # through the matrix twice, and the rows' activations and gradients
        return {"bytes": nu * el * 8 * (6 + 8) + nu * (4 * 64 * 2 + 3 * 16 * 2) * 3,
                "flops": nu * (6 * dense + el * (2 * 16 * 6 + 2 * 8))}
    lists = 0 if wc else nu * 4 * el
    stages = 10 if case["model"] in ("two_phase", "ensemble") else 6
    step = (4 * n * (es * (1 + stages) + (0 if wc else el)) + lists + n * 8 * (12 * d + 16)
            + (0 if wc else assemble + solve))
    return {"bytes": case["n"] * step,
            "flops": case["n"] * n * (es * 20 * stages + el * (0 if wc else 60 + 2 * iters))}


# ---- 64-bit references in plain torch ---------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pairs(pos, radius):
    """Every ordered pair (i, j), j != i, closer than radius, sorted by i, and
    its distance."""
    n, d = pos.shape
    lo = pos.min(0).values
    cell = ((pos - lo) / (radius * (1 + 1e-9))).floor().long()
    dims = [int(v) + 1 for v in cell.max(0).values]
    key = cell[:, 0]
    for a in range(1, d):
        key = key * dims[a] + cell[:, a]
    order = torch.argsort(key, stable=True)
    total = int(np.prod(dims))
    count = torch.bincount(key, minlength=total)
    start = torch.cumsum(count, 0) - count
    rows, cols, dist = [], [], []
    ids = torch.arange(n, device=pos.device)
    for off in np.ndindex(*[3] * d):
        c = cell + torch.tensor(off, device=pos.device) - 1
        ok = torch.ones(n, dtype=torch.bool, device=pos.device)
        k = torch.zeros(n, dtype=torch.long, device=pos.device)
        for a in range(d):
            ok &= (c[:, a] >= 0) & (c[:, a] < dims[a])
            k = k * dims[a] + c[:, a].clamp(0, dims[a] - 1)
        m = torch.where(ok, count[k], 0)
        s = start[k]
        for q in range(int(m.max()) if n else 0):
            i = ids[m > q]
            j = order[s[i] + q]
            r = (pos[j] - pos[i]).square().sum(1).sqrt()
            keep = (r < radius) & (j != i)
            rows.append(i[keep])
            cols.append(j[keep])
            dist.append(r[keep])
    i, j, r = torch.cat(rows), torch.cat(cols), torch.cat(dist)
    by = torch.argsort(i * n + j)
    return i[by], j[by], r[by]


def _positions(cs):
    p = np.stack([cs.x, cs.y] + ([cs.z] if cs.dim == 3 else []), 1)
    return torch.from_numpy(p).to(_device())


def _system(case, seed):
    """The PPE of the block inputs: value and pair of every coupling, diagonal
    and right-hand side per particle (functions.cu:869-1005, method 1)."""
    cs, pnd, bcon, n0s, n0l = _block_inputs(case, seed)
    p = _block_params(cs)
    pos = _positions(cs)
    i, j, r = _pairs(pos, p.re_l)
    b = torch.from_numpy(bcon).to(pos.device)
    m = (b[i] == 0) & (b[j] != -1)
    i, j, r = i[m], j[m], r[m]
    val = 2.0 * cs.dim / p.lambda_ * (p.re_l / r - 1.0) / n0l / p.rho1
    unk = b == 0
    # row sums over the padded rows: the same bits each time
    cnt = torch.bincount(i, minlength=cs.tp)
    wide = torch.zeros(cs.tp, max(int(cnt.max()), 1), dtype=torch.float64, device=pos.device)
    wide[i, torch.arange(i.numel(), device=pos.device) - (torch.cumsum(cnt, 0) - cnt)[i]] = val
    diag = wide.sum(1) + 1e-7 / p.dt / p.dt
    del wide
    rhs = torch.from_numpy((pnd - n0s) / n0s / p.dt / p.dt).to(pos.device)
    return {"tp": cs.tp, "i": i, "j": j, "r": r, "val": val, "diag": torch.where(unk, diag, 1.0),
            "rhs": torch.where(unk, rhs, 0.0), "bcon": b, "pos": pos, "case": cs, "params": p,
            "pnd": torch.from_numpy(pnd).to(pos.device), "n0l": n0l}


def _solve(s):
    """Conjugate gradients to the last digits in 64 bits."""
    m = s["bcon"][s["j"]] == 0
    i, j, val = s["i"][m], s["j"][m], s["val"][m]

    def times(v):
        return s["diag"] * v - torch.zeros_like(v).index_add_(0, i, val * v[j])

    x = torch.zeros_like(s["rhs"])
    r = s["rhs"].clone()
    p = r / s["diag"]
    z = p
    rz = torch.dot(r, z)
    stop = 1e-15 * float(torch.linalg.norm(r))
    for _ in range(200):
        q = times(p)
        a = rz / torch.dot(p, q)
        x = x + a * p
        r = r - a * q
        if float(torch.linalg.norm(r)) <= stop:
            break
        z = r / s["diag"]
        new = torch.dot(r, z)
        p = z + new / rz * p
        rz = new
    return x


def _rademacher(seed, probe, n):
    with np.errstate(over="ignore"):
        z = (np.uint64(seed) + (np.uint64(probe) << np.uint64(32))
             + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return np.where(z >> np.uint64(63), -1.0, 1.0)


def _exact_grad(case, seed):
    s = _system(case, seed)
    p, dev, cs = s["params"], s["pos"].device, s["case"]
    rows = torch.nonzero(s["bcon"] == 0)[:, 0]
    nu = rows.numel()
    num = torch.full((s["tp"],), -1, dtype=torch.long, device=dev)
    num[rows] = torch.arange(nu, device=dev)
    m = s["bcon"][s["j"]] == 0
    i, j, o = num[s["i"][m]], num[s["j"][m]], s["val"][m]
    off = (s["pos"][s["j"][m]] - s["pos"][s["i"][m]]) / p.re_l
    diag, rhs = s["diag"][rows], s["rhs"][rows]
    zero = torch.zeros(nu, dtype=torch.float64, device=dev)
    osum = zero.index_add(0, i, o)
    f = torch.zeros(nu, 8, dtype=torch.float64, device=dev)
    f[:, 0] = s["pnd"][rows] / s["n0l"]
    f[:, 1] = torch.from_numpy((cs.ptype == 0).astype(np.float64)).to(dev)[rows]
    f[:, 2] = osum / diag
    for a in range(cs.dim):
        f[:, 3 + a] = zero.index_add(0, i, o * off[:, a]) / osum
    w = torch.from_numpy(np.load(WEIGHTS, allow_pickle=False).astype(np.float64)).to(dev)
    w.requires_grad_(True)
    at = 0

    def take(*shape):
        nonlocal at
        k = int(np.prod(shape))
        at += k
        return w[at - k:at].reshape(shape)

    w0, b0 = take(64, 8), take(64)
    h = torch.relu(f @ w0.T + b0)
    for _ in range(3):
        P, U, V, c = take(16, 64), take(64, 64), take(64, 16), take(64)
        msg = h @ P.T
        agg = torch.zeros(nu, 16, dtype=torch.float64, device=dev)
        agg = agg.index_add(0, i, o[:, None] * msg[j]) / osum[:, None]
        h = torch.relu(h @ U.T + agg @ V.T + c)
    wo, bo = take(2, 64), take(2)
    out = h @ wo.T + bo
    g = torch.exp(0.5 * torch.tanh(out[:, 0]))
    sc = torch.sqrt(2.5 * torch.sigmoid(out[:, 1] - math.log(1.5)))
    one = 2.0 * cs.dim / p.lambda_ * (p.re_l / p.dl - 1.0) / s["n0l"] / p.rho1
    strong = o >= 0.25 * one
    si, sj = i[strong], j[strong]
    so = o[strong] / diag[si] / diag[sj]
    loss = 0.0
    for probe in range(4):
        v = rhs if probe == 0 else torch.from_numpy(_rademacher(12345, probe, nu)).to(dev)
        z = g / diag * v + sc * zero.index_add(0, si, so * (sc * v)[sj])
        e = diag * z - zero.index_add(0, i, o * z[j]) - v
        loss = loss + e.square().sum() / v.square().sum() / 4
    loss.backward()
    return {"loss": np.array([float(loss.detach())]), "grad": w.grad}


def exact(case, seed):
    kind = case["kind"]
    if kind == "steps":
        return None                            # hundreds of chained stages on a moving state
    if kind == "density":
        base = _lattice(case["wx"], case["wy"], case["wz"], case["l0"], _tank(case))
        cs = vx.jitter(base, 0.1 * base.l0, seed=seed)
        p = _block_params(cs) if case["radii"] == "two" else vx.set_box(
            vx.default_params(cs.dim, cs.l0), cs)
        i, _, r = _pairs(_positions(cs), p.re_s)
        n = torch.zeros(cs.tp, dtype=torch.float64, device=r.device)
        return {"N": n.index_add_(0, i, p.re_s / r - 1.0)}
    if kind == "pressure":
        s = _system(case, seed)
        x = _solve(s)
        return {"PNEW": x.clamp(s["params"].pmin, 4.5 * s["tp"]), "SOURCE": s["rhs"]}
    if kind == "slot":
        s = _system(case, seed)
        return {"pnew": torch.cat([torch.zeros(1, dtype=torch.float64, device=s["rhs"].device),
                                   _solve(s)])}
    return _exact_grad(case, seed)
