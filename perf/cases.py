"""The work a user of the library has it do, as cases that can be timed and compared.

Every case goes through the public entry points (alens_amd.capi, the ctypes face of
include/alens_capi.h) as a simulation program does: rods are loaded once, a number of steps relax
the random start, and a pass is one constraint step at that state, with its impulses and velocities
read back into the program's own arrays (a program that couples proteins or writes results reads
them on the host).  A step does not move the rods (the Euler call does), so a pass can be repeated.

Fields of a case: "do" is step, solve, predict or train.
  step     system ("filament", "box", "dense_box", "layer", "replicas"), rods (replicas: systems and
           the range of rods per system), relax (steps taken before), graph (captured steps), precision (0 FP64,
           1 FP32 iterations with FP64 refinement), network (learned warm start), stress (the program also
           reads the constraint stress, as the reference's step loop does)
  solve    the stand-alone BCQP solve on rows the program brings itself
  predict  the warm-start network on feature rows
  train    the warm-start network's training on (features, impulse) pairs
"""
import ctypes
import math

import numpy as np
import torch

from alens_amd import capi, systems, warmstart

# constraint rows per rod and BBPGD iterations of a pass, as these systems have them
ROWS = {"filament": 2.0, "box": 0.8, "dense_box": 3.05, "layer": 2.36, "replicas": 2.7}
ITERS = {"filament": 45, "box": 37, "dense_box": 125, "layer": 100, "replicas": 110}


def listed():
    return [
        # a bead-spring filament, the reference's flexible filament example: spheres linked by bilateral
        # springs handed over every step through the constraint pool; latency decides
        dict(name="filament_400", do="step", system="filament", rods=400, relax=0, graph=False, precision=0,
             network=False, stress=True),
        # a sparse 3-D suspension of 1,000 rods: the smallest collision-only step
        dict(name="box_1k", do="step", system="box", rods=1000, relax=0, graph=False, precision=0,
             network=False, stress=False),
        # the reference's dense monolayer example has 9,702 rods; plain steps as the C++ adapter runs them
        dict(name="layer_9k7", do="step", system="layer", rods=9702, relax=12, graph=False, precision=0,
             network=False, stress=True),
        # a mid-size layer in captured steps
        dict(name="layer_45k", do="step", system="layer", rods=45_001, relax=12, graph=True, precision=0,
             network=False, stress=False),
        # the benchmark's 200,000-rod layer and 1,000,000-rod lognormal box, captured steps
        dict(name="layer_200k", do="step", system="layer", rods=200_000, relax=12, graph=True, precision=0,
             network=False, stress=False),
        dict(name="box_1m", do="step", system="dense_box", rods=1_000_000, relax=8, graph=True, precision=0,
             network=False, stress=False),
        # the FP32 form with the learned warm start, at the layer's size and in a 3-D box
        dict(name="form_layer_200k", do="step", system="layer", rods=200_000, relax=12, graph=True, precision=1,
             network=True, stress=False),
        dict(name="form_box_60k", do="step", system="dense_box", rods=60_000, relax=10, graph=True, precision=1,
             network=True, stress=False),
        # a parameter sweep: 64 independent replicas of uneven size, boxes and layers, in one launch
        dict(name="replicas_64", do="step", system="replicas", systems=64, lo=2000, hi=20_000, relax=6,
             graph=True, precision=0, network=False, stress=False),
        # BCQPSolver on rows from the program's own collision finder
        dict(name="solve_30k", do="solve", rods=30_000, rows=75_011),
        # the network alone: inference, and one epoch of training at the default batch
        dict(name="predict_250k", do="predict", rows=250_003),
        dict(name="train_120k", do="train", rows=120_000, batch=4096, epochs=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["step"] * 8 + ["solve", "predict", "train"])
    if do == "solve":
        n = _log_int(rng, 300, 60_000)
        return dict(do=do, rods=n, rows=int(n * rng.uniform(0.8, 2.6)))
    if do == "predict":
        return dict(do=do, rows=_log_int(rng, 1000, 500_000))
    if do == "train":
        return dict(do=do, rows=_log_int(rng, 5000, 200_000), batch=rng.choice([1024, 2048, 4096, 8192]), epochs=1)
    system = rng.choice(["filament", "box", "dense_box", "layer", "layer", "replicas"])
    if system == "replicas":
        return dict(do=do, system=system, systems=rng.randint(3, 64), lo=2000, hi=_log_int(rng, 4000, 20_000), relax=6,
                    graph=rng.random() < 0.7, precision=rng.choice([0, 0, 1]), network=False, stress=False)
    lo, hi = {"filament": (100, 4000), "box": (600, 200_000), "dense_box": (16_000, 900_000),
              "layer": (500, 300_000)}[system]
    n = _log_int(rng, lo, hi)
    fresh = system == "filament" or (system == "box" and n <= 2500)
    form = not fresh and rng.random() < 0.3
    return dict(do=do, system=system, rods=n, relax=0 if fresh else 8, graph=not fresh and rng.random() < 0.6,
                precision=1 if form else 0, network=form, stress=n <= 20_000 and rng.random() < 0.5)


# ---- systems ----------------------------------------------------------------------------------
FILAMENT = dict(col_buf=0.02, viscosity=1.0, kT=0.00411, dt=1e-4, tol=1e-5, max_ite=1_000_000, seed=1234,
                box_lo=(-5, -5, -5), box_hi=(5, 5, 5), pbc=(0, 0, 0))
LINK_KAPPA, LINK_GAP, BEAD = 3650.0, 0.0002, 0.01


def _filament(n, seed):
    """Beads along a gentle helix, jittered by a tenth of a per cent of their diameter."""
    rng = np.random.default_rng(seed)
    step = 2 * BEAD + LINK_GAP
    R, pitch = 1.5, 0.08
    w = step / math.hypot(R, pitch / (2 * math.pi))
    a = w * np.arange(n)
    c = np.stack([R * np.cos(a), R * np.sin(a), pitch * a / (2 * math.pi) - 1.0], axis=1)
    c = c + rng.normal(0, 2e-5, (n, 3))
    d = np.tile([0.0, 0.0, 1.0], (n, 1))
    rods = dict(gid=np.arange(n, dtype=np.int32), center=c, dir=d, length=np.zeros(n), radius=np.full(n, BEAD),
                immovable=None)
    return rods, dict(FILAMENT, seed=seed % (1 << 31))


def _links(rods):
    """Springs between consecutive beads, from surface to surface along the line of centres."""
    c = rods["center"]
    n = len(c)
    d = c[:-1] - c[1:]
    dist = np.linalg.norm(d, axis=1)
    nrm = d / dist[:, None]
    return dict(I=np.arange(n - 1), J=np.arange(1, n), nrm=nrm, pos=BEAD * nrm, delta0=dist - 2 * BEAD - LINK_GAP)


def _blocks(links):
    """The pool's blocks (alens_con_block), as setProteinConstraints leaves them."""
    m = len(links["I"])
    arr = (capi.ConBlock * m)()
    for e in range(m):
        b = arr[e]
        b.delta0, b.kappa, b.bilateral = links["delta0"][e], LINK_KAPPA, 1
        b.gid_i, b.gid_j = int(links["I"][e]), int(links["J"][e])
        for a in range(3):
            n = links["nrm"][e, a]
            b.norm_i[a], b.norm_j[a] = n, -n
            b.pos_i[a], b.pos_j[a] = -links["pos"][e, a], links["pos"][e, a]
            for q in range(3):
                b.stress[3 * a + q] = -links["nrm"][e, a] * links["nrm"][e, q] * 2 * BEAD
    return arr


def _replica_sizes(case):
    """Rods per replica: evenly spread over the logarithm of lo .. hi, in no order."""
    k = (np.arange(case["systems"]) * 29 % 61 + 0.5) / 61
    return np.round(case["lo"] * (case["hi"] / case["lo"]) ** k).astype(int)


def _replicas(case, seed):
    """Independent systems, boxes and layers in turn, as systems.replicas builds them, of given sizes."""
    parts, first = [], 0
    for q, n in enumerate(_replica_sizes(case)):
        n = int(n)
        if q % 2 == 0:
            rods, cfg = systems.lognormal_3d(n=n, box=(n / 64.0) ** (1 / 3), lmax=1.5, seed=seed + 7 * q + 1)
        else:
            rods, cfg = systems.monolayer_slab(n=n, side=math.sqrt(n / 20.0), seed=seed + 7 * q + 2)
        parts.append((dict(rods, gid=rods["gid"] + first), {k: cfg[k] for k in ("box_lo", "box_hi", "pbc", "monolayer")}))
        first += n
    return parts, dict(systems.COMMON, box_lo=(0, 0, 0), box_hi=(1, 1, 1), pbc=(0, 0, 0), seed=seed)


def _system(case, seed):
    """(rods or list of systems, configuration) of a step case."""
    kind = case["system"]
    if kind == "filament":
        return _filament(case["rods"], seed)
    if kind == "replicas":
        return _replicas(case, seed)
    return systems.scaled({"box": "small_3d", "dense_box": "lognormal_3d", "layer": "monolayer_slab"}[kind],
                          case["rods"], seed=seed)


# ---- rows and features a program brings itself --------------------------------------------------
SOLVE = dict(dt=1e-4, tol=1e-5, max_ite=100_000)


def _rows(case, seed):
    """A contact network: rod k touches rods near it in index order; gaps of both signs."""
    rng = np.random.default_rng(seed)
    n, m = case["rods"], case["rows"]
    I = np.sort(rng.integers(0, n, m))
    J = (I + 1 + np.minimum(rng.geometric(0.02, m), n - 2)) % n
    I, J = np.minimum(I, J).astype(np.int32), np.maximum(I, J).astype(np.int32)
    order = np.lexsort((J, I))
    I, J = I[order], J[order]
    nrm = rng.normal(size=(m, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    t = rng.normal(size=(n, 3))
    t /= np.linalg.norm(t, axis=1, keepdims=True)
    s, u = rng.uniform(-0.5, 0.5, m), rng.uniform(-0.5, 0.5, m)
    rI, rJ = np.cross(s[:, None] * t[I], nrm), np.cross(u[:, None] * t[J], nrm)
    b = rng.normal(0.008, 0.012, m)
    mob = np.empty((n, 6))
    mob[:, :3] = t
    mob[:, 3:] = _drag(np.full(n, 1.0), np.full(n, systems.RADIUS), 0.01)
    return dict(n=n, I=I, J=J, nrm=nrm, rI=rI, rJ=rJ, b=b, mob=mob)


def _features(m, seed):
    """Feature rows with the ranges that relaxed contact states have, and impulses to learn."""
    rng = np.random.default_rng(seed)
    X = np.zeros((m, 16), np.float32)
    gap = rng.uniform(-0.004, 0.025, m)
    nrm = rng.normal(size=(m, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    v = rng.normal(0, 0.006, (m, 3))
    L = np.exp(rng.normal(0, 0.25, (m, 2)))
    prev = np.where(rng.random(m) < 0.4, rng.exponential(0.3, m), 0.0)
    X[:, 0], X[:, 1:4], X[:, 4:6], X[:, 6:9], X[:, 9:11], X[:, 11] = gap, nrm, rng.uniform(-1, 1, (m, 2)), v, L, prev
    push = np.maximum(0.0, -(gap + np.sum(nrm * v, axis=1)))
    gamma = (40.0 * push * L[:, 0] + 0.2 * prev * (push > 0)).astype(np.float32)
    return X, gamma


# ---- what a program has in hand, and a pass -----------------------------------------------------
class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    if case["do"] == "solve":
        s.ctx = capi.Context(**SOLVE)
        s.rows = _rows(case, seed)
        return s
    if case["do"] in ("predict", "train"):
        s.ctx = capi.Context()
        s.X, s.gamma = _features(case["rows"], seed)
        s.net = warmstart.load()
        s.ctx.mlp_set(*s.net)
        return s
    data, cfg = _system(case, seed)
    ctx = s.ctx = capi.Context(**dict(cfg, precision=case["precision"], warm_start=2 if case["network"] else 0))
    s.blocks = None
    if case["system"] == "replicas":
        ctx.set_systems(data)
        ctx.sort_rods()
    else:
        ctx.set_rods(data)
        if case["system"] == "filament":
            s.blocks = _blocks(_links(data))
        elif case["relax"]:
            ctx.sort_rods()
    if case["network"]:
        ctx.mlp_set(*warmstart.load())
    if case["graph"]:
        ctx.set_graph(True)
    for _ in range(case["relax"]):
        if s.blocks is not None:
            _add(ctx, s.blocks)
        ctx.step()
        ctx.euler()
    # the program's arrays for the results: velocities, and impulses with room for twice the usual rows
    s.u = np.zeros(6 * ctx.n)
    s.gamma = np.zeros(int(2 * ROWS[case["system"]] * _rods(case)) + 512)
    return s


def _rods(case):
    if case["system"] != "replicas":
        return case["rods"]
    return int(_replica_sizes(case).sum())


def _add(ctx, blocks):
    ctx._check(capi.lib().alens_add_constraints(ctx._h, len(blocks), blocks))


def _f64(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def run(s):
    ctx, case = s.ctx, s.case
    if case["do"] == "solve":
        r = s.rows
        gamma, rep = ctx.bcqp_solve(r["n"], r["I"], r["J"], r["nrm"], r["rI"], r["rJ"], r["b"], r["mob"])
        return {"gamma": gamma, "iters": rep["iters"]}
    if case["do"] == "predict":
        return {"gamma0": ctx.mlp_predict(s.X)}
    if case["do"] == "train":
        ctx.mlp_set(*s.net)
        loss = ctx.mlp_train(s.X, s.gamma, epochs=case["epochs"], batch=case["batch"], lr=1e-3, seed=5)
        return {"params": ctx.mlp_get()[0], "loss": loss}
    if s.blocks is not None:
        _add(ctx, s.blocks)
    rep = ctx.step()
    m = rep["n_con"]
    if s.gamma.size < m:
        raise RuntimeError(f"{m} rows: the impulse array holds {s.gamma.size}")
    ctx._check(capi.lib().alens_get_gamma(ctx._h, _f64(s.gamma)))
    ctx._check(capi.lib().alens_get_velocity(ctx._h, _f64(s.u), None, None, None))
    out = {"rows": m, "iters": rep["iters"] + rep["iters_fp32"], "gamma": s.gamma, "u": s.u}
    if case["stress"]:
        out["stress"], out["link_stress"] = ctx.con_stress()
    return out


def work(case):
    """Bytes and operations a pass cannot do without: every matvec of the solve streams the operator's rows
    and the rod vectors once (per row 23 words and 16 B of indices, per rod 18 words), collection and
    write-back touch rods and rows once."""
    if case["do"] == "predict":
        m = case["rows"]
        return {"bytes": 68.0 * m + 4 * 9473, "flops": 2.0 * m * (16 * 64 + 2 * 64 * 64 + 64)}
    if case["do"] == "train":
        m = case["rows"] // case["batch"] * case["batch"] * case["epochs"]
        return {"bytes": 68.0 * m + 24 * 9473.0, "flops": 6.0 * m * (16 * 64 + 2 * 64 * 64 + 64)}
    if case["do"] == "solve":
        n, m, it, w = case["rods"], case["rows"], 92, 8
    else:
        kind, n = case["system"], _rods(case)
        m, it, w = ROWS[kind] * n, ITERS[kind], 4 if case["precision"] else 8
    matvec = m * (23 * w + 16) + 18 * w * n
    return {"bytes": it * matvec + 192.0 * m + 328.0 * n, "flops": it * (74.0 * m + 25.0 * n)}


# ---- the same results in 64 bits ----------------------------------------------------------------
def _drag(L, r, mu):
    """1/zperp, 1/zpar - 1/zperp, 1/zrot of rods; spheres (L < 2 r) by Stokes."""
    ball = L < 2 * r
    bb = -(1.0 + 2.0 * np.log(r / np.where(ball, 4 * r, L)))
    zpar = np.where(ball, 6 * np.pi * mu * r, 8 * np.pi * mu * L / (2 * bb))
    zperp = np.where(ball, 6 * np.pi * mu * r, 8 * np.pi * mu * L / (bb + 2))
    zrot = np.where(ball, 8 * np.pi * mu * r ** 3, 2 * np.pi * mu * L ** 3 / (3 * (bb + 2)))
    return np.stack([1 / zperp, 1 / zpar - 1 / zperp, 1 / zrot], axis=1)


def _philox(ctr, key):
    """Philox4x32-10 on arrays of counters."""
    c = [np.asarray(x, np.uint64) for x in ctr]
    k0, k1 = key
    mask = np.uint64(0xFFFFFFFF)
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & mask, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1),
             p0 & mask]
    return c


def _brownian(gid, seed, step):
    z = []
    key = (seed & 0xFFFFFFFF, seed >> 32)
    for q in range(3):
        one = np.ones(len(gid), np.uint64)
        o = _philox([np.asarray(gid, np.uint64), one * np.uint64(step), one * np.uint64(0), one * np.uint64(q)], key)
        u1 = (((o[0] << np.uint64(21)) ^ (o[1] >> np.uint64(11))).astype(np.float64) + 1.0) * 2.0 ** -53
        u2 = ((o[2] << np.uint64(21)) ^ (o[3] >> np.uint64(11))).astype(np.float64) * 2.0 ** -53
        R = np.sqrt(-2.0 * np.log(u1))
        z += [R * np.cos(2 * np.pi * u2), R * np.sin(2 * np.pi * u2)]
    return np.stack(z, axis=1)


def _closest(ci, ti, hi, cj, tj, hj):
    """Arc positions of the closest points of two segments (rows of arrays)."""
    dot = lambda a, b: np.sum(a * b, axis=1)  # noqa: E731
    r = ci - cj
    b, d, e = dot(ti, tj), dot(ti, r), dot(tj, r)
    det = 1.0 - b * b
    s = np.clip(np.where(det > 1e-14, (b * e - d) / np.where(det > 1e-14, det, 1.0), 0.0), -hi, hi)
    u = np.clip(b * s + e, -hj, hj)
    s = np.clip(b * u - d, -hi, hi)
    return s, u


def _contacts(rods, cfg):
    """Pairs I < J closer than col_buf, in ascending (I, J): brute force over all pairs."""
    c, t, r = rods["center"], rods["dir"], rods["radius"]
    L = rods["length"]
    h = np.where(L < 2 * r, 0.0, 0.5 * L)
    box = np.asarray(cfg["box_hi"], float) - np.asarray(cfg["box_lo"], float)
    pbc = np.asarray(cfg["pbc"], bool)
    I, J = np.triu_indices(len(L), 1)
    d = c[J] - c[I]
    img = np.where(pbc, -np.round(d / box), 0.0)
    near = np.linalg.norm(d + img * box, axis=1) < h[I] + h[J] + r[I] + r[J] + cfg["col_buf"]
    I, J, img = I[near], J[near], img[near]
    cj = c[J] + img * box
    s, u = _closest(c[I], t[I], h[I], cj, t[J], h[J])
    D = (c[I] + s[:, None] * t[I]) - (cj + u[:, None] * t[J])
    dist = np.linalg.norm(D, axis=1)
    gap = dist - r[I] - r[J]
    k = gap < cfg["col_buf"]
    I, J, D, dist = I[k], J[k], D[k], dist[k]
    return dict(I=I, J=J, nrm=D / dist[:, None], posI=s[k, None] * t[I], posJ=u[k, None] * t[J], gap=gap[k], D=D)


def _lcp(r, dt, lb, invk, device, tol=1e-13, most=60_000):
    """gamma of the bounded-constraint problem by projected gradients with Barzilai-Borwein steps, far below
    the tolerance of a run, and the generalised forces D gamma."""
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=device)  # noqa: E731
    I, J = dev(np.asarray(r["I"], np.int64)), dev(np.asarray(r["J"], np.int64))
    wI = torch.cat([dev(r["nrm"]), dev(r["rI"])], dim=1)
    wJ = -torch.cat([dev(r["nrm"]), dev(r["rJ"])], dim=1)
    mob, b, lb, invk = dev(r["mob"]), dev(r["b"]), dev(lb), dev(invk)
    n = len(mob)

    def force(x):
        f = torch.zeros(n, 6, dtype=torch.float64, device=device)
        return f.index_add_(0, I, wI * x[:, None]).index_add_(0, J, wJ * x[:, None])

    def velocity(f):
        t = mob[:, :3]
        along = (t * f[:, :3]).sum(1, keepdim=True)
        return torch.cat([mob[:, 3:4] * f[:, :3] + mob[:, 4:5] * along * t, mob[:, 5:6] * f[:, 3:]], dim=1)

    def grad(x):
        u = velocity(force(x))
        return dt * ((wI * u[I]).sum(1) + (wJ * u[J]).sum(1)) + invk * x + b

    x = torch.zeros_like(b).maximum(lb)
    g = grad(x)
    ag = grad(g) - b
    alpha = (g * g).sum() / (g * ag).sum()
    for it in range(1, most + 1):
        xn = (x - alpha * g).maximum(lb)
        gn = grad(xn)
        sv, yv = xn - x, gn - g
        x, g = xn, gn
        if it % 25 == 0 and float((x - (x - g).maximum(lb)).abs().max()) < tol:
            break
        sy = (sv * yv).sum()
        new = (sv * sv).sum() / sy if it % 2 else sy / (yv * yv).sum()
        alpha = torch.where(torch.isfinite(new) & (new > 0), new, alpha)
    f = force(x)
    return x.cpu().numpy(), velocity(f).cpu().numpy()


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _exact_step(case, seed):
    rods, cfg = _system(case, seed)
    cfg = dict(systems.COMMON, **cfg)
    n, t = len(rods["length"]), rods["dir"]
    mob = np.concatenate([t, _drag(rods["length"], rods["radius"], cfg["viscosity"])], axis=1)
    z = _brownian(rods["gid"], cfg["seed"], 0)
    sq, sp, sr = np.sqrt(mob[:, 3]), np.sqrt(mob[:, 3] + mob[:, 4]), np.sqrt(mob[:, 5])
    along = ((sp - sq) * np.sum(t * z[:, :3], axis=1))[:, None] * t
    unc = math.sqrt(2 * cfg["kT"] / cfg["dt"]) * np.concatenate([sq[:, None] * z[:, :3] + along, sr[:, None] * z[:, 3:]], axis=1)
    k = _contacts(rods, cfg)
    mc = len(k["I"])
    lb, invk = np.zeros(mc), np.zeros(mc)
    links = _links(rods) if case["system"] == "filament" else None
    if links is not None:
        k = dict(I=np.concatenate([k["I"], links["I"]]), J=np.concatenate([k["J"], links["J"]]),
                 nrm=np.concatenate([k["nrm"], links["nrm"]]), posI=np.concatenate([k["posI"], -links["pos"]]),
                 posJ=np.concatenate([k["posJ"], links["pos"]]), gap=np.concatenate([k["gap"], links["delta0"]]), D=k["D"])
        lb = np.concatenate([lb, np.full(len(links["I"]), -np.inf)])
        invk = np.concatenate([invk, np.full(len(links["I"]), 1.0 / LINK_KAPPA)])
    r = dict(k, rI=np.cross(k["posI"], k["nrm"]), rJ=np.cross(k["posJ"], k["nrm"]), mob=mob)
    w = np.sum(r["nrm"] * (unc[k["I"], :3] - unc[k["J"], :3]) + r["rI"] * unc[k["I"], 3:] - r["rJ"] * unc[k["J"], 3:], axis=1)
    r["b"] = k["gap"] + cfg["dt"] * w
    gamma, u = _lcp(r, cfg["dt"], lb, invk, _device())
    full = np.zeros(int(2 * ROWS[case["system"]] * n) + 512)
    full[:len(gamma)] = gamma
    out = {"rows": None, "iters": None, "gamma": full, "u": (unc + u).reshape(-1)}
    if case["stress"]:
        out["stress"] = np.einsum("k,ki,kj->ij", gamma[:mc], k["D"][:mc], k["nrm"][:mc])
        out["link_stress"] = np.zeros((3, 3)) if links is None else -2 * BEAD * np.einsum(
            "k,ki,kj->ij", gamma[mc:], links["nrm"], links["nrm"])
    return out


def _net(P, norm, X):
    """The network in 64 bits: scaled impulses of feature rows."""
    W1, b1, W2, b2, W3, b3, w4, b4 = torch.split(P, [1024, 64, 4096, 64, 4096, 64, 64, 1])
    h = (X[:, :12].double() - norm[:12]) * norm[12:24]
    silu = torch.nn.functional.silu
    h = silu(h @ W1.view(64, 16)[:, :12].T + b1)
    h = silu(h @ W2.view(64, 64).T + b2)
    h = silu(h @ W3.view(64, 64).T + b3)
    return torch.nn.functional.softplus(h @ w4 + b4)


def _exact_train(case, seed):
    X, gamma = _features(case["rows"], seed)
    P, norm = (torch.as_tensor(a, device=_device()).double() for a in warmstart.load())
    X = torch.as_tensor(X, device=P.device)
    t = torch.as_tensor(gamma, device=P.device).double() / norm[24]
    m, B = case["rows"], case["batch"]
    mask = (1 << 64) - 1
    rs, step = 5 ^ 0xD1B54A32D192ED03, 0
    m1, m2 = torch.zeros_like(P), torch.zeros_like(P)
    loss = []
    for _ in range(case["epochs"]):
        idx = list(range(m))
        for i in range(m - 1, 0, -1):  # the order of the library's seeded shuffle
            rs ^= rs >> 12
            rs = (rs ^ (rs << 25)) & mask
            rs ^= rs >> 27
            j = (((rs * 2685821657736338717) & mask) >> 11) % (i + 1)
            idx[i], idx[j] = idx[j], idx[i]
        idx = torch.tensor(idx, device=P.device)
        got = []
        for q in range(m // B):
            pick = idx[q * B:(q + 1) * B]
            p = P.clone().requires_grad_(True)
            err = ((_net(p, norm, X[pick]) - t[pick]) ** 2).mean()
            g, = torch.autograd.grad(err, p)
            step += 1
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            P = P - 1e-3 * (m1 / (1 - 0.9 ** step)) / (torch.sqrt(m2 / (1 - 0.999 ** step)) + 1e-8)
            got.append(float(err))
        loss.append(sum(got) / len(got))
    return {"params": P.cpu().numpy(), "loss": np.array(loss)}


def exact(case, seed):
    if case["do"] == "predict":
        X, _ = _features(case["rows"], seed)
        P, norm = (torch.as_tensor(a, device=_device()).double() for a in warmstart.load())
        return {"gamma0": (norm[24] * _net(P, norm, torch.as_tensor(X, device=P.device))).cpu().numpy()}
    if case["do"] == "train":
        return _exact_train(case, seed)
    if case["do"] == "solve":
        r = _rows(case, seed)
        gamma, _ = _lcp(r, SOLVE["dt"], np.zeros(len(r["b"])), np.zeros(len(r["b"])), _device())
        return {"gamma": gamma, "iters": None}
    # states that earlier steps of the library have relaxed, and systems too large to search pair by pair,
    # have no value of their own
    if case["relax"] or case["system"] == "replicas" or case["rods"] > 2500:
        return None
    return _exact_step(case, seed)
