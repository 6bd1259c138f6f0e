"""Solves whose operator stays on the chip against the general kernel: the same products and sums in the same
order, so iteration counts, iterates and velocities agree bit for bit.  A schedule named in the environment
(ALENS_SOLVER_SPLIT=1, its default value) selects the general kernel."""
import numpy as np
import pytest

from alens_amd import capi, systems

from .test_gpu_parity import assert_bits
from .test_gpu_pool import make_ext

pytestmark = pytest.mark.gpu


def both_paths(monkeypatch, run):
    monkeypatch.setenv("ALENS_SOLVER_SPLIT", "1")
    want = run()
    monkeypatch.delenv("ALENS_SOLVER_SPLIT")
    return run(), want


def rows_problem(m):
    """m rows over about m / 2 rods of four slots each; m = 3000 hangs every row on rod 0, whose slots then
    outgrow a block."""
    rng = np.random.default_rng(m)
    hub = m == 3000
    n = m + 1 if hub else m // 2 + 5
    r = np.arange(m)
    I = np.zeros(m, np.int64) if hub else r * n // m
    J = r + 1 if hub else (I + 1 + r % 3) % n
    nrm = rng.normal(size=(m, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    return n, I, J, nrm, rng.normal(size=(m, 3)), rng.normal(size=(m, 3)), rng.normal(size=m), rng.uniform(0.5, 2.0, (n, 6))


def steps(make, nstep, ext=None):
    out = []
    with make() as c:
        for s in range(nstep):
            if s == 1 and ext is None:
                c.set_graph(True)
            if ext is not None:
                c.add_constraints(ext)
            r = c.step()
            out.append((r["iters"], r["iters_fp32"], r["n_con"], c.gamma().copy(), c.velocity()["u"].copy()))
            c.euler()
        return out, c.graph_info()


def comb():
    """3,200 short rods lie across one long one, which so has more slots than a block holds."""
    k = 3200
    x = 1.0 + 0.0245 * np.arange(k)
    long = k * 0.0245 + 0.2
    cfg = dict(systems.COMMON, box_lo=(0, 0, 0), box_hi=(long + 3, 4, 4), pbc=(0, 0, 0), monolayer=0, kT=-1.0,
               max_ite=12)  # (the long rod is summed by one lane)
    rods = dict(gid=np.arange(k + 1, dtype=np.int32), radius=np.full(k + 1, 0.0125), immovable=None,
                center=np.vstack([[1.0 + 0.01225 * (k - 1), 2.0, 2.0], np.c_[x, np.full(k, 2.0), np.full(k, 2.0245)]]),
                dir=np.vstack([[1.0, 0.0, 0.0], np.tile([0.0, 1.0, 0.0], (k, 1))]), length=np.r_[long, np.full(k, 0.2)])
    return rods, cfg


@pytest.mark.parametrize("case", [("rows", m) for m in (1, 512, 513, 1024, 1025, 131072, 131073, 262144, 262145, 3000)] +
                         [(kind, p) for kind in ("slab", "batch", "small", "sparse", "rows_of_the_caller") for p in (0, 1)] + [("comb", 0)],
                         ids=lambda c: f"{c[0]}-{c[1]}")
def test_resident_matches_general(monkeypatch, case):
    kind, v = case
    if kind == "rows":  # the edges of a chunk, of one block, and of one and two row groups on each of 256 blocks
        prob = rows_problem(v)
        x0 = np.random.default_rng(1).uniform(0.0, 0.1, v)

        def solve():
            with capi.Context(box_lo=(0, 0, 0), box_hi=(1, 1, 1), pbc=(0, 0, 0), tol=1e-9, max_ite=25, dt=1e-2) as c:
                return [c.bcqp_solve(*prob, x0=x) for x in (None, x0, 1e6 * x0)]
        got, want = both_paths(monkeypatch, solve)
        for (ga, ra), (gb, rb) in zip(got, want):
            assert ra == dict(rb, **{k: ra[k] for k in ra if k.startswith("t_")})
            assert_bits(ga, gb, f"gamma, {v} rows")
        return
    ext = None
    if kind == "batch":  # 40 systems: more shares than blocks, which take them in turn
        parts, cfg = systems.replicas(nsys=40, nmin=2000, nmax=14000, seed=31)
    elif kind == "comb":
        rods, cfg = comb()
    elif kind in ("small", "sparse"):  # one block holds the solve; it holds the rows, but not so many rods
        rods, cfg = systems.small_3d(n=800 if kind == "small" else 4000, box=3.8 if kind == "small" else 10.0, seed=35)
    elif kind == "slab":  # rods in random order: a block's rows touch more rods than its LDS keeps
        rods, cfg = systems.scaled("monolayer_slab", 60000, seed=32)
    else:
        rods, cfg = systems.small_3d(n=900, box=3.8, seed=33)
        ext = make_ext(rods, 24, seed=34)

    def make():
        c = capi.Context(**dict(cfg, precision=v))
        c.set_systems(parts) if kind == "batch" else c.set_rods(rods)
        return c
    (got, info), (want, _) = both_paths(monkeypatch, lambda: steps(make, 4, ext))
    for s, (a, b) in enumerate(zip(got, want)):
        assert a[:3] == b[:3] and a[0] + a[1] > 3, (s, a[:3], b[:3])
        assert_bits(a[3], b[3], f"gamma, step {s}")
        assert_bits(a[4], b[4], f"U, step {s}")
    if ext is None:
        assert info["replays"] >= 1, info
    if kind == "comb":  # the captured step found that a share does not fit, and was redone
        assert info["overflows"] >= 1, info
