"""Which kernel a solve takes, at the edges of what each holds: one block up to 1,024 rows while its slots and rods fit;
512-row chunks on 256 blocks, one, two or (FP32) four to a block; slots; else the kernel that streams its operator.
A schedule named in the environment selects that one.  (That all give the same bits is tested elsewhere.)"""
import numpy as np
import pytest

from alens_amd import capi, systems

from .test_gpu_pool import make_ext
from .test_gpu_resident import comb, rows_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,want", [(1, "block"), (512, "block"), (1024, "block"), (1025, "chip1"), (131072, "chip1"),
                                       (131073, "chip2"), (262144, "chip2"), (262145, "stream"), (3000, "stream")])
def test_stand_alone(monkeypatch, rows, want):
    prob = rows_problem(rows)
    with capi.Context(box_lo=(0, 0, 0), box_hi=(1, 1, 1), pbc=(0, 0, 0), tol=1e-9, max_ite=2, dt=1e-2) as c:
        assert c.route() == (None, None)
        c.bcqp_solve(*prob)
        assert c.route() == (want, None)
        if rows == 1025:
            c.bcqp_solve(*prob, static=True)
            assert c.route()[0] == "stream"
            monkeypatch.setenv("ALENS_SOLVER_SPLIT", "1")
            c.bcqp_solve(*prob)
            assert c.route()[0] == "stream"


# rows of the third step, so that both a plain and a captured step are seen
@pytest.mark.parametrize("kind,n,precision,want", [
    ("small", 800, 0, ("block", None)), ("small", 4000, 0, ("chip1", None)), ("small", 800, 1, ("block", "chip1")),
    ("pool", 900, 0, ("block", None)), ("slab", 20000, 1, ("chip1", "chip1")), ("slab", 60000, 0, ("chip2", None)),
    ("slab", 110000, 1, ("stream", "chip4")), ("box", 60000, 1, ("chip2", "chip2")), ("comb", 0, 0, ("stream", None))])
def test_steps(kind, n, precision, want):
    ext = None
    if kind == "comb":
        rods, cfg = comb()
    elif kind in ("small", "pool"):
        rods, cfg = systems.small_3d(n=n, box=3.8 if n < 1000 else 10.0, seed=35)
        ext = make_ext(rods, 24, seed=34) if kind == "pool" else None
    else:
        rods, cfg = systems.scaled("monolayer_slab" if kind == "slab" else "lognormal_3d", n, seed=32)
    with capi.Context(**dict(cfg, precision=precision)) as c:
        c.set_rods(rods)
        c.sort_rods()
        rows, seen = [], []
        for s in range(4):
            if s == 1:
                c.set_graph(True)
            if ext is not None:
                c.add_constraints(ext)
            rows.append(c.step()["n_con"])
            seen.append(c.route())
            c.euler()
        assert seen[2:] == [want, want], (rows, seen)


@pytest.mark.parametrize("headroom,want", [(None, "chip2"), ("8", "stream")])
def test_exchange_memory_past_4_gib(monkeypatch, headroom, want):
    """11 million rows in 256 systems: a captured step whose capacities need more exchange memory than 32-bit offsets
    reach streams its operator; with less head room it runs on the chip.  The plain step before it has the same rows."""
    if headroom:
        monkeypatch.setenv("ALENS_GRAPH_HEADROOM", headroom)
    parts, off = [], 0
    for q in range(256):
        rods, cfg = systems.scaled("monolayer_slab", 6500, seed=q)
        parts.append((dict(rods, gid=rods["gid"] + off), {k: cfg[k] for k in ("box_lo", "box_hi", "pbc", "monolayer")}))
        off += 6500
    with capi.Context(**dict(systems.COMMON, max_ite=3)) as c:
        c.set_systems(parts)
        c.sort_rods()
        c.set_graph(True)
        reps, routes, gam = [], [], []
        for _ in range(3):
            reps.append(c.step())
            routes.append(c.route()[0])
            gam.append(c.gamma())
        info = c.graph_info()
    assert reps[0]["n_con"] * 8 * 48 + off * 96 > 1 << 32, reps[0]  # three (x, g) pairs a row, two velocities a rod
    assert routes == ["chip2", want, want], routes
    assert info["captures"] == 1 and info["replays"] == 2, info
    for r, g in zip(reps[1:], gam[1:]):
        assert (r["n_con"], r["iters"]) == (reps[0]["n_con"], reps[0]["iters"])
        assert np.array_equal(g.view(np.uint64), gam[0].view(np.uint64))
