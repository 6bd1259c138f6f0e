"""Batches on the chip whose shares wait for blocks, with systems that have nothing to solve among them (no rods, rods
apart from each other) first, in between and last, and one of a single row: against the general kernel, to the bit."""
import numpy as np
import pytest

from alens_amd import capi, systems

from .test_gpu_parity import assert_bits
from .test_gpu_resident import both_paths, steps

pytestmark = pytest.mark.gpu


def pair(gap, gid):
    """Two parallel rods, their surfaces `gap` apart, in a box of their own."""
    r = systems.RADIUS
    rods = dict(gid=np.array([gid, gid + 1], np.int32), center=np.array([[2.0, 2.0, 2.0], [2.0, 2.0, 2.0 + 2 * r + gap]]),
                dir=np.tile([1.0, 0.0, 0.0], (2, 1)), length=np.ones(2), radius=np.full(2, r), immovable=None)
    return rods, dict(box_lo=(0, 0, 0), box_hi=(4, 4, 4), pbc=(0, 0, 0), monolayer=0)


def nothing():
    z = np.zeros
    return (dict(gid=z(0, np.int32), center=z((0, 3)), dir=z((0, 3)), length=z(0), radius=z(0), immovable=None),
            dict(box_lo=(0, 0, 0), box_hi=(4, 4, 4), pbc=(0, 0, 0), monolayer=0))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nsys,nmin,nmax", [(40, 2000, 14000), (2, 3000, 3001)])
def test_systems_without_rows(monkeypatch, nsys, nmin, nmax, precision):
    parts, cfg = systems.replicas(nsys=nsys, nmin=nmin, nmax=nmax, seed=51)
    g = 10_000_000
    parts = [pair(1.0, g), nothing()] + parts[:nsys // 2] + [nothing(), pair(1.0, g + 2), pair(0.01, g + 4)] + \
        parts[nsys // 2:] + [pair(1.0, g + 6), nothing()]

    def make():
        c = capi.Context(**dict(cfg, precision=precision))
        c.set_systems(parts)
        return c
    (got, info), (want, _) = both_paths(monkeypatch, lambda: steps(make, 4))
    for s, (a, b) in enumerate(zip(got, want)):
        assert a[:3] == b[:3] and a[0] + a[1] > 3, (s, a[:3], b[:3])
        assert_bits(a[3], b[3], f"gamma, step {s}")
        assert_bits(a[4], b[4], f"U, step {s}")
    assert info["replays"] >= 1, info


@pytest.mark.parametrize("kind,nsys,n,precision,want", [
    ("monolayer_slab", 5, 9000, 0, ("chip2", None)),       # two turns
    ("lognormal_3d", 6, 38000, 0, ("chip2", None)),        # three, two systems at a time
    ("lognormal_3d", 8, 34000, 0, ("stream", None)),       # eight, one at a time
    ("lognormal_3d", 24, 16000, 0, ("chip2", None)),       # eight, three at a time
    ("monolayer_slab", 5, 4000, 1, ("chip2", "chip2")),    # FP32: one turn
    ("lognormal_3d", 12, 16000, 1, ("chip2", "chip4")),    # two, nine at a time
    ("lognormal_3d", 4, 60000, 1, ("stream", "stream")),   # two, two at a time
    ("lognormal_3d", 24, 16000, 1, ("chip2", "stream"))])  # four
def test_turns(monkeypatch, kind, nsys, n, precision, want):
    """Batches that take turns on the chip, or too many of them: the kernel, the bits, and no captured step in vain."""
    parts, first = [], 0
    for q in range(nsys):
        rods, cfg = systems.scaled(kind, n, seed=7 * q + 1)
        parts.append((dict(rods, gid=rods["gid"] + first), {k: cfg[k] for k in ("box_lo", "box_hi", "pbc", "monolayer")}))
        first += n

    def run():
        out = []
        with capi.Context(**dict(systems.COMMON, precision=precision, max_ite=40)) as c:
            c.set_systems(parts)
            c.sort_rods()
            c.set_graph(True)
            for _ in range(3):  # an exact-size step, then captured ones, of the same rods
                r = c.step()
                out.append((r["n_con"], r["iters"], r["iters_fp32"], c.gamma(), c.velocity()["u"], c.route()))
            return out, c.graph_info()
    (got, info), (ref, _) = both_paths(monkeypatch, run)
    for s, (a, b) in enumerate(zip(got, ref)):
        assert a[:3] == b[:3], (s, a[:3], b[:3])
        assert_bits(a[3], b[3], f"gamma, step {s}")
        assert_bits(a[4], b[4], f"U, step {s}")
    assert [a[5] for a in got] == [want] * 3 and ref[0][5][0] == "stream", [a[5] for a in got]
    assert info["replays"] == 2 and info["captures"] == 1 and info["overflows"] == 0, info


@pytest.mark.parametrize("case", ["batch", "grown"])
def test_plan_that_suits_one_form(monkeypatch, case):
    """Captured steps in the FP32 form where one form's plan suits and the other's does not: the step is redone, and
    neither solve runs on the cleared one.  batch: FP64 takes turns on the chip, FP32 would take too many.  grown: the
    rows outgrow the one block that held the FP64 solve, the FP32 solve still fits."""
    if case == "batch":
        parts, first = [], 0
        for q in range(24):
            rods, cfg = systems.scaled("monolayer_slab", 20000, seed=7 * q + 1)
            parts.append((dict(rods, gid=rods["gid"] + first), {k: cfg[k] for k in ("box_lo", "box_hi", "pbc", "monolayer")}))
            first += 20000
        cfg = dict(systems.COMMON, max_ite=25)
    else:
        rods, cfg = systems.small_3d(n=1000, box=3.8, seed=35)
        cfg["max_ite"] = 200
        parts = None
        z = rods["center"][:, 2]
        push = np.zeros((1000, 6))
        push[:, 2] = np.where(z > np.median(z), -400.0, 400.0)

    def run():
        out = []
        with capi.Context(**dict(cfg, precision=1)) as c:
            c.set_systems(parts) if parts else c.set_rods(rods)
            c.sort_rods()
            c.set_graph(True)
            for s in range(5 if parts else 14):
                r = c.step(f_ext=None if parts else push if s >= 2 else 0 * push)
                out.append((r["n_con"], r["iters"], r["iters_fp32"], c.gamma(), c.velocity()["u"], c.route()))
                c.euler()
            return out, c.graph_info()
    (got, info), (ref, _) = both_paths(monkeypatch, run)
    for s, (a, b) in enumerate(zip(got, ref)):
        assert a[:3] == b[:3], (s, a[:3], b[:3])
        assert_bits(a[3], b[3], f"gamma, step {s}")
        assert_bits(a[4], b[4], f"U, step {s}")
    seen = [(a[0], a[5]) for a in got]
    assert info["overflows"] >= 1 and info["replays"] >= 1, (info, seen)
    want = ("chip2", "stream") if parts else ("block", "chip1")
    assert {want, ("stream", "stream") if parts else ("chip1", "chip1")} <= {r for _, r in seen}, (info, seen)
