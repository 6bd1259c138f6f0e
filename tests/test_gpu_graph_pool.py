"""Graph mode with caller rows now and then: a step with them has exact sizes, the steps before and after it are
captured ones.  Everything read after each step (rows, impulses, velocities, stress, features, the network's energy)
agrees bit for bit with a context that never captures: with few caller rows, with more than the captured capacity
(so that the row buffers move), and where the captured step has more rows than the exact one, on chip and in the FP32
form."""
import numpy as np
import pytest

from alens_amd import capi, systems
from oracle import mlp_oracle as MO

from .test_gpu_mlp import _data
from .test_gpu_parity import assert_bits
from .test_gpu_pool import make_ext

pytestmark = pytest.mark.gpu


def test_captured_after_caller_rows():
    """The first captured step follows one with caller rows, whose bounds and compliances are not its own."""
    rods, cfg = systems.small_3d(n=900, box=3.8, seed=41)
    ext = make_ext(rods, 300, seed=6)
    ctx = [capi.Context(**cfg) for _ in range(2)]
    for c in ctx:
        c.set_rods(rods)
    ctx[0].set_graph(True)
    for s in range(4):
        if s == 0:
            for c in ctx:
                c.add_constraints(ext)
        ra, rb = (c.step() for c in ctx)
        assert (ra["n_con"], ra["iters"]) == (rb["n_con"], rb["iters"]), (s, ra, rb)
        assert_bits(ctx[0].gamma(), ctx[1].gamma(), f"gamma, step {s}")
        for c in ctx:
            c.euler()
    assert ctx[0].graph_info()["replays"] == 3


@pytest.mark.parametrize("kind,n,me,precision", [("small_3d", 900, 24, 0), ("small_3d", 900, 24, 1), ("small_3d", 4000, 4000, 0),
                                                 ("monolayer_slab", 9000, 40, 0), ("monolayer_slab", 9000, 9000, 0),
                                                 ("monolayer_slab", 40000, 40, 1)])
def test_pool_rows_between_captured_steps(monkeypatch, kind, n, me, precision):
    # caller rows past the captured capacity; else room for the rows of the captured steps that follow
    monkeypatch.setenv("ALENS_GRAPH_HEADROOM", "1.05" if me == n else "3")
    rods, cfg = systems.scaled(kind, n, seed=n + me)
    ext = make_ext(rods, me, seed=5)
    _, norm = _data(1, 64)
    ctx = [capi.Context(**dict(cfg, precision=precision)) for _ in range(2)]
    for c in ctx:
        c.set_rods(rods)
        c.mlp_set(MO.init_params(3), norm)
    ctx[0].set_graph(True)
    z = rods["center"][:, 2]
    out = np.zeros((n, 6))
    out[:, 2] = np.where(z > np.median(z), 20.0, -20.0)
    ncol = []
    for s in range(8):
        if s in (3, 5):
            for c in ctx:
                c.add_constraints(ext)
        f = out if s < 3 else -out  # apart, then together: in the slab, many more rows after step 5
        ra, rb = (c.step(f_ext=f) for c in ctx)
        ncol.append(ra["n_con"] - (me if s in (3, 5) else 0))
        assert (ra["n_con"], ra["iters"], ra["iters_fp32"]) == (rb["n_con"], rb["iters"], rb["iters_fp32"]), (s, ra, rb)
        a, b = ctx
        assert_bits(a.gamma(), b.gamma(), f"gamma, step {s}")
        va, vb = a.velocity(), b.velocity()
        for k in va:
            assert_bits(va[k], vb[k], f"{k}, step {s}")
        ga, gb = a.constraint_arrays(), b.constraint_arrays()
        for k in ga:
            assert np.array_equal(ga[k], gb[k]) if ga[k].dtype.kind == "i" else assert_bits(ga[k], gb[k], f"{k}, step {s}") is None
        for x, y in zip(a.con_stress(), b.con_stress()):
            assert_bits(np.asarray(x), np.asarray(y), f"stress, step {s}")
        assert np.array_equal(a.features().view(np.uint32), b.features().view(np.uint32)), s
        if s not in (3, 5):
            ea, eb = a.mlp_energy(grad=True), b.mlp_energy(grad=True)
            assert ea[0] == eb[0] and np.array_equal(ea[1].view(np.uint32), eb[1].view(np.uint32)), s
        for c in ctx:
            c.euler()
    if me == 40:
        assert ncol[6] > 1.5 * ncol[5], ncol
    info = ctx[0].graph_info()
    assert info["captures"] >= 3 and info["replays"] >= 3 and info["capture_failures"] == 0, info
