"""Graph mode with caller rows now and then."""
import pytest

from alens_amd import capi, systems

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
