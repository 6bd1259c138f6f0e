"""Stand-alone solves of rows in any order (the adjacency is made on the device) against the FP64 oracle, to the bit:
one row, a slice's edge, rows in random order with repeated pairs, rods without rows, few rods with many rows each,
and more sort digits than one."""
import numpy as np
import pytest

from alens_amd import capi
from oracle import oracle as O

from .test_gpu_parity import assert_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(2, 1), (64, 63), (65, 130), (40, 3000), (5000, 700), (3000, 9000), (70000, 66000)])
def test_rows_in_any_order(n, m):
    rng = np.random.default_rng(n + m)
    I = rng.integers(0, n, m).astype(np.int32)
    J = ((I + 1 + rng.integers(0, n - 1, m)) % n).astype(np.int32)
    rw = {k: rng.normal(size=(m, 3)) for k in ("nrm", "rI", "rJ")}
    rw["nrm"] /= np.linalg.norm(rw["nrm"], axis=1)[:, None]
    rw = {k: v.reshape(-1) for k, v in rw.items()}
    rw["b"] = rng.normal(size=m)
    mob = rng.uniform(0.5, 2.0, 6 * n)
    cfg = dict(tol=1e-9, max_ite=15, dt=1e-2)
    with capi.Context(box_lo=(0, 0, 0), box_hi=(1, 1, 1), pbc=(0, 0, 0), **cfg) as c:
        for _ in range(2):  # the second call finds the buffers of the first
            g, rep = c.bcqp_solve(n, I, J, rw["nrm"], rw["rI"], rw["rJ"], rw["b"], mob)
            og, orep = O.bbpgd(n, I, J, rw, mob, O.make_cfg(**cfg))
            assert_bits(g, og, "gamma")
            assert rep["iters"] == orep["iters"]
            I, J = J, I  # and other rows
