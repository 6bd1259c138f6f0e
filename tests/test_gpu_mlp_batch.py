"""The one-pass training gradient at the edges of its split: one tile of 16 samples, fewer tiles than waves of a
block, a last block with idle waves, all blocks full, and a second turn of some waves.  Oracle: FP64 with the
kernel's bfloat16 operand roundings.  An operand on a rounding boundary may round the other way (about 5e-5 of
them, FP32 sums against FP64), which moves one unit of one sample by 2^-8: below 1e-3 of a block's gradient."""
import numpy as np
import pytest

from alens_amd import capi
from oracle import mlp_oracle as MO

from .test_gpu_mlp import _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [16, 48, 80, 16384, 16400, 32800])
def test_gradient_at_edges_of_the_split(B):
    X, norm = _data(B, B)
    X[:, 12:] = 3.0  # unused columns stay out of it
    P = MO.init_params(B)
    t = np.random.default_rng(B).random(B).astype(np.float32)
    with capi.Context() as ctx:
        ctx.mlp_set(P, norm)
        g, loss = ctx.mlp_gradient(X, t)
        again = ctx.mlp_gradient(X, t)
    assert loss == again[1] and np.array_equal(g.view(np.uint32), again[0].view(np.uint32))
    rl, rg = MO.loss_and_grad(P, norm, X, t, bf=True)
    assert abs(loss - rl) <= 1e-4 * rl
    edges = [MO.PW1, MO.PB1, MO.PW2, MO.PB2, MO.PW3, MO.PB3, MO.PW4, MO.PB4, MO.NPARAM]
    for a, b in zip(edges, edges[1:]):
        assert np.linalg.norm(g[a:b] - rg[a:b]) <= 2e-3 * np.linalg.norm(rg[a:b]), (a, b)
