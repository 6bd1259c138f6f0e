"""The training gradient where hidden units leave the range of exp: far below zero a unit and its slope are 0, far above
it is its input.  Oracle: FP64 with the kernel's bfloat16 operand roundings; the bound is that of ordinary inputs."""
import numpy as np
import pytest

from alens_amd import capi
from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("z", [-3.0e38, -1.0e30, -1.0e4, -89.0, -87.0, -86.0, 86.0, 87.0, 1.0e4, 1.0e30])
def test_units_out_of_range(z):
    """Every second unit of the first layer gets z; where z is large, the next layer's weights bring it back."""
    rng = np.random.default_rng(7)
    P = MO.init_params(4)
    W1, W2 = P[MO.PW1:MO.PB1].reshape(64, 16), P[MO.PW2:MO.PB2].reshape(64, 64)
    W1[:, 0] = 0.0
    W1[::2] = 0.0
    W1[::2, 0] = 1.0
    X = np.zeros((64, 16), np.float32)
    X[:, 1:12] = rng.normal(size=(64, 11))
    X[:, 0] = z
    if z > 0:
        W2[:, ::2] = W2[:, ::2] / np.float32(z)
    norm = np.concatenate([np.zeros(12), np.ones(12), [0.7]]).astype(np.float32)
    t = rng.random(64).astype(np.float32)
    with np.errstate(over="ignore"):
        rl, rg = MO.loss_and_grad(P, norm, X, t, bf=True)
    with capi.Context() as ctx:
        ctx.mlp_set(P, norm)
        g, loss = ctx.mlp_gradient(X, t)
    assert abs(loss - rl) <= 1e-4 * rl, (loss, rl)
    edges = [MO.PB1, MO.PW2, MO.PB2, MO.PW3, MO.PB3, MO.PW4, MO.PB4, MO.NPARAM]  # (W1's own gradient holds z as a factor)
    for a, b in zip(edges, edges[1:]):
        assert np.isfinite(g[a:b]).all()
        assert np.linalg.norm(g[a:b] - rg[a:b]) <= 2e-3 * np.linalg.norm(rg[a:b]), (a, b)
