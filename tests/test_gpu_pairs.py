"""Pairs and their order against the FP64 oracle, to the bit, where cells are crowded: fewer rods than a wave, more
than the block's stage reaches, rods with hundreds of rows each; inside the box and across its periodic corner."""
import numpy as np
import pytest

from alens_amd import systems

from .test_gpu_parity import compare_full, gpu_step, O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,corner", [(2, False), (63, True), (130, False), (400, True)])
def test_crowded_cells(n, corner):
    rng = np.random.default_rng(n)
    cfg = dict(systems.COMMON, box_lo=(0, 0, 0), box_hi=(4, 4, 4), pbc=(1, 1, 1), monolayer=0, max_ite=4)
    d = rng.normal(size=(n, 3))
    c = (0.0 if corner else 1.9) + 0.12 * rng.normal(size=(n, 3))
    rods = dict(gid=np.arange(n, dtype=np.int32), center=np.mod(c, 4.0), dir=d / np.linalg.norm(d, axis=1)[:, None],
                length=rng.uniform(0.1, 0.6, n), radius=np.full(n, 0.0125), immovable=None)
    ctx, g = gpu_step(rods, cfg)
    ctx.close()
    assert n == 2 or g["report"]["n_con"] > n
    compare_full(rods, cfg, g, O.step(rods, O.cfg_from_dict(cfg)))
