"""Constraint stress sums against the same sums over the step's constraint blocks, added row by row: to the bit, for
no row, fewer rows than one part of the device's work (8,192), several parts, and a batch with its boxes."""
import numpy as np
import pytest

from alens_amd import capi, systems

from .test_gpu_parity import assert_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["none", "few", "parts", "batch"])
def test_stress_sums_in_row_order(kind):
    if kind == "batch":
        parts, cfg = systems.replicas(nsys=3, nmin=2000, nmax=5000, seed=41)
    else:
        rods, cfg = systems.scaled("monolayer_slab", 14000, seed=42) if kind == "parts" else \
            systems.small_3d(n=600 if kind == "few" else 1, box=3.5, seed=43)
    with capi.Context(**cfg) as c:
        c.set_systems(parts) if kind == "batch" else c.set_rods(rods)
        m = c.step()["n_con"]
        assert {"none": m == 0, "few": 0 < m < 8192}.get(kind, m > 3 * 8192 if kind == "parts" else m > 8192), m
        blocks = c.constraint_blocks()
        got, ext = c.con_stress()
    want = np.zeros(9)
    for b in blocks[:m]:
        want = want + b.gamma * np.array(b.stress[:])
    assert_bits(got, want, "stress sum")
    assert not ext.any()
