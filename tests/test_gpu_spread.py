"""Brick plans of handles with few atoms: bricks of about one wave of home
atoms down to a single cell, on both layouts, against the oracle bit for bit
(bricks decide only how neighbourhoods are staged)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rho,shifted,precision", [
    (500, 0.85, False, 0),     # two cells per axis: a brick is one cell, its halo the same cells' images
    (1000, 0.8442, False, 0),  # 37 atoms a cell: one cell per brick
    (3458, 0.8442, True, 0),   # three cells per brick
    (3458, 0.8442, False, 1),
    (20011, 0.8442, False, 0),  # more bricks than one per CU would need
    (3001, 0.3, False, 0),     # 7 atoms a cell on average: layers on both layouts
    (4093, 0.1, True, 0),      # a gas on sparse bricks
])
def test_small_bricks_against_the_oracle(oracle, lj, n, rho, shifted, precision):
    if rho >= 0.3:
        parts, side = lj.fcc_count_array(n, rho, 1.0, 11)
    else:
        side = float(np.float32((n / rho) ** (1.0 / 3.0)))
        parts = lj.random_insertion_array(n, [side] * 3, 0.9, 1.0, 11)
    pos, vel = np.ascontiguousarray(parts["pos"]), np.ascontiguousarray(parts["vel"])
    sim = lj.LennardJones(parts, lj.Settings([side] * 3, 2.5, 0.004, skin=0.3, shifted_force=shifted,
                                             precision=precision))
    ref = oracle.Sim(pos, vel, [side] * 3, cutoff=2.5, skin=0.3, dt=0.004, shifted_force=shifted,
                     precision=precision)
    c = sim.debug_counters()
    assert c["bricks"] >= min(256, n // 128)
    assert (c["sparse_bricks"] > 0) == (rho <= 0.3) and (c["sparse_bricks"] < c["bricks"]) == (rho >= 0.3)
    for steps in (1, 60):
        sim.run(steps)
        ref.run(steps)
        assert list(sim.measure_now().raw) == list(ref.measure().raw)
        np.testing.assert_array_equal(sim.debug_state()[0], ref.state()[0])
        np.testing.assert_array_equal(sim.debug_state()[1], ref.state()[1])
