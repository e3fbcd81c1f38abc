"""Captured steps: the first call that steps leaves every graph the handle will
use, so that no later call waits for a capture, whatever its length and
whichever of its position sets is the present one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (20, 1, 20, 2, 3, 16, 1, 4, 8, 31, 5, 6, 47, 100)


@pytest.mark.parametrize("n,form", [(1000, "nve"), (9000, "nve"), (1000, "langevin"), (9000, "nose_hoover")])
def test_no_call_after_the_first_captures(lj, n, form):
    parts, side = lj.fcc_count_array(n, 0.8442, 1.0, 7)
    th = {"nve": None, "langevin": lj.Langevin(1.0, 1.0, 5), "nose_hoover": lj.NoseHoover(1.0, 0.5)}[form]
    sim = lj.LennardJones(parts, lj.Settings([side] * 3, 2.5, 0.004, skin=0.3, thermostat=th))
    one = lj.LennardJones(parts, lj.Settings([side] * 3, 2.5, 0.004, skin=0.3, thermostat=th))
    for s in (sim, one):
        s.run(5)
    captured = sim.debug_launches()["captures"]
    assert captured > 0
    for k, steps in enumerate(LENGTHS):
        if k == 5:
            sim.record_heat_current(3)  # a new series keeps the captured steps
        sim.run(steps)
        if 5 <= k < 8:
            sim.sample_heat_current()
        assert sim.debug_launches()["captures"] == captured, f"a call of {steps} steps"
    for _ in range(sum(LENGTHS)):
        one.run(1)
    assert list(sim.measure_now().raw) == list(one.measure_now().raw)
    np.testing.assert_array_equal(sim.debug_state()[0], one.debug_state()[0])
    np.testing.assert_array_equal(sim.debug_state()[1], one.debug_state()[1])


def test_no_call_of_a_forked_batch_captures(oracle, lj):
    # both layouts on two streams, steps of many launches: single steps are replayed too
    specs = []
    for k in range(4):
        n, rho = (9000, 0.8442) if k % 2 else (9000, 0.05)
        side = (n / rho) ** (1.0 / 3.0)
        specs.append((lj.lattice_array(n, side, 1.0, 5 + k), lj.Settings([side] * 3, 2.5, 0.004, skin=0.3)))
    sim = lj.Batch(specs)
    c = sim.debug_counters()
    assert 0 < c["sparse_bricks"] < c["bricks"]
    sim.run(2)
    captured = sim.debug_launches()["captures"]
    for steps in LENGTHS:
        sim.run(steps)
        assert sim.debug_launches()["captures"] == captured, f"a call of {steps} steps"
    ms, got = sim.measure_now(), sim.read_particle_array()
    for k, (parts, st) in enumerate(specs):
        ref = oracle.Sim(np.ascontiguousarray(parts["pos"]), np.ascontiguousarray(parts["vel"]), list(st.box_size),
                         cutoff=2.5, skin=0.3, dt=0.004)
        ref.run(2 + sum(LENGTHS))
        assert list(ms[k].raw) == list(ref.measure().raw), f"replica {k}"
        np.testing.assert_array_equal(got["pos"][9000 * k:9000 * (k + 1)], ref.read_particles()[0])


def test_a_new_plan_or_form_captures_once(lj):
    parts, side = lj.fcc_count_array(2000, 0.8442, 1.0, 7)
    sim = lj.LennardJones(parts, lj.Settings([side] * 3, 2.5, 0.004, skin=0.3))
    sim.run(3)
    for change in (lambda: sim.tune(), lambda: sim.set_heat_exchange(lj.HeatExchange((0.0, 2.0), (6.0, 8.0), 0.01))):
        change()
        sim.run(3)
        captured = sim.debug_launches()["captures"]
        for steps in (20, 7, 2, 20):
            sim.run(steps)
        assert sim.debug_launches()["captures"] == captured
