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


@pytest.mark.parametrize("sizes,rho,box,thermostat", [
    ((8192,), 0.8442, None, 0),              # the one-workgroup rebuild chain's largest system
    ((8193,), 0.8442, None, 0),              # ... and one atom past it
    ((1023, 1024, 1025, 1), 0.8442, 10.6, 0),  # around its workgroup's width, and a single atom
    ((700,), None, 56.1, 0),                 # 8000 cells, most of them empty
    ((700,), None, 58.9, 0),                 # 9261 cells: past its cell limit
    ((1025,), 0.8442, None, 1),              # the drift leaves the maxima (Langevin)
])
def test_rebuild_chain_against_the_oracle(oracle, lj, sizes, rho, box, thermostat):
    specs = []
    for k, n in enumerate(sizes):
        side = box or (n / rho) ** (1.0 / 3.0)
        if box and n < 1000:
            parts = lj.random_insertion_array(n, [side] * 3, 0.9, 1.5, 31 + k)
        else:
            parts = lj.lattice_array(n, side, 1.0, 31 + k)
        th = lj.Langevin(1.0, 1.0, 5 + k) if thermostat else None
        specs.append((parts, lj.Settings([side] * 3, 2.5, 0.005, skin=0.3, thermostat=th)))
    sim = lj.Batch(specs)
    for steps in (1, 17, 62):
        sim.run(steps)
    ms, allp = sim.measure_now(), sim.read_particle_array()
    off = 0
    for k, (parts, st) in enumerate(specs):
        ref = oracle.Sim(np.ascontiguousarray(parts["pos"]), np.ascontiguousarray(parts["vel"]), list(st.box_size),
                         cutoff=2.5, skin=0.3, dt=0.005, thermostat=thermostat, temperature=1.0 if thermostat else 0.0,
                         friction=1.0 if thermostat else 0.0, seed=5 + k)
        ref.run(80)
        r = ref.measure()
        assert list(ms[k].raw) == list(r.raw) and ms[k].list_rebuilds == r.list_rebuilds, f"replica {k}"
        pos, vel = ref.read_particles()
        np.testing.assert_array_equal(allp["pos"][off:off + len(parts)], pos)
        np.testing.assert_array_equal(allp["vel"][off:off + len(parts)], vel)
        off += len(parts)


def test_forms_change_around_the_decision(oracle, lj):
    # drift-ahead steps, then a heat exchange (the drift's own maxima), then
    # drift-ahead steps again: each form's first step decides on its own launch
    pos, vel = oracle.lattice(1200, 11.3, 1.0, 3)
    sim = lj.LennardJones((pos, vel), lj.Settings([11.3] * 3, 2.5, 0.004, skin=0.3))
    ref = oracle.Sim(pos, vel, [11.3] * 3, cutoff=2.5, skin=0.3, dt=0.004)
    for exchange in (None, lj.HeatExchange((0.0, 2.0), (5.0, 7.0), 0.05), None):
        sim.set_heat_exchange(exchange)
        if exchange:
            ref.set_heat_exchange(exchange.hot, exchange.cold, exchange.energy)
        else:
            ref.set_heat_exchange(None, None, 0.0)
        for steps in (1, 40):
            sim.run(steps)
            ref.run(steps)
            assert list(sim.measure_now().raw) == list(ref.measure().raw)
            np.testing.assert_array_equal(sim.debug_state()[0], ref.state()[0])


@pytest.mark.parametrize("thermostat", [0, 1])  # drift-ahead steps, which swap the position sets, and plain ones
def test_calls_of_any_length_are_the_same_run(lj, thermostat):
    def simulation():
        parts, side = lj.fcc_count_array(1100, 0.8442, 1.0, 7)
        th = lj.Langevin(1.0, 1.0, 5) if thermostat else None
        return lj.LennardJones(parts, lj.Settings([side] * 3, 2.5, 0.004, skin=0.3, thermostat=th))
    one, many = simulation(), simulation()
    lengths = (1, 2, 3, 1, 4, 7, 8, 5, 15, 16, 17, 31, 6, 12, 1)
    for steps in lengths:
        many.run(steps)
    for _ in range(sum(lengths)):
        one.run(1)
    assert list(one.measure_now().raw) == list(many.measure_now().raw)
    assert one.measure_now().step == many.measure_now().step == sum(lengths)
    np.testing.assert_array_equal(one.debug_state()[0], many.debug_state()[0])
    np.testing.assert_array_equal(one.debug_state()[1], many.debug_state()[1])


@pytest.mark.parametrize("n,box,cutoff,shifted,precision", [
    (343, 8.6, 2.5, True, 0),     # one block a brick: its crew is the workgroup
    (343, 8.6, 2.5, False, 1),
    (344, 11.0, 2.5, False, 0),   # ... and an atom with no neighbour at all
    (729, 15.0, 4.5, False, 0),   # a droplet: bricks of one to three blocks, lists of up to ~40 octets
    (729, 15.0, 4.5, True, 1),
    (1728, 15.0, 4.5, True, 0),    # 1728 staged atoms leave no room for crews
    (1728, 15.0, 4.5, False, 1),
])
def test_crews_against_the_oracle(oracle, lj, n, box, cutoff, shifted, precision):
    edge = round(n ** (1.0 / 3.0))
    grid = np.resize(np.stack(np.meshgrid(*[np.arange(edge)] * 3, indexing="ij"), -1).reshape(-1, 3), (n, 3))
    rng = np.random.default_rng(17)
    pos = np.ascontiguousarray((grid - 0.5 * (edge - 1)) * 1.12 + 0.5 * box + rng.uniform(-0.03, 0.03, (n, 3)))
    if n == 344:
        pos[-1] = 0.1
    vel = np.ascontiguousarray(rng.normal(0.0, 0.7, (n, 3)))
    vel -= vel.mean(axis=0)
    sim = lj.LennardJones((pos, vel), lj.Settings([box] * 3, cutoff, 0.003, skin=0.3, shifted_force=shifted,
                                                  precision=precision))
    ref = oracle.Sim(pos, vel, [box] * 3, cutoff=cutoff, skin=0.3, dt=0.003, shifted_force=shifted,
                     precision=precision)
    for steps in (1, 40):
        sim.run(steps)
        ref.run(steps)
        assert list(sim.measure_now().raw) == list(ref.measure().raw)
        np.testing.assert_array_equal(sim.debug_state()[0], ref.state()[0])
        np.testing.assert_array_equal(sim.debug_state()[1], ref.state()[1])


def test_shared_list_builds_against_the_oracle(oracle, lj):
    # replicas of other sizes and densities on both layouts, each rebuilding on
    # its own steps: several workgroups build each brick's lists
    specs = []
    for k, (n, rho, t) in enumerate([(1000, 0.8442, 0.7), (3001, 0.05, 1.5), (2048, 0.8, 1.2), (700, 0.3, 1.0),
                                     (1, 0.02, 1.0)]):
        side = (n / rho) ** (1.0 / 3.0)
        parts = lj.lattice_array(n, max(side, 5.7), t, 41 + k)
        specs.append((parts, lj.Settings([max(side, 5.7)] * 3, 2.5, 0.004, skin=0.3)))
    sim = lj.Batch(specs)
    for steps in (1, 30, 69):
        sim.run(steps)
    ms, allp = sim.measure_now(), sim.read_particle_array()
    off = 0
    for k, (parts, st) in enumerate(specs):
        ref = oracle.Sim(np.ascontiguousarray(parts["pos"]), np.ascontiguousarray(parts["vel"]), list(st.box_size),
                         cutoff=2.5, skin=0.3, dt=0.004)
        ref.run(100)
        r = ref.measure()
        assert list(ms[k].raw) == list(r.raw) and ms[k].list_rebuilds == r.list_rebuilds, f"replica {k}"
        pos, vel = ref.read_particles()
        np.testing.assert_array_equal(allp["pos"][off:off + len(parts)], pos)
        np.testing.assert_array_equal(allp["vel"][off:off + len(parts)], vel)
        off += len(parts)


@pytest.mark.parametrize("replicas,n,density,crews", [
    (1, 8000, 0.8442, True),     # fewer dense bricks than CUs
    (1, 16384, 0.8442, False),   # ... and more, of one system
    (250, 64, 0.36, False),      # ... and of many that are a few cells each
    (32, 1000, 0.8442, False),
])
def test_crews_only_where_every_dense_brick_has_a_cu(oracle, lj, tmp_path, replicas, n, density, crews):
    side = (n / density) ** (1.0 / 3.0)
    specs = [(lj.lattice_array(n, side, 1.0, 5 + k), lj.Settings([side] * 3, 2.5, 0.004, skin=0.3))
             for k in range(replicas)]
    sim = lj.LennardJones(*specs[0]) if replicas == 1 else lj.Batch(specs)
    c = sim.debug_counters()
    assert (c["bricks"] - c["sparse_bricks"] <= 256) == crews
    assert sim.debug_launches()["crews"] == crews
    sim.run(40)
    path = tmp_path / "state"
    sim.save(path)
    back = type(sim).load(path)
    assert back.debug_launches()["crews"] == crews
    sim.tune(2)
    c = sim.debug_counters()
    assert sim.debug_launches()["crews"] == (c["bricks"] - c["sparse_bricks"] <= 256)
    sim.run(34)
    back.run(40)
    a, b = sim.read_particle_array(), back.read_particle_array()
    np.testing.assert_array_equal(a["pos"], b["pos"])
    for k in {0, replicas - 1}:
        parts, st = specs[k]
        ref = oracle.Sim(np.ascontiguousarray(parts["pos"]), np.ascontiguousarray(parts["vel"]), [side] * 3, cutoff=2.5,
                         skin=0.3, dt=0.004)
        ref.run(80)
        np.testing.assert_array_equal(a["pos"][k * n:(k + 1) * n], ref.read_particles()[0])


@pytest.mark.parametrize("n,rho,sparse", [
    (20000, 0.3, False),  # small bricks that stage few atoms of a fluid that is not dilute
    (45000, 0.2, False),
    (30011, 0.5, False),
    (45000, 0.05, True),  # ... and a gas, which the sparse layout is for
])
def test_a_spread_fluid_takes_one_layout(oracle, lj, n, rho, sparse):
    side = (n / rho) ** (1.0 / 3.0)
    if rho >= 0.3:
        parts, side = lj.fcc_count_array(n, rho, 1.3, 3)
    else:
        parts = lj.random_insertion_array(n, [side] * 3, 0.9, 1.3, 3)
    sim = lj.LennardJones(parts, lj.Settings([side] * 3, 2.5, 0.004, skin=0.3))
    ref = oracle.Sim(np.ascontiguousarray(parts["pos"]), np.ascontiguousarray(parts["vel"]), [side] * 3, cutoff=2.5,
                     skin=0.3, dt=0.004)
    c = sim.debug_counters()
    assert c["sparse_bricks"] == (c["bricks"] if sparse else 0)
    for steps in (1, 25):
        sim.run(steps)
        ref.run(steps)
        assert list(sim.measure_now().raw) == list(ref.measure().raw)
        np.testing.assert_array_equal(sim.debug_state()[0], ref.state()[0])


@pytest.mark.parametrize("shifted,precision,thermostat", [(False, 0, 0), (True, 0, 1), (True, 1, 0), (False, 1, 1)])
def test_crews_beside_cut_bricks(oracle, lj, tmp_path, shifted, precision, thermostat):
    # a film whose bricks outgrow the stage and are cut, in vapour whose bricks
    # take crews: planned without limits, loaded from a state file under the rules
    rng = np.random.default_rng(29)
    a = 15.0 / 14
    film = np.stack(np.meshgrid(np.arange(14), np.arange(14), np.arange(11), indexing="ij"), -1).reshape(-1, 3) * a
    gas = np.stack(np.meshgrid(np.arange(4), np.arange(4), np.arange(6), indexing="ij"), -1).reshape(-1, 3) * 3.6
    pos = np.concatenate([film + [0.5, 0.5, 12.5], np.where([False, False, True], gas + 26.0, gas + 0.5) % [15.0, 15.0, 36.0]])
    pos = np.ascontiguousarray((pos + rng.uniform(-0.04, 0.04, pos.shape)) % [15.0, 15.0, 36.0])
    vel = rng.normal(0.0, 0.8, pos.shape)
    vel = np.ascontiguousarray(vel - vel.mean(axis=0))
    box = [15.0, 15.0, 36.0]
    th = lj.Langevin(0.8, 0.5, 3) if thermostat else None
    with lj.debug_plan(stage_fill=100.0, sparse_fill=-1.0, parts=True):
        made = lj.LennardJones((pos, vel), lj.Settings(box, 2.5, 0.003, thermostat=th, skin=0.3, shifted_force=shifted,
                                                       precision=precision))
    ref = oracle.Sim(pos, vel, box, cutoff=2.5, skin=0.3, dt=0.003, shifted_force=shifted, precision=precision,
                     thermostat=thermostat, temperature=0.8 if thermostat else 0.0,
                     friction=0.5 if thermostat else 0.0, seed=3)
    made.run(1)
    ref.run(1)
    path = tmp_path / "film.state"
    made.save(path)
    sim = lj.LennardJones.load(path)
    assert sim.debug_launches()["crews"] and not made.debug_launches()["crews"]
    sim.record_heat_current(4)
    ref.record_heat_current(4)
    before = sim.debug_counters()
    for steps in (1, 40, 2, 120):  # fewer than the periodic check of the plan
        sim.run(steps)
        ref.run(steps)
        sim.sample_heat_current()
        ref.sample_heat_current()
        assert list(sim.measure_now().raw) == list(ref.measure().raw)
        np.testing.assert_array_equal(sim.debug_state()[0], ref.state()[0])
        np.testing.assert_array_equal(sim.debug_state()[1], ref.state()[1])
    after = sim.debug_counters()
    cut = after["stage_overflow_builds"] - before["stage_overflow_builds"]
    assert 0 < cut < (after["rebuilds"] - before["rebuilds"]) * after["bricks"]  # some bricks were cut, not all
    np.testing.assert_array_equal(sim.read_heat_current_raw(), ref.read_heat_current())
