"""vlj_debug_cells tells what the device holds: the slots are put in cell order
by the positions their lists were built from, so a slot that holds an atom of
another cell shows. And the rebuilds' order of the atoms against the oracle's."""
import numpy as np
import pytest

from helpers import sc_liquid
from test_state_checks import sections

pytestmark = pytest.mark.gpu


def test_an_atom_in_another_cells_range_shows(oracle, lj, tmp_path):
    # a state file whose first and last slot have exchanged the positions their
    # lists were built from; nothing is launched on it
    pos, vel, box = sc_liquid(oracle, n_side=9)
    sim = lj.LennardJones((pos, vel), lj.Settings([box] * 3, 2.5, 0.005))
    sim.run(30)
    n = sim.count()
    np.testing.assert_array_equal(sim.debug_cells()[2], np.arange(n))
    path = tmp_path / "exchanged.state"
    sim.save(path)
    buf = bytearray(path.read_bytes())
    first = sections(buf)["orig"] - 3 * n * 8  # xb, yb and zb come before the original indices
    for k in range(3):
        built = np.frombuffer(buf, np.float64, n, first + k * n * 8).copy()
        built[[0, -1]] = built[[-1, 0]]
        buf[first + k * n * 8:first + (k + 1) * n * 8] = built.tobytes()
    path.write_bytes(buf)
    back = lj.LennardJones.load(path)
    cell_of, start, got = back.debug_cells()
    in_first, in_last = start[cell_of[0] + 1], start[cell_of[-1]]
    # slot n - 1 comes after the first cell's other atoms, slot 0 before the last one's
    expected = np.concatenate([np.arange(1, in_first), [n - 1], np.arange(in_first, in_last), [0],
                               np.arange(in_last, n - 1)])
    np.testing.assert_array_equal(got, expected)


@pytest.mark.parametrize("n", [729, 8192, 9261])  # the one-workgroup chain, its largest system, and past it
def test_rebuilds_order_the_atoms_as_the_oracle(oracle, lj, n):
    box = (n / 0.8442) ** (1.0 / 3.0)
    pos, vel = oracle.lattice(n, box, 1.2, 4)
    sim = lj.LennardJones((pos, vel), lj.Settings([box] * 3, 2.5, 0.005))
    ref = oracle.Sim(pos, vel, [box] * 3)
    for steps in (0, 25, 25):
        sim.run(steps)
        ref.run(steps)
        assert sim.measure_now().list_rebuilds == ref.measure().list_rebuilds
        np.testing.assert_array_equal(sim.debug_state()[3], ref.state()[3])
        for got, want in zip(sim.debug_cells(), ref.cells()):
            np.testing.assert_array_equal(got, want)
