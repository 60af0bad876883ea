"""Simulation.tune_tile on a grid that four steps run by tiles: what an untuned
simulation runs is among the candidates, and stays where it is the fastest."""
import pytest

from pfpa import model as M
from pfpa.sim import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 256])
def test_tiles_are_a_candidate(gpu, n):
    s = M.make_setup(n, n, bc=1)
    sim = Simulation(s, M.init_matrix_with_particles(n, n, s.dx, 1, seed=4, radius=2e-9))
    heights = []
    set_tile4 = sim.set_tile4

    def record(rows, depth=0):
        heights.append(rows)
        set_tile4(rows, depth)

    sim.set_tile4 = record
    sim.step(64)
    rows, times = sim.tune_tile(launches=40)
    assert 0 in times and len(times) > 5
    # 4.3 against 7.6 us a launch at 128^2, 5.7 against 8.8 at 256^2
    assert rows == 0 and heights[-1] == 0
    sim.close()
    three = Simulation(s, M.init_matrix_with_particles(n, n, s.dx, 1, seed=4, radius=2e-9),
                       steps_per_launch=3)
    assert 0 not in three.tune_tile(launches=2)[1]
    three.close()
