"""Simulation.step takes any whole number of steps: Python and numpy integers
and floats without a fraction, with nucleation on and off."""
import numpy as np
import pytest

from pfpa import model as M
from pfpa.sim import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nucleation", [False, True])
@pytest.mark.parametrize("n", [np.int64(9), np.int32(9), np.uint8(9), 9.0, np.float64(9),
                               np.array(9)])
def test_types_of_a_count(gpu, n, nucleation):
    s = M.make_setup(40, 30, bc=1)
    f = M.init_matrix_with_particles(40, 30, s.dx, 1, seed=2, n_del=1, n_lav=0, radius=1e-9)
    a, b = (Simulation(s, f, nucleation=nucleation, nuc_every=4) for _ in range(2))
    a.step(n)
    a.step(n)
    b.step(18)
    assert a.steps_done == 18
    for x, y in zip(a.fields(), b.fields()):
        assert np.array_equal(x, y)
    with pytest.raises((ValueError, KeyError)):
        a.step(2.5)
    a.close()
    b.close()
