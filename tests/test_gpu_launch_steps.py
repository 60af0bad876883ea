"""Steps per launch of a Simulation, asked for and by default, for each kind of
mask: what launch_steps says is what step() launches, counted by its calls of
pf_advance_* at one step count, and the results do not depend on it."""
import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa.sim import Simulation

pytestmark = pytest.mark.gpu

WANT = {"five": {None: 4, 1: 1, 2: 2, 3: 3, 4: 4}, "nine": {None: 4, 1: 1, 2: 2, 3: 2, 4: 4},
        "lopsided": {None: 1, 1: 1, 2: 1, 3: 1, 4: 1}}


@pytest.mark.parametrize("kind", sorted(WANT))
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_launch_steps(gpu, dtype, kind):
    s = M.make_setup(70, 50, bc=0)
    if kind == "nine":
        s.mask = M.nine_point_mask(s.dx, 1.3 * s.dx)
    elif kind == "lopsided":
        s.mask = list(s.mask)
        s.mask[3] *= 1.1
    f = M.init_matrix_with_particles(70, 50, s.dx, 0, seed=2, n_del=1, n_lav=1, radius=1e-9)
    results = []
    for asked, want in WANT[kind].items():
        sim = Simulation(s, f, dtype=dtype, steps_per_launch=asked)
        assert sim.launch_steps == want, asked
        most, native = [], sim._advance

        def advance(*args):
            most.append(args[-3])       # steps per launch
            return native(*args)

        sim._advance = advance
        sim.step(11)
        assert len(most) == 1
        assert sim.launch_steps == min(want, most[0]) and most[0] >= want
        results.append(sim.fields())
        sim.close()
    for other in results[1:]:
        for x, y in zip(results[0], other):
            assert np.array_equal(x, y)


def test_bad_requests(gpu):
    s = M.make_setup(40, 30, bc=1)
    f = M.init_matrix_with_particles(40, 30, s.dx, 1, seed=2, n_del=1, n_lav=0, radius=1e-9)
    for mask in (s.mask, M.nine_point_mask(s.dx, s.dx)):
        s.mask = mask
        for bad in (0, 5, -1):
            with pytest.raises(ValueError):
                Simulation(s, f, steps_per_launch=bad)
