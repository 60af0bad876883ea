"""pf_advance_*: n steps in one call give the bits of n one-step launches, for
five- and nine-point masks (grouped up to four steps per launch), for masks
that are neither (one per launch), on grids at the edges of strips and chunks
and on those too small for a multi-step launch."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa.sim import Simulation

pytestmark = pytest.mark.gpu


def _setup(Nx, Ny, bc, kind):
    s = M.make_setup(Nx, Ny, bc=bc, dt_rule=3e-7)
    if kind == "nine":
        s.mask = M.nine_point_mask(s.dx, s.dx)
    if kind == "nine oblong":
        s.mask = M.nine_point_mask(s.dx, 1.3 * s.dx)
    if kind == "lopsided":
        s.mask = list(s.mask)
        s.mask[3] *= 1.1
    return s


@pytest.mark.parametrize("kind", ["five", "nine", "nine oblong", "lopsided"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("shape", [(2, 9), (3, 3), (4, 4), (55, 9), (57, 58), (121, 33), (60, 301)])
def test_advance_matches_one_step_launches(gpu, shape, bc, dtype, kind):
    Nx, Ny = shape
    s = _setup(Nx, Ny, bc, kind)
    rng = np.random.default_rng(7 * Nx + Ny)
    shp = (Ny + 2, Nx + 2)
    pd = np.clip(rng.uniform(-0.3, 1.3, shp), 0, 1)
    f0 = [0.3 + 0.01 * rng.standard_normal(shp), 0.02 + 0.005 * rng.standard_normal(shp), pd,
          np.clip(rng.uniform(-0.5, 1.0, shp), 0, 1) * (pd < 0.3)]
    f0 = [M.fill_ghosts(a, bc) for a in f0]
    a = Simulation(s, f0, dtype=dtype)
    b = Simulation(s, f0, dtype=dtype, steps_per_launch=1)
    for n in (0, 1, 3, 6, 11):
        a.step(n)
        for _ in range(n):
            b.step(1)
        assert a.steps_done == b.steps_done
        for x, y in zip(a.fields(), b.fields()):
            assert np.array_equal(x, y), (n, np.abs(x - y).max())
    a.close()
    b.close()


def test_advance_refuses_bad_calls(gpu):
    s = M.make_setup(64, 48, bc=1)
    sim = Simulation(s, M.init_matrix_with_particles(64, 48, s.dx, 1, n_del=1, n_lav=0,
                                                     radius=2e-9))
    from pfpa._lib import lib
    vec = lambda f: (ctypes.c_void_p * 4)(*[x.data_ptr() for x in f])  # noqa: E731
    in_b = ctypes.c_int()
    call = lambda a, b, most, nx=66: lib().pf_advance_f64(  # noqa: E731
        sim.ctx, nx, 50, 1, ctypes.byref(sim.P), a, b, 4, most, ctypes.byref(in_b), None)
    a, b = vec(sim.a), vec(sim.b)
    assert call(a, b, 5) == 1 and call(a, b, 0) == 1          # steps per launch
    assert call(a, a, 4) == 1                                 # one set for both
    assert call(a, vec([sim.b[0], sim.b[0], sim.b[2], sim.b[3]]), 4) == 1
    assert call(vec([sim.a[0], sim.a[0], sim.a[2], sim.a[3]]), b, 4) == 1
    assert call(None, b, 4) == 1 and call(a, None, 4) == 1
    assert call(a, b, 4, nx=2) == 1                           # no interior
    sim.close()
