"""A matrix at rest stays at rest: where both compositions are gamma's
equilibrium ones everywhere the potentials are zero, and the Laplacian of a
constant adds nothing, though the mask's entries do not add up to zero in
their last bits (at a cell of 0.25 nm the five-point ones leave 5e-16 of the
neighbours' weight).  FP32 storage relative to that composition shows it: the
stored values start at 0.

Tolerance: x - xe comes out below 2^-53, so the potentials are below 1e-4 J/m^3
(Hessians up to 1.1e11) and a step, whose coefficients dt D A_gamma m are below
1e-13, adds less than 1e-13 x 1e-15 x 1e-4 = 1e-32: 1e-30 in 64 steps.  The
Laplacian of the constant would have added 1e-20 a step.
"""
import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa.sim import Simulation

pytestmark = pytest.mark.gpu

XE = (0.52421634830562147, 0.01299272922003303)


@pytest.mark.parametrize("nine", [False, True])
@pytest.mark.parametrize("spl", [1, 2, 3, 4, None])
def test_equilibrium_stays(gpu, spl, nine):
    nx, ny = 70, 50
    s = M.make_setup(nx, ny, dx=0.25e-9, bc=1)
    if nine:
        s.mask = M.nine_point_mask(s.dx, s.dx)
    one = np.ones((ny + 2, nx + 2))
    sim = Simulation(s, [XE[0] * one, XE[1] * one, 0 * one, 0 * one], dtype=torch.float32,
                     steps_per_launch=spl, storage_offset=XE)
    sim.step(64)
    for k in range(4):
        assert float(sim.a[k].abs().max()) < 1e-30, k
    sim.close()


def test_unbalanced_mask_adds_its_constant(gpu):
    """Weights that do not add up to zero by more than rounding keep their
    Laplacian of a constant: x' = x + dt D xe (sum of the weights)."""
    nx, ny = 40, 30
    s = M.make_setup(nx, ny, dx=0.25e-9, bc=1)
    s.mask = list(s.mask)
    s.mask[4] *= 1 - 1e-9
    one = np.ones((ny + 2, nx + 2))
    sim = Simulation(s, [XE[0] * one, XE[1] * one, 0 * one, 0 * one], dtype=torch.float32,
                     storage_offset=XE)
    sim.step(1)
    total = sum(s.mask)
    for k, row in enumerate((s.DCr, s.DNb)):
        want = s.dt * (row[0] * XE[0] + row[1] * XE[1]) * total
        assert float(sim.a[k].reshape(-1)[0]) == pytest.approx(want, rel=1e-6)
    sim.close()
