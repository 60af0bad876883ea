"""The gradients of the energy sum are quotients, rounded once: with phi_delta
varying along one axis only, phi_Laves = 0 and kappa_delta = 1, the gradient map
is (a / (2 h))^2 dV, each operation rounded, so it is compared bit for bit with
numpy's.  Spacings whose reciprocals round up and down, a subnormal reciprocal
and one that overflows, and with values that are not finite or whose quotients
or squares are not."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wild", [False, True])
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("h", [2.5e-10, 3.1e-10, 0.7, 3.0, 5e-10 / 7, 8e307, 1e-309])
def test_gradient_map_is_a_rounded_quotient(gpu, h, axis, wild):
    Nx, Ny = 131, 77
    nx, ny = Nx + 2, Ny + 2
    rng = np.random.default_rng(5)
    line = rng.uniform(0, 1, ny if axis == 0 else nx)
    if wild:
        line[5], line[20], line[40], line[60], line[70:] = np.inf, np.nan, 1e160, 1e308, 1e-200
        line[71], line[73] = 3e-200, 1.1e-308
    phi = M.fill_ghosts(np.ascontiguousarray(np.broadcast_to(
        line[:, None] if axis == 0 else line[None, :], (ny, nx))), 1)
    f = [np.full((ny, nx), 0.3), np.full((ny, nx), 0.02), phi, np.zeros((ny, nx))]
    dev = [torch.as_tensor(np.ascontiguousarray(a)).cuda() for a in f]
    other = 1.0 / h if 1e-300 < h < 1e300 else 1.0        # dV = 1 or h
    d = (other, h) if axis == 0 else (h, other)           # (dx, dy)
    chem, grad = [torch.zeros((ny, nx), dtype=torch.float64, device="cuda") for _ in range(2)]
    out = torch.zeros(3, dtype=torch.float64, device="cuda")
    ctx = ctypes.c_void_p()
    check(lib().pf_ctx_create(ctypes.byref(ctx)), "pf_ctx_create")
    check(lib().pf_energy_f64(ctx, nx, ny, 1, d[0], d[1], (ctypes.c_double * 2)(1.0, 0.0),
                              (ctypes.c_double * 2)(0.0, 0.0), 0.0,
                              *[ctypes.c_void_p(t.data_ptr()) for t in dev],
                              ctypes.c_void_p(chem.data_ptr()), ctypes.c_void_p(grad.data_ptr()),
                              ctypes.c_void_p(out.data_ptr()), None), "pf_energy")
    got = grad.cpu().numpy()[1:-1, 1:-1]
    lib().pf_ctx_destroy(ctx)
    def difference(ax):
        return phi[2:, 1:-1] - phi[:-2, 1:-1] if ax == 0 else phi[1:-1, 2:] - phi[1:-1, :-2]

    with np.errstate(all="ignore"):
        g = difference(axis) / (2.0 * h)
        # along the other axis 0, or NaN where the line is not finite
        want = (g * g + difference(1 - axis)) * (d[0] * d[1])
    assert np.array_equal(got, want, equal_nan=True)
