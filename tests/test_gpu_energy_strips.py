"""The free-energy sum's strips and chunks at their edges (pf_energy_*): strips
of 62 columns against grids just below, at and above a multiple, chunks of one
row and of several with a short last one, and more strips than waves.  Per-cell
maps within 1e-12 of the largest value of the oracle's, as for small grids; the
totals within relative 1e-12 of the exact sum of the oracle's maps (every term
is positive, so a sum is as accurate as its terms)."""
import ctypes
import math

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import check, lib

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.mark.parametrize("shape,bc,dtype", [
    ((61, 5), 0, torch.float64), ((62, 7), 1, torch.float32), ((63, 6), 0, torch.float32),
    ((124, 9), 1, torch.float64), ((125, 1499), 0, torch.float64),
    ((63, 4099), 1, torch.float64), ((620, 3001), 0, torch.float32),
    ((683, 2750), 1, torch.float64), ((253960, 2), 1, torch.float64),
])
def test_energy_at_strip_and_chunk_edges(gpu, oracle, shape, bc, dtype):
    Nx, Ny = shape
    nx, ny = Nx + 2, Ny + 2
    rng = np.random.default_rng(31 * Nx + Ny)
    size = (ny, nx)
    f = [0.3 + 0.05 * rng.standard_normal(size), 0.05 + 0.02 * rng.standard_normal(size),
         np.clip(rng.uniform(-0.3, 1.3, size), 0, 1), np.clip(rng.uniform(-0.5, 1.0, size), 0, 1)]
    f[3] *= f[2] < 0.3
    dev = [torch.as_tensor(M.fill_ghosts(a, bc)).to(device="cuda", dtype=dtype) for a in f]
    host = [a.double().cpu().numpy() for a in dev]
    dx, dy = 2.5e-10, 3.1e-10
    kappa, omega, Omega = M.kappa(), M.omega(), M.OMEGA_3PHASE
    _, wchem, wgrad = oracle.energy(host, bc, dx, dy, kappa, omega, Omega, maps=True)
    wchem, wgrad = wchem[1:-1, 1:-1], wgrad[1:-1, 1:-1]

    maps = [torch.full(size, np.nan, dtype=torch.float64, device="cuda") for _ in range(2)]
    outs = [torch.full((3,), np.nan, dtype=torch.float64, device="cuda") for _ in range(2)]
    fn = lib().pf_energy_f64 if dtype == torch.float64 else lib().pf_energy_f32
    ctx = ctypes.c_void_p()
    check(lib().pf_ctx_create(ctypes.byref(ctx)), "pf_ctx_create")
    for out, m in zip(outs, (maps, [None, None])):
        check(fn(ctx, nx, ny, bc, dx, dy, (ctypes.c_double * 2)(*kappa),
                 (ctypes.c_double * 2)(*omega), Omega,
                 *[ctypes.c_void_p(t.data_ptr()) for t in dev],
                 *[ctypes.c_void_p(t.data_ptr()) if t is not None else None for t in m],
                 ctypes.c_void_p(out.data_ptr()), None), "pf_energy")
    torch.cuda.synchronize()
    lib().pf_ctx_destroy(ctx)

    for got, want in zip(maps, (wchem, wgrad)):
        got = got.cpu().numpy()
        assert np.abs(got[1:-1, 1:-1] - want).max() <= TOL * np.abs(want).max()
        for edge in (got[0], got[-1], got[:, 0], got[:, -1]):   # ghost ring untouched
            assert np.isnan(edge).all()
    chem, grad = math.fsum(wchem.ravel()), math.fsum(wgrad.ravel())
    for got, want in zip(outs[0].tolist(), (chem + grad, chem, grad)):
        assert got == pytest.approx(want, rel=TOL)
    assert torch.equal(outs[0], outs[1])   # the same bits without maps
