"""The multi-step march's treatment of matrix rows (|phi| below 2^-72 over a
wave's columns) and quiet rows (phi all +0): chunks of 32 rows or more take it.
Whatever the phase fields hold, a launch gives the bits of as many one-step
launches, which know no such rows."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import PfParams, check, lib

pytestmark = pytest.mark.gpu


def _phi(kind, Ny, Nx, rng):
    y, x = np.mgrid[0:Ny + 2, 0:Nx + 2]
    zero = np.zeros((Ny + 2, Nx + 2))
    if kind in ("quiet", "nonfinite", "large"):
        return zero, zero.copy()
    if kind == "negative zero":
        return -zero, zero.copy()
    r = np.hypot(y - Ny / 3, x - Nx / 2)
    if kind == "tails":                # an interface and its decay through every threshold
        return np.exp(-np.maximum(r - 6, 0) / 0.7), 0.5 * np.exp(-r / 0.4)
    if kind == "one particle":         # +0 all round
        return (r < 5).astype(float), zero
    # small values of both signs on either side of the threshold
    mag = 2.0 ** rng.uniform(-80, -52, zero.shape)
    return mag * rng.choice([-1.0, 1.0], zero.shape), np.where(y > Ny // 2, mag, 0.0)


@pytest.mark.parametrize("kind", ["quiet", "negative zero", "tails", "one particle", "tiny",
                                  "nonfinite", "large"])
@pytest.mark.parametrize("k,dtype", [(4, torch.float64), (4, torch.float32), (3, torch.float32)])
@pytest.mark.parametrize("bc,shape", [(0, (57, 150)), (1, (130, 67))])
def test_matrix_rows_match_one_step_launches(gpu, bc, shape, k, dtype, kind):
    Nx, Ny = shape
    s = M.make_setup(Nx, Ny, bc=bc)
    rng = np.random.default_rng(11)
    xCr = rng.uniform(0.28, 0.33, (Ny + 2, Nx + 2))
    xNb = rng.uniform(0.02, 0.027, (Ny + 2, Nx + 2))
    if kind == "nonfinite":
        xCr[Ny // 2, Nx // 2], xNb[Ny - 20, 9] = np.nan, np.inf
    if kind == "large":
        xCr[Ny // 2, Nx // 2], xNb[Ny - 20, 9] = 1e200, -9.0
    fields = [M.fill_ghosts(a, bc) for a in (xCr, xNb) + _phi(kind, Ny, Nx, rng)]
    P = PfParams()
    P.dt, P.alpha = s.dt, s.alpha
    for i in range(2):
        P.DCr[i], P.DNb[i] = s.DCr[i], s.DNb[i]
        P.kappa[i], P.omega[i], P.Lmob[i] = s.kappa[i], s.omega[i], s.Lmob[i]
    for i in range(9):
        P.mask[i] = s.mask[i]
    L = lib()
    ctx = ctypes.c_void_p()
    check(L.pf_ctx_create(ctypes.byref(ctx)), "pf_ctx_create")
    check(getattr(L, "pf_ctx_set_tile%d" % k)(ctx, 64, 0), "tile")
    ext = "f64" if dtype == torch.float64 else "f32"

    def run(name, a, *extra):
        out = [torch.full_like(x, 7.0) for x in a]
        ptrs = [ctypes.c_void_p(t.data_ptr()) for t in a + out]
        check(getattr(L, name + ext)(ctx, Nx + 2, Ny + 2, bc, ctypes.byref(P), *ptrs, *extra,
                                     None), name)
        return out

    want = got = [torch.as_tensor(f).to(device="cuda", dtype=dtype).reshape(-1) for f in fields]
    for _ in range(3):
        for _ in range(k):
            want = run("pf_step_", want, None)
        got = run("pf_step%d_" % k, got)
        for f in range(4):
            assert np.array_equal(got[f].cpu().numpy(), want[f].cpu().numpy(), equal_nan=True), f
    torch.cuda.synchronize()
    L.pf_ctx_destroy(ctx)
