"""Nine-point masks in the four-step march that takes matrix and quiet rows
apart: chunks just below, at and above the height from which it does, alone and
with FP32's fair shares of a SIMD (all waves resident at once), against one-step
launches bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import PfParams, check, lib

from test_gpu_matrix_rows import _phi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["quiet", "negative zero", "tails", "one particle", "tiny",
                                  "nonfinite", "large"])
@pytest.mark.parametrize("bc,shape,rows,dtype", [
    (0, (57, 150), 19, torch.float64), (1, (57, 150), 20, torch.float64),
    (0, (130, 167), 64, torch.float32), (1, (130, 167), 64, torch.float64),
    (0, (1100, 1061), 20, torch.float32),            # 1080 waves
])
def test_nine_point_modes_match_one_step_launches(gpu, bc, shape, rows, dtype, kind):
    Nx, Ny = shape
    s = M.make_setup(Nx, Ny, bc=bc)
    mask = M.nine_point_mask(s.dx, s.dx)
    rng = np.random.default_rng(13)
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
        P.mask[i] = mask[i]
    L = lib()
    ctx = ctypes.c_void_p()
    check(L.pf_ctx_create(ctypes.byref(ctx)), "pf_ctx_create")
    check(L.pf_ctx_set_tile4(ctx, rows, 0), "tile")
    ext = "f64" if dtype == torch.float64 else "f32"
    advance = getattr(L, "pf_advance_" + ext)
    in_b = ctypes.c_int()

    def run(a, steps, most):
        sets = [t.clone() for t in a], [torch.full_like(t, 7.0) for t in a]
        ptrs = [(ctypes.c_void_p * 4)(*[t.data_ptr() for t in x]) for x in sets]
        check(advance(ctx, Nx + 2, Ny + 2, bc, ctypes.byref(P), *ptrs, steps, most,
                      ctypes.byref(in_b), None), "pf_advance")
        return sets[in_b.value]

    start = [torch.as_tensor(f).to(device="cuda", dtype=dtype).reshape(-1) for f in fields]
    want, got = run(start, 8, 1), run(start, 8, 4)
    for f in range(4):
        assert np.array_equal(got[f].cpu().numpy(), want[f].cpu().numpy(), equal_nan=True), f
    torch.cuda.synchronize()
    L.pf_ctx_destroy(ctx)
