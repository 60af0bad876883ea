"""The four-step launch whose waves are all resident at once, share their SIMDs
fairly and take matrix and quiet rows apart: chunks of the shortest height that
does so, of the greatest (FP64) and beyond it (FP32), each with a short last
chunk, and one block of waves more and fewer than it takes, against one-step
launches bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import PfParams, check, lib

from test_gpu_matrix_rows import _phi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["quiet", "tails", "tiny", "nonfinite"])
@pytest.mark.parametrize("bc,shape,rows,dtype", [
    (0, (1100, 640), 12, torch.float64), (1, (1101, 619), 12, torch.float32),
    (1, (1100, 603), 12, torch.float64),             # 1020 waves
    (0, (1121, 1520), 31, torch.float64), (1, (1064, 2070), 38, torch.float32),
    (1, (2240, 611), 12, torch.float64),             # 2040 waves
    (0, (2240, 625), 12, torch.float64),             # 2120 waves
])
def test_fair_modes_match_one_step_launches(gpu, bc, shape, rows, dtype, kind):
    Nx, Ny = shape
    s = M.make_setup(Nx, Ny, bc=bc)
    rng = np.random.default_rng(7)
    xCr = rng.uniform(0.28, 0.33, (Ny + 2, Nx + 2))
    xNb = rng.uniform(0.02, 0.027, (Ny + 2, Nx + 2))
    if kind == "nonfinite":
        xCr[Ny // 2, Nx // 2], xNb[Ny - 20, 9] = np.nan, np.inf
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
    check(L.pf_ctx_set_tile4(ctx, rows, 0), "tile")
    ext = "f64" if dtype == torch.float64 else "f32"

    def run(name, a, *extra):
        out = [torch.full_like(x, 7.0) for x in a]
        ptrs = [ctypes.c_void_p(t.data_ptr()) for t in a + out]
        check(getattr(L, name + ext)(ctx, Nx + 2, Ny + 2, bc, ctypes.byref(P), *ptrs, *extra,
                                     None), name)
        return out

    want = got = [torch.as_tensor(f).to(device="cuda", dtype=dtype).reshape(-1) for f in fields]
    for _ in range(2):
        for _ in range(4):
            want = run("pf_step_", want, None)
        got = run("pf_step4_", got)
        for f in range(4):
            assert np.array_equal(got[f].cpu().numpy(), want[f].cpu().numpy(), equal_nan=True), f
    torch.cuda.synchronize()
    L.pf_ctx_destroy(ctx)
