"""The four-step kernel's tiles on small grids (sides 8, 12 and 16, one cell
per thread) against one-step launches: grids at the edges of a tile, of each
tile size's range and beyond it, where the march runs (the last two with all
of its waves resident and sharing their SIMDs fairly), both boundary modes and
storage types."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import PfParams, check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 4), (7, 5), (8, 16), (9, 17), (128, 128), (129, 128),
                                   (192, 191), (193, 192), (255, 256), (257, 256), (5, 2000),
                                   (1999, 6), (264, 263), (362, 355), (365, 367),
                                   (1021, 1543), (1400, 1100)])
@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_tiles_match_one_step_launches(gpu, dtype, bc, shape):
    Nx, Ny = shape
    s = M.make_setup(Nx, Ny, bc=bc, dt_rule=3e-7)
    rng = np.random.default_rng(Nx + 31 * Ny)
    shp = (Ny + 2, Nx + 2)
    pd = np.clip(rng.uniform(-0.3, 1.3, shp), 0, 1)
    f = [0.3 + 0.01 * rng.standard_normal(shp), 0.02 + 0.005 * rng.standard_normal(shp), pd,
         np.clip(rng.uniform(-0.5, 1.0, shp), 0, 1) * (pd < 0.3)]
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
    ext = "f64" if dtype == torch.float64 else "f32"

    def run(name, a, *extra):
        out = [torch.full_like(x, np.nan) for x in a]
        ptrs = [ctypes.c_void_p(t.data_ptr()) for t in a + out]
        check(getattr(L, name + ext)(ctx, Nx + 2, Ny + 2, bc, ctypes.byref(P), *ptrs, *extra,
                                     None), name)
        return out

    start = [torch.as_tensor(M.fill_ghosts(a, bc)).to(device="cuda", dtype=dtype) for a in f]
    want = start
    for _ in range(4):
        want = run("pf_step_", want, None)
    got = run("pf_step4_", start)
    for k in range(4):  # interior and ghost ring
        assert np.array_equal(got[k].cpu().numpy(), want[k].cpu().numpy()), k
    torch.cuda.synchronize()
    L.pf_ctx_destroy(ctx)
