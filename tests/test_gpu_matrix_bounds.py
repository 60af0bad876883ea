"""Step parameters for which matrix and quiet rows may not be taken apart: not
finite, or so large that four steps could raise a phase field past the bounds.
Launches of several steps give the bits of as many one-step launches with them
too, the NaN of a phase field included."""
import ctypes

import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa._lib import PfParams, check, lib

from test_gpu_matrix_rows import _phi

pytestmark = pytest.mark.gpu


def _change(P, what):
    if what == "NaN in DCr":
        P.DCr[1] = np.nan
    elif what == "NaN in DNb":
        P.DNb[0] = np.nan
    elif what == "infinite DNb":
        P.DNb[1] = np.inf
    elif what == "NaN kappa":
        P.kappa[0] = np.nan
    elif what == "NaN omega":
        P.omega[1] = np.nan
    elif what == "NaN mobility":
        P.Lmob[0] = np.nan
    elif what == "NaN alpha":
        P.alpha = np.nan
    elif what == "large kappa":         # kappa dt L sum |m| = 24
        P.kappa[0] = 24.0 / (P.dt * P.Lmob[0] * sum(abs(m) for m in P.mask))
    elif what == "large diffusivity":   # the potentials overflow within four steps
        P.DCr[0] = 1e60
    else:
        assert what == "large well"
        P.omega[0] = 20.0 / (P.dt * P.Lmob[0])


@pytest.mark.parametrize("what", ["NaN in DCr", "NaN in DNb", "infinite DNb", "NaN kappa",
                                  "NaN omega", "NaN mobility", "NaN alpha", "large kappa",
                                  "large diffusivity", "large well"])
@pytest.mark.parametrize("kind", ["quiet", "tiny"])
@pytest.mark.parametrize("k,dtype,nine", [(4, torch.float64, False), (4, torch.float32, False),
                                          (3, torch.float32, False), (4, torch.float64, True)])
def test_parameters_out_of_bounds_match_one_step_launches(gpu, k, dtype, nine, kind, what):
    Nx, Ny, bc = 130, 67, 1
    s = M.make_setup(Nx, Ny, bc=bc)
    rng = np.random.default_rng(17)
    size = (Ny + 2, Nx + 2)
    x = (rng.uniform(0.28, 0.33, size), rng.uniform(0.02, 0.027, size))
    fields = [M.fill_ghosts(a, bc) for a in x + _phi(kind, Ny, Nx, rng)]
    mask = M.nine_point_mask(s.dx, s.dx) if nine else s.mask
    P = PfParams()
    P.dt, P.alpha = s.dt, s.alpha
    for i in range(2):
        P.DCr[i], P.DNb[i] = s.DCr[i], s.DNb[i]
        P.kappa[i], P.omega[i], P.Lmob[i] = s.kappa[i], s.omega[i], s.Lmob[i]
    for i in range(9):
        P.mask[i] = mask[i]
    _change(P, what)
    L = lib()
    ctx = ctypes.c_void_p()
    check(L.pf_ctx_create(ctypes.byref(ctx)), "pf_ctx_create")
    check(getattr(L, "pf_ctx_set_tile%d" % k)(ctx, 64, 0), "tile")
    advance = L.pf_advance_f64 if dtype == torch.float64 else L.pf_advance_f32
    in_b = ctypes.c_int()

    def run(a, most):
        sets = [t.clone() for t in a], [torch.full_like(t, 7.0) for t in a]
        ptrs = [(ctypes.c_void_p * 4)(*[t.data_ptr() for t in x]) for x in sets]
        check(advance(ctx, Nx + 2, Ny + 2, bc, ctypes.byref(P), *ptrs, k, most,
                      ctypes.byref(in_b), None), "pf_advance")
        return sets[in_b.value]

    start = [torch.as_tensor(f).to(device="cuda", dtype=dtype).reshape(-1) for f in fields]
    want, got = run(start, 1), run(start, k)
    for f in range(4):
        assert np.array_equal(got[f].cpu().numpy(), want[f].cpu().numpy(), equal_nan=True), f
    torch.cuda.synchronize()
    L.pf_ctx_destroy(ctx)
