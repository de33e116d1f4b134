"""dyn_core's sub-step kernel (dyncore.hip: strips of 58 columns, streamed rows)
against the stage kernels where its strips, row blocks and edge forms end: one
and two strips (a second one of 1 or 3 columns), row blocks of 4 and of more,
the smallest domain, six faces, a domain without cube edges, and the orders
that need more than the slopes.  The FP64 forms evaluate the same expressions
in the same order, so every element of every array is equal."""
import dataclasses

import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,n,npz,hord,bounded", [
    (1, 8, 1, 8, False), (6, 9, 2, 10, False), (1, 58, 3, 8, False), (1, 59, 2, 11, False), (6, 61, 2, 9, False),
    (1, 130, 40, 8, False), (1, 77, 5, 13, False), (1, 61, 3, 8, True), (1, 59, 2, 10, True)])
def test_rows_equal_stages(gpu_ready, nt, n, npz, hord, bounded):
    case = cases.make_case(f"{nt}xC{n}L{npz}", n=n, npz=npz, nq=1, ntiles=nt, courant=1.6, delp_kind=1,
                           delp_amp=(0.05, 0.2), seed=n)
    uc, vc = cases.c_grid_winds(case, 3)
    grids = [dataclasses.replace(g, bounded_domain=bounded) for g in case.grids]
    print(f"[dyn_core rows] {nt} x C{n} L{npz} hord {hord} bounded {bounded}", flush=True)
    out = []
    for form in (fa.FORM_PLAIN64, fa.FORM_FUSED64):
        ctx = fa.Context(grids, npz)
        dev = [torch.from_numpy(np.asarray(a, dtype=np.float64).ravel(order="F")).cuda() for a in (uc, vc, case.dp1)]
        d = dev[2].numel()
        sizes = (d, uc.size // 3, vc.size // 3, nt * npz * n * (n + 1), nt * npz * n * (n + 1))
        rest = [torch.zeros(s, dtype=torch.float64, device="cuda") for s in sizes]
        fa.dyn_core_fluxes(ctx, form, 3, case.dt / 3, hord, *dev, *rest)
        out.append([a.cpu().numpy() for a in (dev[2], *rest)])
        ctx.close()
    for a, b, k in zip(*out, ("delp", "dp1", "cx", "cy", "mfx", "mfy")):
        np.testing.assert_array_equal(a, b, err_msg=k)
