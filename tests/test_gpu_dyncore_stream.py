"""dyn_core's sub-steps on a stream of the caller's, six faces: the halo refresh
between sub-steps runs in order with them.  Every array equals, element for
element, the call on the context's stream."""
import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [fa.FORM_PLAIN64, fa.FORM_FUSED64, fa.FORM_FUSED32])
def test_caller_stream(gpu_ready, form):
    n, npz, sub = 40, 20, 5
    case = cases.make_case("6xC40L20", n=n, npz=npz, nq=1, ntiles=6, courant=1.6, delp_kind=1, delp_amp=(0.05, 0.2),
                           seed=4)
    uc, vc = cases.c_grid_winds(case, sub)
    dt = np.float32 if form == fa.FORM_FUSED32 else np.float64
    ctx = fa.Context(case.grids, npz)
    side = torch.cuda.Stream()
    print(f"[dyn_core stream] 6 x C{n} L{npz} form {form}", flush=True)
    out = []
    for stream in (None, side.cuda_stream):
        dev = [torch.from_numpy(np.asarray(a, dtype=dt).ravel(order="F")).cuda() for a in (uc, vc, case.dp1)]
        sizes = (dev[2].numel(), uc.size // sub, vc.size // sub, 6 * npz * n * (n + 1), 6 * npz * n * (n + 1))
        rest = [torch.zeros(s, dtype=dev[0].dtype, device="cuda") for s in sizes]
        torch.cuda.synchronize()
        fa.dyn_core_fluxes(ctx, form, sub, case.dt / sub, 8, *dev, *rest, stream=stream)
        torch.cuda.synchronize()
        out.append([a.cpu().numpy() for a in (dev[2], *rest)])
    ctx.close()
    for a, b, k in zip(*out, ("delp", "dp1", "cx", "cy", "mfx", "mfy")):
        np.testing.assert_array_equal(a, b, err_msg=k)
