"""The step with the target thickness in the source's own array (delp_out = dp1):
the transport reads the source thickness in every sub-cycle, so the remap's
tables and the target wait for it.  Every output equals, element for element,
the call with arrays of its own."""
import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases

pytestmark = pytest.mark.gpu


def _dev(a, dtype):
    return torch.from_numpy(np.asarray(a, dtype=dtype).ravel(order="F")).cuda()


@pytest.mark.parametrize("form,nt,n,pipeline", [
    (fa.FORM_FUSED32, 1, 130, None), (fa.FORM_FUSED32, 1, 130, 2), (fa.FORM_FUSED32, 6, 24, None),
    (fa.FORM_FUSED64, 1, 130, None), (fa.FORM_FUSED64, 6, 24, None), (fa.FORM_PLAIN64, 1, 24, None),
    ("noalloc", 1, 60, None)])
def test_target_over_source(gpu_ready, form, nt, n, pipeline):
    npz, nq = 12, 5
    case = cases.make_case(f"{nt}xC{n}L12Q5", n=n, npz=npz, nq=nq, ntiles=nt, jet=True, courant=2.4, delp_kind=1,
                           delp_amp=(0.05, 0.2), seed=n, with_pt=True)
    w = np.float64 if form in (fa.FORM_FUSED64, fa.FORM_PLAIN64) else np.float32
    print(f"[same dp] form {form} {nt} x C{n} pipeline {pipeline}", flush=True)
    out = []
    for same in (False, True):
        ctx = fa.Context(case.grids, npz)
        if pipeline is not None:
            fa.set_pipeline(ctx, pipeline)
        q, pt = _dev(case.q, w), _dev(case.pt, w)
        wind = [_dev(getattr(case, k), w) for k in ("cx", "cy", "mfx", "mfy")]
        ab = [_dev(case.ak, np.float64), _dev(case.bk, np.float64)]
        q1, dp1 = torch.zeros_like(q), _dev(case.dp1, np.float64)
        delp = dp1 if same else torch.zeros_like(dp1)
        if form == "noalloc":
            fa.step_dev_noalloc(ctx, nq, q, q1, pt, dp1, delp, *wind, *ab, case.ptop, 8, 9, 10)
        else:
            fa.step_dev(ctx, form, nq, q, q1, pt, dp1, delp, *wind, *ab, case.ptop, 8, 9, 10)
        torch.cuda.synchronize()
        out.append([a.cpu().numpy() for a in (q1, delp, pt)])
        ctx.close()
    assert not np.array_equal(out[0][1], np.asarray(case.dp1).ravel(order="F"))
    for a, b, k in zip(*out, ("q", "delp", "pt")):
        np.testing.assert_array_equal(a, b, err_msg=k)
