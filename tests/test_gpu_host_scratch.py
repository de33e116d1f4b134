"""Device memory of the FP64 host-array transport: without sub-cycles no second
copy of the tracers (beside the staged one in and out); with them, in a context
whose scratch grows in the middle of the call, results as in one that has it
already."""
import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases

pytestmark = pytest.mark.gpu


def _call(ctx, case):
    a = {k: np.array(getattr(case, k), order="F", copy=True) for k in ("q", "dp1", "mfx", "mfy", "cx", "cy")}
    n1 = case.n + 1
    ns = fa.tracer_2d_1L(ctx, a["q"], a["dp1"], a["mfx"], a["mfy"], a["cx"], a["cy"], n1, n1, case.npz, case.nq, 8)
    return a, ns


def test_no_second_copy(gpu_ready):
    case = cases.make_case("C90L40Q24", n=90, npz=40, nq=24, courant=0.5, delp_kind=1, delp_amp=(0.05, 0.1), seed=3)
    ctx = fa.Context(case.grids, case.npz)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    print("[host scratch] C90 L40 Q24", flush=True)
    _, ns = _call(ctx, case)
    used = free - torch.cuda.mem_get_info()[0]
    ctx.close()
    assert ns.max() == 1
    # staged: q in and out, dp1 and a double copy, four winds; scratch: two area fluxes
    assert used <= 2 * case.q.nbytes + 8 * 1.1 * case.dp1.nbytes + 16 * 2 ** 20, used / case.q.nbytes


def test_grown_in_the_call(gpu_ready):
    case = cases.make_case("C40L12Q5", n=40, npz=12, nq=5, jet=True, courant=2.4, delp_kind=1, delp_amp=(0.05, 0.1),
                           seed=4)
    print("[host scratch] C40 L12 Q5, sub-cycled", flush=True)
    new = fa.Context(case.grids, case.npz)
    one, ns = _call(new, case)
    two, _ = _call(new, case)
    new.close()
    assert ns.max() > 1
    for k in one:
        np.testing.assert_array_equal(one[k], two[k], err_msg=k)
