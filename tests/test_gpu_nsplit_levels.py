"""Sub-cycle counts where one wave takes them over the levels (k_nsplit): level
counts either side of the wave, per level and as one count for all levels, the
largest Courant number planted on the first, the last and a middle level.  The
counts and every tracer equal the oracle's (bit for bit in FP64: 1e-12 per
cell)."""
import numpy as np
import pytest

import fv3atm_amd as fa
from fv3atm_amd import cases
from oracle import oracle
from tests._util import assert_close, interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npz,peak,per_level", [(1, 0, False), (63, 62, False), (64, 0, False), (65, 64, False),
                                                (65, 64, True), (129, 70, False), (130, 129, True)])
def test_counts(gpu_ready, npz, peak, per_level):
    case = cases.make_case(f"C8L{npz}", n=8, npz=npz, nq=1, courant=0.4, delp_kind=1, delp_amp=(0.05, 0.1), seed=npz)
    for f in ("cx", "cy", "mfx", "mfy"):
        a = getattr(case, f).copy()
        a[:, :, peak] *= 6.0
        setattr(case, f, np.asfortranarray(a))
    print(f"[nsplit] L{npz} peak {peak + 1} per_level {per_level}", flush=True)
    ref = oracle.tracer_2d(case, "1L" if per_level else "2d")
    ctx = fa.Context(case.grids, npz)
    a = {k: np.array(getattr(case, k), order="F", copy=True) for k in ("q", "dp1", "mfx", "mfy", "cx", "cy")}
    fn = fa.tracer_2d_1L if per_level else fa.tracer_2d
    ns = fn(ctx, a["q"], a["dp1"], a["mfx"], a["mfy"], a["cx"], a["cy"], 9, 9, npz, 1, case.hord)
    ctx.close()
    np.testing.assert_array_equal(ns, ref["nsplit"])
    assert ref["nsplit"].max() >= 2
    assert_close(interior(a["q"]), interior(ref["q"]), 1e-12, "q", floor=1e-300)
