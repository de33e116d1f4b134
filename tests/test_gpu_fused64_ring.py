"""The FP64 fused transport's LDS row ring on tiles large enough for every
kernel kind (interior strips with whole and partial row blocks, edge strips'
lean rows, corners), with a partial wave of tracers, several rounds of them and
several sub-cycles, one tile and six faces, against the FP64 oracle: the same
operations in the same order, so the parity bar of the FP64 forms (1e-12 per
cell)."""
import numpy as np
import pytest

import fv3atm_amd as fa
from fv3atm_amd import cases
from tests._util import assert_close, interior
from tests.test_gpu_fused import reference, run_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nq,nt,hord,rows", [(184, 5, 1, 8, 0), (184, 1, 1, 8, 17), (125, 2, 6, 8, 0), (184, 2, 1, 10, 0)])
def test_every_kind(gpu_ready, n, nq, nt, hord, rows):
    case = cases.make_case(f"{nt}xC{n}L6Q{nq}", n=n, npz=6, nq=nq, ntiles=nt, jet=True, courant=2.4, delp_kind=1,
                           delp_amp=(0.05, 0.15), seed=n + nq, with_pt=True)
    case.hord = hord
    ref = reference(case)
    print(f"[fused64] {nt} x C{n} Q{nq} hord {hord} rows {rows} nsplit", np.unique(ref["nsplit"]).tolist(), flush=True)
    got = run_step(case, fa.FORM_FUSED64, rows=rows, cfg=12 if rows else 0)
    for k in ("q", "delp", "pt"):
        assert_close(interior(got[k]), interior(ref[k]), 1e-12, k, floor=1e-300)
