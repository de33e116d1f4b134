"""The remap over shared column tables (mapz_fields.hip) against the FP64
oracle where its blocks, windows and dispatch have edges: the shortest column,
levels either side of a block of 8 and of the one-thread-per-column fallback
(km > 255), both layer-integral forms (nq 5 and 6), every kord, fillz, column
counts that do not fill a wave, six faces.  Both sides evaluate the same
expressions in the same order, so the tolerance is the parity bar of the FP64
forms (1e-12 per cell)."""
import numpy as np
import pytest

import fv3atm_amd as fa
from fv3atm_amd import cases
from oracle import oracle
from tests._util import assert_close, interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,km,nq,kord,fill,nt", [
    (8, 4, 1, 9, False, 1), (9, 5, 2, 10, False, 1), (9, 7, 5, 10, False, 1), (13, 8, 6, 9, True, 1),
    (11, 9, 7, 17, False, 1), (16, 16, 2, 10, True, 1), (10, 127, 3, 8, False, 1), (10, 128, 1, 9, False, 1),
    (8, 255, 1, 10, False, 1), (8, 256, 1, 9, False, 1), (12, 15, 2, 9, False, 6)])
def test_matches_oracle(gpu_ready, n, km, nq, kord, fill, nt):
    case = cases.make_case(f"{nt}xC{n}L{km}Q{nq}", n=n, npz=km, nq=nq, ntiles=nt, delp_kind=1, delp_amp=(0.05, 0.3),
                           seed=km, with_pt=True)
    rng = np.random.default_rng(km * 31 + n)
    # rough tracers with negative cells, so that every limiter and fillz act
    q = np.asfortranarray(case.q + rng.normal(0.0, 0.2, case.q.shape))
    print(f"[remap] {nt} x C{n} L{km} Q{nq} kord {kord} fill {fill}", flush=True)
    ref = oracle.remap_tracers(case, q, case.dp1, case.pt, kord_tr=kord, kord_tm=10, fill=fill)
    ctx = fa.Context(case.grids, km)
    got = [np.array(x, order="F") for x in (q, case.dp1, case.pt)]
    fa.lagrangian_to_eulerian_tracers(ctx, km, nq, case.ak, case.bk, case.ptop, got[1], got[0], got[2], kord, 10,
                                      184.0, fill)
    ctx.close()
    for a, b, what in zip(got, ref, ("q", "delp", "pt")):
        assert_close(interior(a), interior(b), 1e-12, what, floor=1e-300)
        np.testing.assert_array_equal(a[:3], b[:3])  # halos untouched
