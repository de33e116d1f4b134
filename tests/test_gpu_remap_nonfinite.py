"""The remap of tracers with an infinite cell: the same numbers, infinities and
NaNs in every cell as the oracle's, in columns in step (window within the ring)
and at their own pace, and finite columns untouched by their neighbours."""
import numpy as np
import pytest

import fv3atm_amd as fa
from fv3atm_amd import cases
from oracle import oracle
from tests._util import interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thin,kord", [(1, 9), (2, 10), (3, 9), (3, 17), (8, 8)])
def test_infinite_cells(gpu_ready, thin, kord):
    n, km, nq = 13, 40, 2
    case = cases.make_case(f"C{n}L{km}Q{nq}", n=n, npz=km, nq=nq, ntiles=1, delp_kind=1, delp_amp=(0.05, 0.1), seed=thin,
                           with_pt=True)
    rng = np.random.default_rng(thin)
    q = np.asfortranarray(case.q + rng.uniform(0.5, 1.0, case.q.shape))
    for at in range(0, 19 * 19, 3):
        q[at % 19, at // 19, rng.integers(0, km), at % nq] = np.inf if at % 2 else -np.inf
    # source layers thinner by `thin` in the upper half, thicker below: a target there takes in several
    dp1 = case.dp1.copy()
    up = dp1[:, :, :km // 2] / thin
    dp1[:, :, km // 2:] += ((dp1[:, :, :km // 2] - up).sum(axis=2) / (km - km // 2))[:, :, None]
    dp1[:, :, :km // 2] = up
    dp1 = np.asfortranarray(dp1)
    print(f"[remap nonfinite] thin {thin} kord {kord}", flush=True)
    ref = oracle.remap_tracers(case, q, dp1, case.pt, kord_tr=kord, kord_tm=10, fill=False)
    ctx = fa.Context(case.grids, km)
    got = [np.array(x, order="F") for x in (q, dp1, case.pt)]
    fa.lagrangian_to_eulerian_tracers(ctx, km, nq, case.ak, case.bk, case.ptop, got[1], got[0], got[2], kord, 10,
                                      184.0, False)
    ctx.close()
    a, b = interior(got[0]), interior(ref[0])
    assert not np.isfinite(b).all()
    for f in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(f(a), f(b), err_msg=f.__name__)
    ok = np.isfinite(b)
    np.testing.assert_allclose(a[ok], b[ok], rtol=1e-12, atol=0)
