"""The remap's ring of source cells in LDS (mapz_fields.hip): columns of one
block are taken through the target layers in lockstep while one target's source
layers, over the block, fit in the ring, else lane by lane.  Neighbouring
columns are displaced by up to `shift` layers in opposite directions, either
side of the ring's length, and one column may have a layer of negative
thickness.  Both sides evaluate the same expressions in the same order: the
tolerance is the parity bar of the FP64 forms (1e-12 per cell)."""
import numpy as np
import pytest

import fv3atm_amd as fa
from fv3atm_amd import cases
from oracle import oracle
from tests._util import assert_close, interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift,kord,nq,inverted", [
    (0.0, 9, 2, False), (0.4, 10, 6, False), (0.9, 9, 6, False), (1.4, 10, 2, False), (1.9, 9, 3, False),
    (2.1, 17, 2, False), (2.6, 8, 2, False), (7.5, 10, 6, False), (0.4, 9, 6, True)])
def test_matches_oracle(gpu_ready, shift, kord, nq, inverted):
    n, km = 13, 40
    case = cases.make_case(f"C{n}L{km}Q{nq}", n=n, npz=km, nq=nq, ntiles=1, delp_kind=1, delp_amp=(0.0, 0.0), seed=5,
                           with_pt=True)
    rng = np.random.default_rng(int(10 * shift) + kord)
    q = np.asfortranarray(case.q + rng.normal(0.0, 0.2, case.q.shape))
    # layers thinner above and thicker below, or the reverse: the middle
    # interface moves by `shift` layers and the surface pressure stays
    ps = case.ptop + case.dp1.sum(axis=2, keepdims=True)
    base = np.diff(case.ak)[:, None] + np.diff(case.bk)[:, None] * ps.reshape(1, -1)
    half = np.where(np.arange(km) < km // 2, 1.0, -1.0)[:, None] * np.where(np.arange(km) < km // 2,
                                                                           1.0, base[:km // 2].sum(0).mean()
                                                                           / base[km // 2:].sum(0).mean())[:, None]
    sign = np.where(np.arange(base.shape[1]) % 2 == 0, 1.0, -1.0)[None]
    dp = base * (1.0 + sign * half * shift / (km / 2)) * (1.0 + 0.02 * rng.uniform(-1, 1, base.shape))
    dp1 = np.moveaxis(dp.reshape(km, *ps.shape[:2], *ps.shape[3:]), 0, 2)
    assert (dp1 > 0).all()
    if inverted:
        dp1[7, 7, 20] *= -0.1
    dp1 = np.asfortranarray(dp1)
    print(f"[remap] shift {shift} kord {kord} nq {nq} inverted {inverted}", flush=True)
    ref = oracle.remap_tracers(case, q, dp1, case.pt, kord_tr=kord, kord_tm=10, fill=False)
    ctx = fa.Context(case.grids, km)
    got = [np.array(x, order="F") for x in (q, dp1, case.pt)]
    fa.lagrangian_to_eulerian_tracers(ctx, km, nq, case.ak, case.bk, case.ptop, got[1], got[0], got[2], kord, 10,
                                      184.0, False)
    ctx.close()
    for a, b, what in zip(got, ref, ("q", "delp", "pt")):
        assert_close(interior(a), interior(b), 1e-12, what, floor=1e-300)
