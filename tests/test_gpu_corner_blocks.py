"""The fused transport on one cube face whose last row block or last strip of
columns is one or two wide, so that the block or strip before it reads corner
cells as well: n = 12 m + 1 or 2 for the row blocks (12 rows at these sizes),
n = 58 m + 1 or 2 for the strips, with and without interior strips.  Tracers are
smooth waves and the caller's corner halo holds a sentinel that copy_corners
never reads.  FP64 equals the oracle (1e-12 per cell), FP32 stays within a
relative L2 of 1e-5 per tracer, over the tile and over the 6 x 6 cells at each
corner; the adjoint, whose forward sweep is the fused transport, passes the
dot-product test against the staged tangent linear (1e-12)."""
import numpy as np
import pytest

import fv3atm_amd as fa
from fv3atm_amd import cases
from tests._util import assert_close, interior, rel_l2
from tests.test_gpu_fused import reference, run_step
from tests.test_gpu_tlad import Runner, dot, grf

pytestmark = pytest.mark.gpu
NG = 3


def _case(n, npz, nq, **kw):
    case = cases.make_case(f"C{n}L{npz}Q{nq}", n=n, npz=npz, nq=nq, delp_kind=1, delp_amp=(0.05, 0.15), seed=n, **kw)
    x, k, iq = np.arange(n + 2 * NG), np.arange(npz), np.arange(nq)
    case.q = np.asfortranarray(2.0 + np.sin(0.9 * x)[:, None, None, None] * np.cos(0.8 * x + 1.0)[:, None, None]
                               + 0.03 * k[:, None] + 0.5 * iq)
    low, high = slice(0, NG), slice(-NG, None)
    for a, b in ((low, low), (low, high), (high, low), (high, high)):
        case.q[a, b] = 1.0e6
    return case


@pytest.mark.parametrize("n,npz,rows", [(49, 6, 0), (50, 6, 0), (61, 6, 0), (74, 5, 0), (117, 4, 0), (118, 4, 0),
                                        (175, 4, 0), (176, 4, 0), (48, 4, 23), (40, 4, 13)])
def test_step(gpu_ready, n, npz, rows):
    case = _case(n, npz, 2, jet=True, courant=2.4)
    ref = reference(case)
    print(f"[corners] C{n} L{npz} rows {rows} nsplit", np.unique(ref["nsplit"]).tolist(), flush=True)
    got = run_step(case, fa.FORM_FUSED64, rows=rows, cfg=12 if rows else 0)
    assert_close(interior(got["q"]), interior(ref["q"]), 1e-12, "FP64 q", floor=1e-300)
    if npz < 8:
        case = _case(n, 8, 2, jet=True, courant=2.4)  # the FP32 remap needs 8 levels
        ref = reference(case)
    got = run_step(case, fa.FORM_FUSED32, rows=rows, cfg=12 if rows else 0)
    ends = np.r_[0:6, n - 6:n]
    for iq in range(case.nq):
        a, b = interior(got["q"][..., iq]), interior(ref["q"][..., iq])
        e = rel_l2(a, b), rel_l2(a[np.ix_(ends, ends)], b[np.ix_(ends, ends)])
        assert max(e) <= 1e-5, (iq, e)


@pytest.mark.parametrize("n", [49, 74, 117])
def test_adjoint(gpu_ready, n):
    case = _case(n, 6, 1, courant=0.9, q_split=2)
    print(f"[corners] adjoint C{n} L6", flush=True)
    r = Runner(case, False, 2, 9)
    dq, y = grf(case.q.shape, 1), grf(case.q.shape, 2)
    _, dq1, _ = r.tl(case.q, dq)
    qb = r.ad(case.q, y)
    r.ctx.close()
    lhs, rhs = dot(dq1, y), dot(dq, qb)
    assert abs(lhs - rhs) <= 1e-12 * abs(lhs), (lhs, rhs)
