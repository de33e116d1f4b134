"""Tangent linear and adjoint of states with NaN and infinite cells."""
import numpy as np
import pytest

from fv3atm_amd import cases
from tests._util import interior
from tests.test_gpu_tlad import Runner, grf

pytestmark = pytest.mark.gpu


def _case(seed):
    return cases.make_case("C40L12Q2", n=40, npz=12, nq=2, courant=1.5, q_split=2, delp_kind=1, delp_amp=(0.05, 0.2),
                           seed=seed)


@pytest.mark.parametrize("value", [np.nan, -np.inf])
def test_tangent_of_a_bad_thickness(gpu_ready, value):
    """A remapped value that is not finite has a NaN tangent (Dual's division)."""
    case = _case(3)
    rng = np.random.default_rng(3)
    for i, j, k in rng.integers((3, 3, 0), (43, 43, 12), (25, 3)):
        case.dp1[i, j, k] = value
    r = Runner(case, False, 2, 9)
    print(f"[tlad nonfinite] dp1 {value}", flush=True)
    q1, dq1, _ = r.tl(case.q, grf(case.q.shape, 1))
    r.ctx.close()
    bad = ~np.isfinite(interior(q1))
    assert bad.any()
    assert np.isnan(interior(dq1)[bad]).all()
