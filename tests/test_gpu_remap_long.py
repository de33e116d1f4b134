"""The FP32 column-shared remap at its largest column: 511 and 512 levels against
the FP64 oracle (relative L2 1e-5 per tracer, 1e-6 for pt, the bars of the FP32
step; the target thickness is FP64: 1e-12), and 513
refused."""
import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases
from tests._util import assert_close, interior, rel_l2
from tests.test_gpu_fused import reference, run_step

pytestmark = pytest.mark.gpu


def _case(npz):
    case = cases.make_case(f"C10L{npz}Q2", n=10, npz=npz, nq=2, courant=0.6, delp_kind=1, delp_amp=(0.05, 0.1),
                           seed=npz, with_pt=True)
    k = np.arange(npz) / npz
    x = np.arange(16)
    case.q = np.asfortranarray(2.0 + 0.3 * np.sin(9.0 * k)[:, None] * np.cos(0.4 * x)[:, None, None, None]
                               + 0.2 * np.sin(0.5 * x)[:, None, None] + 0.5 * np.arange(2))
    return case


@pytest.mark.parametrize("npz", [511, 512])
def test_step_matches_oracle(gpu_ready, npz):
    case = _case(npz)
    print(f"[remap long] C10 L{npz}", flush=True)
    ref = reference(case)
    got = run_step(case, fa.FORM_FUSED32)
    for iq in range(case.nq):
        assert rel_l2(interior(got["q"][..., iq]), interior(ref["q"][..., iq])) <= 1e-5, iq
    assert rel_l2(interior(got["pt"]), interior(ref["pt"])) <= 1e-6
    assert_close(interior(got["delp"]), interior(ref["delp"]), 1e-12, "delp")


def test_longer_is_refused(gpu_ready):
    with pytest.raises(RuntimeError, match="512"):
        run_step(_case(513), fa.FORM_FUSED32)
    torch.cuda.synchronize()
