"""A step refused for its Courant numbers (no level has a sub-cycle count, every
one of them a NaN) leaves every output as it was, and the context runs the next
step as a new one does."""
import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases

pytestmark = pytest.mark.gpu


def _dev(a, dtype):
    return torch.from_numpy(np.asarray(a, dtype=dtype).ravel(order="F")).cuda()


@pytest.mark.parametrize("form,nt,n", [(fa.FORM_FUSED32, 1, 130), (fa.FORM_FUSED32, 6, 70), (fa.FORM_FUSED64, 1, 130),
                                       (fa.FORM_FUSED64, 6, 70)])
def test_outputs_untouched(gpu_ready, form, nt, n):
    npz, nq = 12, 3
    case = cases.make_case(f"{nt}xC{n}L12Q3", n=n, npz=npz, nq=nq, ntiles=nt, courant=0.8, delp_kind=1,
                           delp_amp=(0.05, 0.2), seed=n, with_pt=True)
    w = np.float64 if form == fa.FORM_FUSED64 else np.float32
    print(f"[refused] form {form} {nt} x C{n}", flush=True)
    q, ab = _dev(case.q, w), [_dev(case.ak, np.float64), _dev(case.bk, np.float64)]
    wind = [_dev(getattr(case, k), w) for k in ("cx", "cy", "mfx", "mfy")]
    dp1 = _dev(case.dp1, np.float64)

    def step(ctx, cx, cy, q1, pt, delp):
        fa.step_dev(ctx, form, nq, q, q1, pt, dp1, delp, cx, cy, *wind[2:], *ab, case.ptop, 8, 9, 10)
        torch.cuda.synchronize()

    bad = [torch.full_like(a, float("nan")) for a in wind[:2]]
    ctx, new = fa.Context(case.grids, npz), fa.Context(case.grids, npz)
    fa.set_transport(ctx, False, 0)
    out = [torch.full_like(q, 7.0), _dev(case.pt, w), torch.full_like(dp1, 5.0)]
    keep = [a.clone() for a in out]
    with pytest.raises(RuntimeError, match="nsplit < 1"):
        step(ctx, *bad, *out)
    torch.cuda.synchronize()
    for a, b, k in zip(out, keep, ("q", "pt", "delp")):
        assert torch.equal(a, b), k
    fa.set_transport(ctx, True, 0)
    step(ctx, *wind[:2], *out)
    step(new, *wind[:2], *keep)
    ctx.close()
    new.close()
    for a, b, k in zip(out, keep, ("q", "pt", "delp")):
        assert torch.equal(a, b), k


@pytest.mark.parametrize("form", [fa.FORM_FUSED32, fa.FORM_FUSED64])
@pytest.mark.parametrize("n", [20, 48, 62])
def test_refused_at_small_tiles(gpu_ready, form, n):
    """Tiles whose columns leave lanes of a wave without a cell."""
    npz = 9
    case = cases.make_case(f"C{n}L9Q1", n=n, npz=npz, nq=1, delp_kind=1, delp_amp=(0.05, 0.1), seed=n)
    w = np.float64 if form == fa.FORM_FUSED64 else np.float32
    print(f"[refused] form {form} C{n}", flush=True)
    q, dp1 = _dev(case.q, w), _dev(case.dp1, np.float64)
    wind = [_dev(getattr(case, k), w) for k in ("cx", "cy", "mfx", "mfy")]
    for a in wind[:2]:
        a.fill_(float("nan"))
    ctx = fa.Context(case.grids, npz)
    with pytest.raises(RuntimeError, match="nsplit < 1"):
        fa.step_dev(ctx, form, 1, q, torch.zeros_like(q), None, dp1, torch.zeros_like(dp1), *wind,
                    _dev(case.ak, np.float64), _dev(case.bk, np.float64), case.ptop, 8, 9, 10)
    ctx.close()
