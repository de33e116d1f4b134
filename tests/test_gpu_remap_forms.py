"""Paths of the remap in upstream order that its other tests do not take: columns of
one block displaced against each other by more layers than the ring of source cells
holds, for float fields, for the winds' and w's columns and for (value, tangent)
pairs; and columns longer than the tables' kernels take (one thread per column).
FP64 against the oracle (1e-12); the float full remap against itself: a column's
values do not depend on the columns beside it, so that they equal, bit for bit, those
of a call whose columns are all displaced the same way (in step); the tangent linear
by its values (1e-12) and the dot product with the adjoint (1e-12)."""
import numpy as np
import pytest
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases
from oracle import oracle
from tests._util import assert_close, interior
from tests.test_gpu_l2e import _interior, _run_gpu, _run_ref
from tests.test_gpu_tlad import Runner, _dev, dot, grf

pytestmark = pytest.mark.gpu


def _shift(case, shift, same=0):
    """Layers thinner above and thicker below in every second pair of columns along
    i, the reverse in the others (same = 1 or -1: in none, or in all): the middle
    interface moves by `shift` layers and the surface pressure stays."""
    km, dp = case.npz, case.dp1
    ps = case.ptop + dp.sum(axis=2)
    base = np.diff(case.ak) + np.diff(case.bk) * ps[:, :, None]
    up = np.arange(km) < km // 2
    down = base[:, :, up].sum(axis=2, keepdims=True) / base[:, :, ~up].sum(axis=2, keepdims=True)
    pair = np.where(np.arange(dp.shape[0]) // 2 % 2 == 0, 1.0, -1.0)
    sign = (np.full_like(pair, same) if same else pair)[:, None, None]
    case.dp1 = np.asfortranarray(base * (1.0 + sign * np.where(up, 1.0, -down) * shift / (km / 2)))
    assert (case.dp1 > 0).all()
    return case, pair


def _full_case(shift, same=0):
    case, pair = _shift(cases.make_case("C14L40Q2", n=14, npz=40, nq=2, delp_kind=1, delp_amp=(0.02, 0.05), seed=5,
                                        with_pt=True), shift, same)
    st = cases.l2e_state(case, 1)
    st["delp"] = np.asfortranarray(case.dp1)
    return case, st, pair


@pytest.mark.parametrize("shift", [0.4, 2.6, 7.5])
def test_full_remap(gpu_ready, shift):
    case, st, _ = _full_case(shift)
    print(f"[remap forms] full remap, shift {shift}", flush=True)
    ref, _ = _run_ref(case, st, False, 0.0)
    got, _, _ = _run_gpu(case, st, fa.FORM_PLAIN64, False, 0.0)
    for k in ("u", "v", "w", "delz", "pt", "q", "delp"):
        b = _interior(k, ref[k], case.n)
        assert np.abs(_interior(k, got[k], case.n) - b).max() <= 1e-12 * np.abs(b).max(), k


@pytest.mark.parametrize("shift", [2.6, 7.5])
def test_float_columns_alone(gpu_ready, shift):
    print(f"[remap forms] float full remap, shift {shift}", flush=True)
    out = {}
    for same in (0, 1, -1):
        case, st, pair = _full_case(shift, same)
        out[same], _, _ = _run_gpu(case, st, fa.FORM_FUSED32, False, 0.0)
    s = pair[3:-3]
    for k in ("u", "v", "w", "delz", "pt", "q", "delp"):
        a, p, m = (_interior(k, out[x][k], case.n) for x in (0, 1, -1))
        own = s if k != "v" else np.where(pair[2:-3] == pair[3:-2], pair[3:-2], 0.0)  # v: its two cells alike
        assert (own > 0).any() and (own < 0).any()
        np.testing.assert_array_equal(a[own > 0], p[own > 0], err_msg=k)
        np.testing.assert_array_equal(a[own < 0], m[own < 0], err_msg=k)


@pytest.mark.parametrize("shift", [2.6, 7.5])
def test_tangent_linear(gpu_ready, shift):
    case, _ = _shift(cases.make_case("C16L40Q2", n=16, npz=40, nq=2, courant=0.3, q_split=1, delp_kind=1,
                                     delp_amp=(0.02, 0.05), seed=6), shift)
    _check_tl(case, f"tangent linear, shift {shift}")


@pytest.mark.parametrize("npz", [160, 161])
def test_tangent_linear_long(gpu_ready, npz):
    _check_tl(cases.make_case(f"C10L{npz}Q1", n=10, npz=npz, nq=1, courant=0.5, q_split=1, delp_kind=1,
                              delp_amp=(0.05, 0.2), seed=npz), f"tangent linear, {npz} levels")


def _check_tl(case, what):
    print(f"[remap forms] {what}", flush=True)
    r = Runner(case, False, 1, 9)
    dq, y = grf(case.q.shape, 1), grf(case.q.shape, 2)
    q1, dq1, delp = r.tl(case.q, dq)
    qb = r.ad(case.q, y)
    r.ctx.close()
    adv = oracle.tracer_2d(case, "2d")
    ref, delp_ref, _ = oracle.remap_tracers(case, adv["q"], case.dp1, None, kord_tr=9)
    assert_close(interior(q1), interior(ref), 1e-12, "value", floor=1e-300)
    assert_close(interior(delp), interior(delp_ref), 1e-12, "delp")
    lhs, rhs = dot(dq1, y), dot(dq, qb)
    assert abs(lhs - rhs) <= 1e-12 * abs(lhs), (lhs, rhs)


@pytest.mark.parametrize("hydrostatic,nt", [(False, 1), (True, 1), (False, 6)])
def test_full_remap_long(gpu_ready, hydrostatic, nt):
    case = cases.make_case(f"{nt}xC8L256Q2", n=8, npz=256, nq=2, ntiles=nt, delp_kind=1, delp_amp=(0.05, 0.2), seed=3,
                           with_pt=True)
    st = cases.l2e_state(case, 1, hydrostatic=hydrostatic)
    print(f"[remap forms] full remap, 256 levels, hydrostatic {hydrostatic}, {nt} tile(s)", flush=True)
    got, _, _ = _run_gpu(case, st, fa.FORM_PLAIN64, hydrostatic, 0.0)
    ref, _ = _run_ref(case, st, hydrostatic, 0.0)
    for k in ("u", "v", "pt", "q", "delp", "pkz") + (() if hydrostatic else ("w", "delz")):
        a, b = _interior(k, got[k], case.n), _interior(k, ref[k], case.n)
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), k


@pytest.mark.parametrize("nt,n", [(1, 200), (6, 82)])
def test_tracers_in_parts(gpu_ready, nt, n):
    """More tracers than the in-place remap copies at a time (512 MB): each as in a
    call with fewer (six or more: the same integral form)."""
    km, nq, half = 127, 13, 7
    case = cases.make_case(f"{nt}xC{n}L{km}Q1", n=n, npz=km, nq=1, ntiles=nt, delp_kind=1, delp_amp=(0.05, 0.1), seed=n,
                           with_pt=True)
    print(f"[remap forms] {nt} x C{n} L{km}, {nq} tracers", flush=True)
    k = np.arange(km) / km
    q = np.stack([1.0 + 0.5 * np.sin((3.0 + m) * k) for m in range(nq)], axis=-1)  # (level, tracer)
    shape = case.dp1.shape[:3] + (nq,) + case.dp1.shape[3:]
    full = np.empty(shape, order="F")
    full[...] = q.reshape((1, 1, km, nq) + (1,) * (full.ndim - 4))
    assert full.nbytes > 512 << 20
    ctx = fa.Context(case.grids, km)

    def remap(part):
        a = [np.array(x, order="F") for x in (full[:, :, :, part], case.dp1, case.pt)]
        fa.lagrangian_to_eulerian_tracers(ctx, km, a[0].shape[3], case.ak, case.bk, case.ptop, a[1], a[0], a[2], 9, 10)
        return a

    whole, first, rest = remap(slice(0, nq)), remap(slice(0, half)), remap(slice(half - 1, nq))
    ctx.close()
    np.testing.assert_array_equal(whole[0][:, :, :, :half], first[0])
    np.testing.assert_array_equal(whole[0][:, :, :, half - 1:], rest[0])
    for a, b in zip(whole[1:], first[1:]):
        np.testing.assert_array_equal(a, b)
    assert not np.array_equal(whole[0][5, 5], full[5, 5])


def test_derivative_tracers_in_parts(gpu_ready):
    """More tracers than the tangent linear's field launch takes (64) and than the
    adjoint's remap holds scratch for (2 GB): each as in calls with fewer."""
    n, npz, nq = 150, 16, 72
    case = cases.make_case("C150L16Q1", n=n, npz=npz, nq=1, courant=0.4, q_split=1, delp_kind=1, delp_amp=(0.05, 0.1),
                           seed=2)
    assert 8 * n * n * (npz + 2) * 16 * nq > 2 << 30
    print(f"[remap forms] C{n} L{npz}, {nq} tracers, tangent linear and adjoint", flush=True)
    d = {k: _dev(getattr(case, k)) for k in ("dp1", "cx", "cy", "mfx", "mfy", "ak", "bk")}
    g = torch.Generator(device="cuda").manual_seed(1)
    shape = (nq, npz, n + 6, n + 6)
    q0 = 1.0 + torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)
    dq = torch.zeros_like(q0)
    dq[..., 3:-3, 3:-3] = torch.rand((nq, npz, n, n), generator=g, device="cuda", dtype=torch.float64)
    ctx = fa.Context(case.grids, npz)

    def pair(a, b):
        q, dd = q0[a:b].contiguous(), dq[a:b].contiguous()
        q1, dq1, qb = (torch.zeros_like(q) for _ in range(3))
        delp = torch.zeros_like(d["dp1"])
        tail = (d["cx"], d["cy"], d["mfx"], d["mfy"], d["ak"], d["bk"], case.ptop, 8, 9)
        fa.step_tl_dev(ctx, False, 1, b - a, q, dd, q1, dq1, d["dp1"], delp, *tail)
        fa.step_ad_dev(ctx, False, 1, b - a, q, dd, qb, d["dp1"], *tail)
        torch.cuda.synchronize()
        return q1, dq1, qb

    whole = pair(0, nq)
    for a, b in ((0, 10), (58, 70), (62, 72)):
        for x, y in zip(whole, pair(a, b)):
            assert torch.equal(x[a:b], y), (a, b)
    ctx.close()
