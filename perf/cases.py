"""What a program on this path has the framework do, as cases to time and compare.

A case names one kind of call and its sizes:
  step  the device-resident advection + remap step (step_dev), the call a dycore
        makes once per remap interval: FP32 and FP64 fused forms, one tile and
        six faces, per-level sub-cycling or a forced q_split, with and without pt;
  dyn   dyn_core's accumulation of the transport inputs (dyn_core_fluxes);
  l2e   the full Lagrangian_to_Eulerian (lagrangian_to_eulerian_dev), hydrostatic
        and not, with the energy fix-up;
  tlad  the tangent-linear step and its adjoint (step_tl_dev, step_ad_dev), the
        two directions a variational program calls in turn;
  host  the Fortran-style calls on host arrays (tracer_2d_1L, then
        lagrangian_to_eulerian_tracers), copies in and out included.
Arrays the calls update in place are refilled from kept copies inside run(), as
the dynamics refills them in a model.  exact() restates the arithmetic in plain
64-bit torch.
"""
import functools
import math

import numpy as np
import torch

import fv3atm_amd as fa
from fv3atm_amd import cases as fc

NG = 3
F64 = torch.float64
KAPPA, CP, RD, GRAV = fc.KAPPA, fc.CP_AIR, fc.RDGAS, fc.GRAV
PS, PTOP = fc.PS, fc.PTOP


def listed():
    step = dict(kind="step", prec=32, tiles=1, pt=True, split=0, courant=0.9, jet=False)
    return [
        # the smallest call: one coarse tile, one tracer (launches and latency)
        dict(step, name="step32_c48", n=48, npz=32, nq=1, courant=0.4, pt=False),
        # a ragged nested-grid size, few whole strips or blocks, jet sub-cycling
        dict(step, name="step32_c203_odd", n=203, npz=75, nq=11, jet=True, courant=1.9),
        # deformational workload size with a forced q_split of 2 (tracer_2d's rule)
        dict(step, name="step32_c384_split", n=384, npz=64, nq=10, split=2, courant=0.8, pt=False),
        # the global sphere on one device, halos from the neighbouring faces
        dict(step, name="step32_6xc192", n=192, npz=127, nq=8, tiles=6),
        # the production tile: jet winds, per-level sub-cycles, 30 tracers and pt
        dict(step, name="step32_c768", n=768, npz=127, nq=30, jet=True, courant=2.5),
        # the dycore's 64-bit build: a coarse tile and a large one
        dict(step, name="step64_c96", n=96, npz=64, nq=4, prec=64),
        dict(step, name="step64_c384", n=384, npz=127, nq=9, prec=64, jet=True, courant=1.9),
        # the acoustic loop's accumulation, six sub-steps of a C384 tile
        dict(kind="dyn", name="dyn32_c384", n=384, npz=127, sub=6, prec=32, tiles=1),
        # full remap: the non-hydrostatic FP32 state, and a ragged hydrostatic FP64 one
        dict(kind="l2e", name="l2e32_c192", n=192, npz=127, nq=9, prec=32, tiles=1, hydro=False, consv=0.0),
        dict(kind="l2e", name="l2e64_c90_hydro", n=90, npz=63, nq=5, prec=64, tiles=1, hydro=True, consv=1.0),
        # sensitivity work: tangent linear and adjoint with six forced sub-cycles
        dict(kind="tlad", name="tlad_c192", n=192, npz=64, nq=4, split=6, tiles=1),
        # drop-in use from Fortran: host arrays through the library and back
        dict(kind="host", name="host_c96", n=96, npz=64, nq=7),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "step", "step", "step", "dyn", "l2e", "tlad", "host"])
    npz = rng.choice([rng.randint(20, 63), 63, rng.randint(64, 127), 91, 127])
    if kind == "step":
        prec = rng.choice([32, 32, 64])
        tiles = rng.choice([1, 1, 6])
        n = size(32, 150) if tiles == 6 else size(48, 500 if prec == 32 else 300)
        split = rng.choice([0, 0, 2])
        jet = rng.random() < 0.5 and not split
        return dict(kind=kind, n=n, npz=npz, nq=size(1, 24 if prec == 32 else 9), prec=prec, tiles=tiles,
                    pt=rng.random() < 0.5, split=split, jet=jet,
                    courant=round(rng.uniform(1.2, 2.5) if jet else rng.uniform(0.3, 0.95), 2))
    if kind == "dyn":
        return dict(kind=kind, n=size(48, 300), npz=npz, sub=rng.randint(2, 6), prec=rng.choice([32, 64]), tiles=1)
    if kind == "l2e":
        hydro = rng.random() < 0.5
        return dict(kind=kind, n=size(32, 160), npz=npz, nq=rng.randint(1, 9), prec=rng.choice([32, 64]), tiles=1,
                    hydro=hydro, consv=1.0 if hydro else 0.0)
    if kind == "tlad":
        return dict(kind=kind, n=size(32, 150), npz=min(npz, 64), nq=rng.randint(1, 4), split=rng.randint(1, 4), tiles=1)
    return dict(kind=kind, n=size(32, 110), npz=npz, nq=rng.randint(1, 8))


# ---- inputs -------------------------------------------------------------------
@functools.lru_cache(maxsize=16)
def _grid(n, tile):
    return fc.make_grid(n, tile)


@functools.lru_cache(maxsize=2)
def _context(n, npz, tiles, split):
    grids = [_grid(n, t) for t in range(1, tiles + 1)]
    da = fc.sphere_da_min(grids)
    for g in grids:
        g.da_min = da
    ctx = fa.Context(grids, npz)
    fa.set_transport(ctx, split == 0, split)
    return ctx


@functools.lru_cache(maxsize=2)
def _metrics(n, tiles):
    """FP64 device copies of the grid metrics, (tile, j, i) layouts."""
    m = {}
    for k in ("area", "rarea", "dx", "dy", "dxa", "dya", "sin_sg", "xyz_n", "xyz_c"):
        a = np.stack([np.ascontiguousarray(getattr(_grid(n, t), k).T) for t in range(1, tiles + 1)])
        m[k] = torch.from_numpy(a).cuda()
    m["sin_sg"] = m["sin_sg"].transpose(0, 1)  # (9, tile, j, i)
    return m


class _Rand:
    def __init__(self, seed):
        self.cpu = np.random.default_rng(seed)
        self.gpu = torch.Generator(device="cuda").manual_seed(int(seed))

    def uniform(self, lo, hi, *shape):
        return self.cpu.uniform(lo, hi, shape or None)

    def noise(self, *shape):  # in [-1, 1), FP64 on the device
        return torch.rand(*shape, device="cuda", dtype=F64, generator=self.gpu) * 2 - 1

    def waves(self, xyz, count=5, top=4.0):
        """A smooth function of position on the sphere, about unit size; xyz (tile, j, i, 3)."""
        out = 0
        for _ in range(count):
            k = torch.tensor(self.uniform(-top, top, 3), device="cuda", dtype=F64)
            out = out + float(self.uniform(0.4, 1.0)) * torch.sin(xyz @ k + float(self.uniform(0, 6.28)))
        return out / count ** 0.5


def _levels(npz, jet):
    if not jet:
        return torch.ones(npz, device="cuda", dtype=F64)
    z = fc.std_height(PTOP + (np.arange(npz) + 0.5) * (PS - PTOP) / npz)
    s = 10.0 + 60.0 * np.exp(-((z - 10.0e3) / 3.0e3) ** 2)
    return torch.from_numpy(s / s.max()).cuda()


def _winds(c, r, m, courant, speed):
    """Courant numbers and mass fluxes of a stream-function flow (with a small
    divergence), scaled so that the largest Courant number is `courant`."""
    n, npz = c["n"], len(speed)
    psi = r.waves(m["xyz_n"])                                   # corners (tile, nd+1, nd+1)
    sl = slice(NG, NG + n + 1)
    ax = (psi[:, 1:, :] - psi[:, :-1, :])[:, :, sl]             # area flux through x-faces, all rows
    ay = -(psi[:, :, 1:] - psi[:, :, :-1])[:, sl, :]            # through y-faces, all columns
    dxm, dxp = m["dxa"][:, :, NG - 1:NG + n], m["dxa"][:, :, NG:NG + n + 1]
    dym, dyp = m["dya"][:, NG - 1:NG + n, :], m["dya"][:, NG:NG + n + 1, :]
    s = m["sin_sg"]
    mx = m["dy"][:, :, sl] * torch.where(ax > 0, dxm * s[2][:, :, NG - 1:NG + n], dxp * s[0][:, :, NG:NG + n + 1])
    my = m["dx"][:, sl, :] * torch.where(ay > 0, dym * s[3][:, NG - 1:NG + n, :], dyp * s[1][:, NG:NG + n + 1, :])
    cx, cy = ax / mx, ay / my
    f = courant / max(float(cx[:, NG:-NG].abs().max()), float(cy[:, :, NG:-NG].abs().max()))
    lev = speed.view(1, npz, 1, 1) * f
    dpr = (PS - PTOP) / npz
    sx = 1 + 0.02 * r.waves(m["xyz_c"])                         # thickness the fluxes carry
    fx = (0.5 * (sx[:, :, 1:] + sx[:, :, :-1]))[:, NG:-NG, NG - 1:NG + n]
    fy = (0.5 * (sx[:, 1:, :] + sx[:, :-1, :]))[:, NG - 1:NG + n, NG:-NG]
    mfx = (ax[:, NG:-NG, :] * fx * dpr)[:, None] * lev
    mfy = (ay[:, :, NG:-NG] * fy * dpr)[:, None] * lev
    return cx[:, None] * lev, cy[:, None] * lev, mfx, mfy


def _thickness(r, m, npz):
    t, nd = m["area"].shape[0], m["area"].shape[1]
    k = torch.arange(npz, device="cuda", dtype=F64).view(1, npz, 1, 1) / npz
    w = 0.05 * (r.waves(m["xyz_c"])[:, None] * torch.cos(6.0 * k) + r.waves(m["xyz_c"])[:, None] * torch.sin(4.0 * k))
    return (PS - PTOP) / npz * (1 + w + 0.1 * r.noise(t, npz, nd, nd))


def _tracers(r, m, npz, nq, dtype):
    """Bells on a small background, discs of constant values and smooth waves,
    varied over the levels; (tile, nq, npz, j, i)."""
    xyz = m["xyz_c"]
    t, nd = xyz.shape[0], xyz.shape[1]
    q = torch.empty(t, nq, npz, nd, nd, device="cuda", dtype=dtype)
    lev = 1 + 0.5 * torch.arange(npz, device="cuda", dtype=F64) / npz
    for iq in range(nq):
        c = xyz[0, nd // 2, nd // 2] + torch.tensor(r.uniform(-0.3, 0.3, 3), device="cuda")
        d = (xyz - c / c.norm()).norm(dim=-1)
        if iq % 3 == 0:
            b = 1e-6 + torch.where(d < 0.5, 0.5 * (1 + torch.cos(math.pi * d / 0.5)), torch.zeros_like(d))
        elif iq % 3 == 1:
            b = 0.1 + 0.9 * (d < 0.45).double()
        else:
            b = 1.5 + 0.7 * r.waves(xyz, top=10.0)
        a, ph = float(r.uniform(0.05, 0.2)), float(r.uniform(0, 6.28))
        v = lev * (1 + a * torch.sin(ph + 9.0 * torch.arange(npz, device="cuda", dtype=F64) / npz))
        for k0 in range(0, npz, 32):
            q[:, iq, k0:k0 + 32] = (b[:, None] * v[k0:k0 + 32].view(1, -1, 1, 1)).to(dtype)
    return q


def _mid_pressure(dp):
    return PTOP + torch.cumsum(dp, 1) - 0.5 * dp


def prepare(case, seed):
    c = dict(case)
    kind, n, npz = c["kind"], c["n"], c["npz"]
    tiles = c.get("tiles", 1)
    r = _Rand(seed)
    m = _metrics(n, tiles)
    s = {"case": c, "ctx": _context(n, npz, tiles, c.get("split", 0) if kind == "step" else 0)}
    ak, bk = fc.hybrid_coefs(npz)
    s["ak"], s["bk"] = torch.from_numpy(ak).cuda(), torch.from_numpy(bk).cuda()
    s["akh"], s["bkh"] = ak, bk
    w = torch.float32 if c.get("prec", 64) == 32 else F64
    nd = n + 2 * NG
    if kind in ("step", "tlad", "host"):
        cour = {"tlad": 0.9 * c.get("split", 1), "host": 0.85}.get(kind, c.get("courant"))
        win = _winds(c, r, m, cour, _levels(npz, c.get("jet", False)))
        s["cx"], s["cy"], s["mfx"], s["mfy"] = (x.to(w).contiguous() for x in win)
        s["dp1"] = _thickness(r, m, npz)
        s["q0"] = _tracers(r, m, npz, c["nq"], w)
    if kind == "step":
        s["q1"], s["delp"] = torch.zeros_like(s["q0"]), torch.zeros_like(s["dp1"])
        if c["pt"]:
            s["pt0"] = (184.0 + 116.0 * (_mid_pressure(s["dp1"]) / PS) ** 0.19).to(w)
            s["pt"] = s["pt0"].clone()
    elif kind == "dyn":
        per = [_winds(c, r, m, 0.3, _levels(npz, True) * float(r.uniform(0.7, 1.0))) for _ in range(c["sub"])]
        dl, dr = m["dxa"][:, None, :, NG - 1:NG + n], m["dxa"][:, None, :, NG:NG + n + 1]
        bl, br = m["dya"][:, None, NG - 1:NG + n, :], m["dya"][:, None, NG:NG + n + 1, :]
        s["bdt"] = 100.0
        s["uc"] = torch.stack([(p[0] * torch.where(p[0] > 0, dl, dr) / s["bdt"]).to(w) for p in per])
        s["vc"] = torch.stack([(p[1] * torch.where(p[1] > 0, bl, br) / s["bdt"]).to(w) for p in per])
        s["delp0"] = _thickness(r, m, npz).to(w)
        s["delp"] = s["delp0"].clone()
        s["dp1"] = torch.zeros_like(s["delp"])
        s["cx"], s["cy"] = torch.zeros_like(s["uc"][0]), torch.zeros_like(s["vc"][0])
        z = functools.partial(torch.zeros, device="cuda", dtype=w)
        s["mfx"], s["mfy"] = z(tiles, npz, n, n + 1), z(tiles, npz, n + 1, n)
    elif kind == "l2e":
        dp = _thickness(r, m, npz)
        lev = torch.arange(npz, device="cuda", dtype=F64).view(1, npz, 1, 1) / (npz - 1)
        X = m["xyz_n"]
        wave = lambda x: r.waves(x)[:, None]  # noqa: E731
        su = 10.0 + 30.0 * torch.sin(math.pi * lev)
        st = {"delp": dp, "q": _tracers(r, m, npz, c["nq"], w)}
        st["u"] = wave(0.5 * (X[:, :, 1:] + X[:, :, :-1])) * su + 0.5 * r.noise(tiles, npz, nd + 1, nd)
        st["v"] = wave(0.5 * (X[:, 1:] + X[:, :-1])) * su + 0.5 * r.noise(tiles, npz, nd, nd + 1)
        st["pt"] = 184.0 + 116.0 * (_mid_pressure(dp) / PS) ** KAPPA
        i = slice(NG, NG + n)
        pe = torch.cat([torch.full_like(dp[:, :1], PTOP), PTOP + torch.cumsum(dp, 1)], 1)[:, :, i, i]
        dlp = torch.log(pe).diff(dim=1)
        st["pkz"] = torch.exp(KAPPA * torch.log(pe)).diff(dim=1) / (KAPPA * dlp)
        if not c["hydro"]:
            st["w"] = wave(m["xyz_c"]) * (0.2 + torch.sin(math.pi * lev)) + 0.05 * r.noise(tiles, npz, nd, nd)
            st["ws"] = 0.05 * r.waves(m["xyz_c"])[:, i, i]
            st["delz"] = -RD / GRAV * st["pt"][:, :, i, i] * st["pkz"] * dlp
        st = {k: v.to(F64 if k in ("delp", "pkz") else w).contiguous() for k, v in st.items()}
        z = functools.partial(torch.zeros, device="cuda", dtype=F64)
        out = dict(pe=z(tiles, n + 2, npz + 1, n + 2), peln=z(tiles, n, npz + 1, n), pk=z(tiles, npz + 1, n, n),
                   ps=z(tiles, nd, nd), te0_2d=z(tiles, n, n))
        s["keep"] = st
        s["state"] = {**{k: v.clone() for k, v in st.items()}, **out}
    elif kind == "tlad":
        s["ctx"] = _context(n, npz, tiles, 0)
        inner = torch.zeros_like(s["q0"])
        inner[..., NG:-NG, NG:-NG] = 1
        s["dq0"], s["qbar1"] = (r.noise(*s["q0"].shape) * inner for _ in range(2))
        for k in ("q1", "dq1", "qbar0"):
            s[k] = torch.zeros_like(s["q0"])
        s["delp"] = torch.zeros_like(s["dp1"])
    elif kind == "host":
        s["pt"] = 184.0 + 116.0 * (_mid_pressure(s["dp1"]) / PS) ** 0.19
        host = {}
        for k in ("q0", "dp1", "pt", "cx", "cy", "mfx", "mfy"):
            host[k] = np.asfortranarray(s.pop(k)[0].cpu().numpy().T)
        s["host"] = host
        s["work"] = {k: host[k].copy(order="F") for k in host}
        s["work"]["delp"] = host["dp1"].copy(order="F")
    return s


# ---- one pass -----------------------------------------------------------------
def run(s):
    c, ctx = s["case"], s["ctx"]
    kind, npz = c["kind"], c["npz"]
    if kind == "step":
        pt = s.get("pt")
        if pt is not None:
            pt.copy_(s["pt0"])
        fa.step_dev(ctx, fa.FORM_FUSED32 if c["prec"] == 32 else fa.FORM_FUSED64, c["nq"], s["q0"], s["q1"], pt,
                    s["dp1"], s["delp"], s["cx"], s["cy"], s["mfx"], s["mfy"], s["ak"], s["bk"], PTOP, 8, 9, 10)
        return {"q": s["q1"], "delp": s["delp"], **({} if pt is None else {"pt": pt})}
    if kind == "dyn":
        s["delp"].copy_(s["delp0"])
        fa.dyn_core_fluxes(ctx, fa.FORM_FUSED32 if c["prec"] == 32 else fa.FORM_FUSED64, c["sub"], s["bdt"], 8,
                           s["uc"], s["vc"], s["delp"], s["dp1"], s["cx"], s["cy"], s["mfx"], s["mfy"])
        return {k: s[k] for k in ("delp", "dp1", "cx", "cy", "mfx", "mfy")}
    if kind == "l2e":
        st = s["state"]
        for k, v in s["keep"].items():
            st[k].copy_(v)
        fa.lagrangian_to_eulerian_dev(ctx, fa.FORM_FUSED32 if c["prec"] == 32 else fa.FORM_PLAIN64, npz, c["nq"],
                                      s["ak"], s["bk"], PTOP, st, kord_tr=9, kord_tm=10, kord_mt=9, kord_wz=9,
                                      hydrostatic=c["hydro"], consv=c["consv"], akap=KAPPA, cp=CP, rdgas=RD,
                                      grav=GRAV)
        return dict(st)
    if kind == "tlad":
        tail = (s["dp1"],), (s["cx"], s["cy"], s["mfx"], s["mfy"], s["ak"], s["bk"], PTOP, 8, 9)
        fa.step_tl_dev(ctx, False, c["split"], c["nq"], s["q0"], s["dq0"], s["q1"], s["dq1"], *tail[0], s["delp"],
                       *tail[1])
        fa.step_ad_dev(ctx, False, c["split"], c["nq"], s["q0"], s["qbar1"], s["qbar0"], *tail[0], *tail[1])
        return {k: s[k] for k in ("q1", "dq1", "delp", "qbar0")}
    h, w = s["host"], s["work"]
    for k in ("q0", "dp1", "pt", "cx", "cy", "mfx", "mfy"):
        np.copyto(w[k], h[k])
    np.copyto(w["delp"], h["dp1"])
    n1 = c["n"] + 1
    nsplit = fa.tracer_2d_1L(ctx, w["q0"], w["dp1"], w["mfx"], w["mfy"], w["cx"], w["cy"], n1, n1, npz, c["nq"], 8)
    fa.lagrangian_to_eulerian_tracers(ctx, npz, c["nq"], s["akh"], s["bkh"], PTOP, w["delp"], w["q0"], w["pt"], 9, 10)
    return {**w, "nsplit": nsplit}


def work(case):
    """Each input read and each output written once; about 110 operations per
    cell, tracer and sub-cycle of the transport and 100 per remapped value."""
    c = dict(case)
    kind, n, npz = c["kind"], c["n"], c["npz"]
    w = c.get("prec", 64) // 8
    cells = c.get("tiles", 1) * n * n * npz
    if kind == "step":
        sp = _levels_split(c)
        f = c["nq"] + (1 if c["pt"] else 0)
        return {"bytes": cells * (2 * w * f + 16 + 4 * w), "flops": cells * (110 * c["nq"] * sp + 100 * f)}
    if kind == "dyn":
        return {"bytes": cells * w * (2 * c["sub"] + 7), "flops": cells * 110 * c["sub"]}
    if kind == "l2e":
        f = c["nq"] + 3 + (0 if c["hydro"] else 2)
        return {"bytes": cells * (2 * w * f + 8 * 7), "flops": cells * (100 * f + 60)}
    if kind == "tlad":
        return {"bytes": cells * (8 * 7 * c["nq"] + 2 * 40 + 8), "flops": cells * c["nq"] * (600 * c["split"] + 600)}
    return {"bytes": cells * 8 * (4 * c["nq"] + 12), "flops": cells * (110 * c["nq"] + 100 * (c["nq"] + 1))}


def _levels_split(c):
    if c["split"]:
        return c["split"]
    if not c["jet"]:
        return 1 + (c["courant"] >= 0.95)
    z = fc.std_height(PTOP + (np.arange(c["npz"]) + 0.5) * (PS - PTOP) / c["npz"])
    s = 10.0 + 60.0 * np.exp(-((z - 10.0e3) / 3.0e3) ** 2)
    return float(np.mean(np.floor(1 + c["courant"] * s / s.max())))


# ---- the same in plain 64-bit torch -------------------------------------------
def _sign(a, b):
    return torch.where(b < 0, -a, a)


def _pert(al, ar):
    d, s = al - ar, 3 * (al + ar)
    a6, d2 = s * d, d * d
    ext = al * ar < 0
    nr = torch.where(a6 < -d2, -2 * al, ar)
    nl = torch.where((a6 > d2) & ~(a6 < -d2), -2 * ar, al)
    z = torch.zeros_like(al)
    return torch.where(ext, nl, z), torch.where(ext, nr, z)


def _ppm(q, c, d):
    """Upwind PPM face values (order 8) along the last axis: q and the widths d
    with three halo cells on each side, c at the n + 1 faces."""
    n = c.shape[-1] - 1
    qm, q0, qp = q[..., :-2], q[..., 1:-1], q[..., 2:]
    xt = 0.25 * (qp - qm)
    hi, lo = torch.maximum(torch.maximum(qm, q0), qp), torch.minimum(torch.minimum(qm, q0), qp)
    dm = _sign(torch.minimum(torch.minimum(xt.abs(), hi - q0), q0 - lo), xt)  # cells -1 .. n+2
    al = 0.5 * (q[..., 1:-2] + q[..., 2:-1]) + (dm[..., :-1] - dm[..., 1:]) / 3  # faces 0 .. n+2
    qc, t = q[..., 2:-2], 2 * dm[..., 1:-1]  # cells 0 .. n+1
    bl = -_sign(torch.minimum(t.abs(), (al[..., :-1] - qc).abs()), t)
    br = _sign(torch.minimum(t.abs(), (al[..., 1:] - qc).abs()), t)
    s11, s14, s15 = 11 / 14, 4 / 7, 3 / 14
    for mirror in (False, True):  # the three cells either end, seen from that end
        f = (lambda x: x.flip(-1)) if mirror else (lambda x: x)
        Q, D, S = f(q)[..., :8], f(d)[..., :8], f(dm)[..., :7]
        if mirror:
            S = -S
        c_ = lambda m: Q[..., m + 2]  # noqa: E731  cell m (from the edge)
        g_ = lambda m: S[..., m + 1]  # noqa: E731
        w_ = lambda m: D[..., m + 2]  # noqa: E731
        e = 0.5 * (((2 * w_(0) + w_(-1)) * c_(0) - w_(0) * c_(-1)) / (w_(-1) + w_(0)) +
                   ((2 * w_(1) + w_(2)) * c_(1) - w_(1) * c_(2)) / (w_(1) + w_(2)))
        four = torch.stack([c_(-1), c_(0), c_(1), c_(2)])
        e = torch.minimum(torch.maximum(e, four.amin(0)), four.amax(0))
        xin = s15 * c_(1) + s11 * c_(2) - s14 * g_(2)
        a3 = 0.5 * (c_(2) + c_(3)) + (g_(2) - g_(3)) / 3
        near = torch.stack([s14 * g_(-1) + s11 * (c_(-1) - c_(0)), e - c_(1), xin - c_(2)], -1)
        far = torch.stack([e - c_(0), xin - c_(1), a3 - c_(2)], -1)
        if mirror:
            far, near = _pert(far.flip(-1), near.flip(-1))
            bl[..., -3:], br[..., -3:] = far, near
        else:
            bl[..., :3], br[..., :3] = _pert(near, far)
    ql, qr = qc[..., :-1], qc[..., 1:]
    return torch.where(c > 0, ql + (1 - c) * (br[..., :-1] - c * (bl[..., :-1] + br[..., :-1])),
                       qr + (1 + c) * (bl[..., 1:] + c * (bl[..., 1:] + br[..., 1:])))


def _corners(q, n, d):
    """q with its corner blocks as copy_corners leaves them for sweep direction d."""
    q, npx, h = q.clone(), n + 1, NG - 1
    for a in range(-2, 1):
        for b in range(-2, 1):
            for ci, cj in ((0, 0), (1, 0), (1, 1), (0, 1)):
                x, y = (npx - a if ci else a), (npx - b if cj else b)
                if d == 1:
                    s = {(0, 0): (y, 1 - x), (1, 0): (npx - y, x - npx + 1), (1, 1): (y, 2 * npx - 1 - x),
                         (0, 1): (npx - y, x - 1 + npx)}[ci, cj]
                else:
                    s = {(0, 0): (1 - y, x), (1, 0): (npx + y - 1, npx - x), (1, 1): (2 * npx - 1 - y, x),
                         (0, 1): (y + 1 - npx, npx - x)}[ci, cj]
                q[..., y + h, x + h] = q[..., s[1] + h, s[0] + h]
    return q


def _faces(q, n):
    """Fills the edge halos of six faces (leading axis) from their neighbours."""
    i = torch.arange(1, n + 1, device=q.device)
    h = NG - 1
    src = q.clone()
    for t in range(6):
        odd = t % 2 == 0  # faces 1, 3, 5
        for e in range(1, NG + 1):
            rev = n + 1 - i
            one, far = torch.full_like(i, e), torch.full_like(i, n + 1 - e)
            table = [((t + 1) % 6, (one, i)), ((t + 2) % 6, (one, rev)), ((t + 4) % 6, (rev, far)), ((t + 5) % 6, (i, far))] \
                if odd else [((t + 2) % 6, (rev, one)), ((t + 1) % 6, (i, one)), ((t + 5) % 6, (far, i)), ((t + 4) % 6, (far, rev))]
            for side, (ts, (x, y)) in enumerate(table):  # east, north, west, south
                v = src[ts][..., y + h, x + h]
                if side == 0:
                    q[t][..., NG:-NG, n + e + h] = v
                elif side == 1:
                    q[t][..., n + e + h, NG:-NG] = v
                elif side == 2:
                    q[t][..., NG:-NG, 1 - e + h] = v
                else:
                    q[t][..., 1 - e + h, NG:-NG] = v
    return q


def _tr(x):
    return x.transpose(-1, -2)


def _tp(q, cx, cy, xf, yf, m, n):
    """fv_tp_2d: averaged face values (fx, fy) of q (tile, level, j, i)."""
    dxa, dya, area = m["dxa"][:, None], m["dya"][:, None], m["area"][:, None]
    i = slice(NG, -NG)
    qy, qx = _corners(q, n, 2), _corners(q, n, 1)
    fy2 = _tr(_ppm(_tr(qy), _tr(cy), _tr(dya)))
    g = yf * fy2
    qi = (qy[..., i, :] * area[..., i, :] + g[..., :-1, :] - g[..., 1:, :]) / \
        (area[..., i, :] + yf[..., :-1, :] - yf[..., 1:, :])
    fx = _ppm(qi, cx[..., i, :], dxa[..., i, :])
    fx2 = _ppm(qx, cx, dxa)
    g = xf * fx2
    qj = (qx[..., :, i] * area[..., :, i] + g[..., :-1] - g[..., 1:]) / (area[..., :, i] + xf[..., :-1] - xf[..., 1:])
    fy = _tr(_ppm(_tr(qj), _tr(cy[..., i]), _tr(dya[..., i])))
    return 0.5 * (fx + fx2[..., i, :]), 0.5 * (fy + fy2[..., i])


def _area_flux(cx, cy, m, n):
    s, f = m["sin_sg"][:, :, None], slice(NG, NG + n + 1)
    up = lambda a: (a[..., NG - 1:NG + n], a[..., f])  # noqa: E731
    dxm, dxp = up(m["dxa"][:, None])
    dym, dyp = (_tr(v) for v in up(_tr(m["dya"][:, None])))
    xf = cx * m["dy"][:, None][..., f] * torch.where(cx > 0, dxm * up(s[2])[0], dxp * up(s[0])[1])
    yf = cy * m["dx"][:, None][..., f, :] * torch.where(cy > 0, dym * _tr(up(_tr(s[3]))[0]), dyp * _tr(up(_tr(s[1]))[1]))
    return xf, yf


def _transport(q, dp1, cx, cy, mfx, mfy, m, n, nsplit):
    """tracer_2d's sub-cycles of one tracer's levels (tile, level, j, i)."""
    xf, yf = _area_flux(cx, cy, m, n)
    i, ra = slice(NG, -NG), m["rarea"][:, None][..., NG:-NG, NG:-NG]
    cx, cy, xf, yf, mfx, mfy = (x / nsplit for x in (cx, cy, xf, yf, mfx, mfy))
    div = (mfx[..., :-1] - mfx[..., 1:] + mfy[..., :-1, :] - mfy[..., 1:, :]) * ra
    d1 = dp1[..., i, i]
    for _ in range(nsplit):
        if q.shape[0] == 6:
            q = _faces(q, n)
        fx, fy = _tp(q, cx, cy, xf, yf, m, n)
        fx, fy = fx * mfx, fy * mfy
        d2 = d1 + div
        q = q.clone()
        q[..., i, i] = (q[..., i, i] * d1 + (fx[..., :-1] - fx[..., 1:] + fy[..., :-1, :] - fy[..., 1:, :]) * ra) / d2
        d1 = d2
    return q


def _nsplit(cx, cy, m, n, split):
    npz = cx.shape[1]
    a = torch.maximum(cx[:, :, NG:-NG, :n].abs(), cy[:, :, :n, NG:-NG].abs())
    b = a + 1 - m["sin_sg"][4][:, None, NG:-NG, NG:-NG]
    top = max(npz // 6 - 1, 0)
    c = torch.cat([a[:, :top].amax((0, 2, 3)), b[:, top:].amax((0, 2, 3))])
    return [split] * npz if split else [int(1 + float(v)) for v in c]


def _advect(s, c, m):
    """The transport of every tracer, in groups of levels with one sub-cycle count."""
    n, npz = c["n"], c["npz"]
    cx, cy, mfx, mfy = (s[k].double() for k in ("cx", "cy", "mfx", "mfy"))
    ns = _nsplit(cx, cy, m, n, c.get("split", 0))
    q = s["q0"].double()
    part = max(1, int(2e7 / (q.shape[0] * n * n)))
    for v in sorted(set(ns)):
        ks = [k for k in range(npz) if ns[k] == v]
        for at in range(0, len(ks), part):
            k = torch.tensor(ks[at:at + part], device=q.device)
            w = [x[:, k] for x in (s["dp1"], cx, cy, mfx, mfy)]
            for iq in range(c["nq"]):
                r = _transport(q[:, iq, k], *w, m, n, v)
                q[:, iq, k, NG:-NG, NG:-NG] = r[..., NG:-NG, NG:-NG]
    return q, ns


def _lim(a1, a2, a3, a4, ext, iv):
    """cs_limiters."""
    if iv == 0:
        dip = (a3 - a2).abs() < -a4
        safe = torch.where(dip, a4, -torch.ones_like(a4))
        dip = dip & (a1 + 0.25 * (a3 - a2) ** 2 / safe + a4 / 12 < 0)
        neg, both = a1 <= 0, dip & (a1 < a3) & (a1 < a2)
        rise, fall = dip & ~both & (a3 > a2), dip & ~both & ~(a3 > a2)
        flat = neg | both
        rise, fall = rise & ~neg, fall & ~neg
    else:
        flat = (a1 - a2) * (a1 - a3) >= 0 if iv == 1 else ext
        d = a3 - a2
        rise = ~flat & (a4 * d < -d * d)
        fall = ~flat & ~rise & (a4 * d > d * d)
    b4 = torch.where(rise, 3 * (a2 - a1), torch.where(fall, 3 * (a3 - a1), torch.where(flat, torch.zeros_like(a4), a4)))
    b2 = torch.where(flat, a1, torch.where(fall, a3 - b4, a2))
    b3 = torch.where(flat, a1, torch.where(rise, a2 - b4, a3))
    return b2, b3, b4


def _profile(a, dp, iv, kord, qmin=None, qs=None):
    """cs_profile / scalar_profile over (level, column): the parabolas (a2, a3, a4)."""
    km = a.shape[0]
    Q, G = [None] * (km + 1), [None] * (km + 1)
    if iv == -2:
        G[1], Q[0] = torch.full_like(a[0], 0.5), 1.5 * a[0]
        for k in range(1, km - 1):
            r = dp[k - 1] / dp[k]
            b = 2 + r + r - G[k]
            Q[k], G[k + 1] = (3 * (a[k - 1] + a[k]) - Q[k - 1]) / b, r / b
        r = dp[km - 2] / dp[km - 1]
        Q[km - 1] = (3 * (a[km - 2] + a[km - 1]) - r * qs - Q[km - 2]) / (2 + r + r - G[km - 1])
        Q[km] = qs
        for k in range(km - 2, -1, -1):
            Q[k] = Q[k] - G[k + 1] * Q[k + 1]
    else:
        r = dp[1] / dp[0]
        b = r * (r + 0.5)
        Q[0], G[0] = ((r + r) * (r + 1) * a[0] + a[1]) / b, (1 + r * (r + 1.5)) / b
        for k in range(1, km):
            r = dp[k - 1] / dp[k]
            b = 2 + r + r - G[k - 1]
            Q[k], G[k] = (3 * (a[k - 1] + r * a[k]) - Q[k - 1]) / b, r / b
        t = 1 + r * (r + 1.5)
        Q[km] = (2 * r * (r + 1) * a[km - 1] + a[km - 2] - t * Q[km - 1]) / (r * (r + 0.5) - t * G[km - 1])
        for k in range(km - 1, -1, -1):
            Q[k] = Q[k] - G[k] * Q[k + 1]
    Q = torch.stack(Q)
    lo, hi = torch.minimum(a[:-1], a[1:]), torch.maximum(a[:-1], a[1:])  # interfaces 2 .. km
    g = a[1:] - a[:-1]
    x = Q[1:-1]
    both = torch.maximum(torch.minimum(x, hi), lo)
    gm, gp = torch.cat([g[:1], g[:-1]]), torch.cat([g[1:], g[-1:]])
    down = torch.minimum(x, hi)
    if iv == 0:
        down = down.clamp(min=0)
    y = torch.where(gm * gp > 0, both, torch.where(gm > 0, torch.maximum(x, lo), down))
    y[0], y[-1] = both[0], both[-1]
    Q = torch.cat([Q[:1], y, Q[-1:]])
    a2, a3 = Q[:-1].clone(), Q[1:].clone()
    ext = torch.zeros_like(a, dtype=torch.bool)
    ext[1:-1] = g[:-1] * g[1:] < 0
    for k in (0, km - 1):
        ext[k] = (a2[k] - a[k]) * (a3[k] - a[k]) > 0
    x0, x1 = 2 * a - (a2 + a3), (a2 - a3).abs()
    e5, e6 = x0.abs() > x1, (3 * x0).abs() > x1
    if iv == 0:
        a2[0] = a2[0].clamp(min=0)
        a3[-1] = a3[-1].clamp(min=0)
    elif iv == -1:
        a2[0] = torch.where(a2[0] * a[0] <= 0, torch.zeros_like(a2[0]), a2[0])
        a3[-1] = torch.where(a3[-1] * a[-1] <= 0, torch.zeros_like(a3[-1]), a3[-1])
    a4 = 3 * (2 * a - (a2 + a3))
    for k, how in ((0, 1), (1, 2), (km - 2, 2), (km - 1, 1)):
        a2[k], a3[k], a4[k] = _lim(a[k], a2[k], a3[k], a4[k], ext[k], how)
    i = slice(2, km - 2)
    b1, b2, b3 = a[i], a2[i], a3[i]
    p1 = b1 - 2 * g[2:-1]
    l1 = p1 + 1.5 * g[3:]
    p2 = b1 + 2 * g[1:-2]
    l2 = p2 - 1.5 * g[:-3]
    mn = lambda *v: functools.reduce(torch.minimum, v)  # noqa: E731
    mx = lambda *v: functools.reduce(torch.maximum, v)  # noqa: E731
    h2 = torch.minimum(torch.maximum(b2, mn(b1, p1, l1)), mx(b1, p1, l1))
    h3 = torch.minimum(torch.maximum(b3, mn(b1, p2, l2)), mx(b1, p2, l2))
    low = torch.zeros_like(ext[i]) if qmin is None else b1 < qmin
    near = lambda e: e[1:km - 3] | e[3:km - 1]  # noqa: E731
    if kord == 9:
        flat = ext[i] & (near(ext) | low)
        hu = ~flat & (a4[i].abs() > (b2 - b3).abs())
    else:
        flat = e5[i] & (near(e5) | low)
        hu = ~flat & torch.where(e5[i], near(e6), e6[i] & near(e5))
    c2 = torch.where(flat, b1, torch.where(hu, h2, b2))
    c3 = torch.where(flat, b1, torch.where(hu, h3, b3))
    c4 = torch.where(flat, torch.zeros_like(b1), 3 * (2 * b1 - (c2 + c3)))
    if iv == 0:
        c2, c3, c4 = _lim(b1, c2, c3, c4, ext[i], 0)
    a2[i], a3[i], a4[i] = c2, c3, c4
    return a2, a3, a4


def _search(p1, p2):
    """Source layer and fraction of every target interface, (level, column)."""
    km = p1.shape[0] - 1
    l = torch.searchsorted(p1.T.contiguous(), p2.T.contiguous()).T.sub(1).clamp(0, km - 1)
    lo, hi = p1.gather(0, l), p1.gather(0, l + 1)
    return l, ((p2 - lo) / (hi - lo)).clamp(0, 1), hi - lo


def _remap(a, p1, p2, where, iv, kord, qmin=None, qs=None):
    """Layer means over p2 of the profiles of a over p1, (level, column)."""
    d = p1[1:] - p1[:-1]
    a2, a3, a4 = _profile(a, d, iv, kord, qmin, qs)
    l, x, w = where
    b2, b3, b4 = a2.gather(0, l), a3.gather(0, l), a4.gather(0, l)
    head = w * x * (b2 + 0.5 * (b4 + b3 - b2) * x - b4 / 3 * x * x)  # from the layer's top
    whole = torch.cumsum(a * d, 0) - a * d
    lt, lb = l[:-1], l[1:]
    s, e = x[:-1], x[1:]
    one = b2[:-1] + 0.5 * (b4 + b3 - b2)[:-1] * (s + e) - b4[:-1] / 3 * (e * (e + s) + s * s)
    gap = (whole.gather(0, lb) - whole.gather(0, lt))
    return torch.where(lt == lb, one, (gap + head[1:] - head[:-1]) / (p2[1:] - p2[:-1]))


def _cols(x):  # (tile, level, j, i) -> (level, column)
    return x.transpose(0, 1).reshape(x.shape[1], -1)


def _uncols(x, like):
    t, k, j, i = like.shape
    return x.reshape(k, t, j, i).transpose(0, 1)


def _interfaces(dp, ak, bk):
    p1 = torch.cat([torch.full_like(dp[:1], PTOP), PTOP + torch.cumsum(dp, 0)])
    p2 = ak.view(-1, 1) + bk.view(-1, 1) * p1[-1]
    p2[0], p2[-1] = PTOP, p1[-1]
    return p1, p2


def _exact_remap(q, dp1, pt, s):
    """Tracers (in place), pt and the Eulerian thickness of the compute domain."""
    delp = dp1.clone()
    rows = dp1.shape[-1] - 2 * NG
    part = max(1, int(6e7 / (rows * dp1.shape[1] * dp1.shape[0])))
    for j0 in range(NG, NG + rows, part):
        b = (Ellipsis, slice(j0, min(j0 + part, NG + rows)), slice(NG, -NG))
        p1, p2 = _interfaces(_cols(dp1[b]), s["ak"], s["bk"])
        where = _search(p1, p2)
        delp[b] = _uncols(p2[1:] - p2[:-1], dp1[b])
        for iq in range(q.shape[1]):
            v = q[:, iq][b]
            q[:, iq][b] = _uncols(_remap(_cols(v), p1, p2, where, 0, 9, 0.0), v)
        if pt is not None:
            pt[b] = _uncols(_remap(_cols(pt[b]), p1, p2, where, 1, 10, 184.0), pt[b])
    return delp


def exact(case, seed):
    c = dict(case)
    kind, n = c["kind"], c["n"]
    s = prepare(c, seed)
    m = _metrics(n, c.get("tiles", 1))
    if kind == "step":
        q, _ = _advect(s, c, m)
        pt = s["pt0"].double() if c["pt"] else None
        delp = _exact_remap(q, s["dp1"], pt, s)
        inner = torch.zeros_like(q[:1, :1, :1])
        inner[..., NG:-NG, NG:-NG] = 1
        q *= inner  # the halo of the result buffer is not written
        return {"q": q, "delp": delp, **({} if pt is None else {"pt": pt})}
    if kind == "dyn":
        return _exact_dyn(s, c, m)
    if kind == "l2e":
        return _exact_l2e(s, c, m)
    if kind == "tlad":
        q, _ = _advect(s, c, m)
        q = q.contiguous()
        delp = _exact_remap(q, s["dp1"], None, s)
        return {"q1": None, "dq1": None, "delp": delp, "qbar0": None}
    dev = {k: torch.from_numpy(np.ascontiguousarray(v.T)).cuda()[None] for k, v in s["host"].items()}
    s.update(dev)
    q, ns = _advect(s, c, m)
    delp = _exact_remap(q, s["dp1"], s["pt"], s)
    if max(ns) > 1:
        return None
    back = lambda x: np.asfortranarray(x[0].cpu().numpy().T)  # noqa: E731
    w = {k: s["host"][k] for k in ("dp1", "cx", "cy", "mfx", "mfy")}
    w.update(q0=back(_corners(q, n, 1)), pt=back(s["pt"]), delp=back(delp), nsplit=np.array(ns, dtype=np.int32))
    return w


def _exact_dyn(s, c, m):
    n = c["n"]
    d = s["delp0"].double()
    ra, i = m["rarea"][:, None][..., NG:-NG, NG:-NG], slice(NG, -NG)
    out = {"dp1": d.clone()}
    acc = [0, 0, 0, 0]
    f = slice(NG, NG + n + 1)
    for it in range(c["sub"]):
        u, v = s["uc"][it].double() * s["bdt"], s["vc"][it].double() * s["bdt"]
        cx = u / torch.where(u > 0, m["dxa"][:, None][..., NG - 1:NG + n], m["dxa"][:, None][..., f])
        cy = v / torch.where(v > 0, m["dya"][:, None][..., NG - 1:NG + n, :], m["dya"][:, None][..., f, :])
        if it and d.shape[0] == 6:
            d = _faces(d, n)
        xf, yf = _area_flux(cx, cy, m, n)
        fx, fy = _tp(d, cx, cy, xf, yf, m, n)
        fx, fy = fx * xf[..., i, :], fy * yf[..., i]
        acc = [a + b for a, b in zip(acc, (cx, cy, fx, fy))]
        d = _corners(d, n, 1)
        d[..., i, i] = d[..., i, i] + (fx[..., :-1] - fx[..., 1:] + fy[..., :-1, :] - fy[..., 1:, :]) * ra
    return {**out, "delp": d, "cx": acc[0], "cy": acc[1], "mfx": acc[2], "mfy": acc[3]}


def _exact_l2e(s, c, m):
    n, npz = c["n"], c["npz"]
    st = {k: v.double().clone() for k, v in s["keep"].items()}
    i, r = slice(NG, -NG), slice(NG - 1, NG + n + 1)
    ak, bk = s["ak"], s["bk"]
    dp = st["delp"]
    pr = torch.cat([torch.full_like(dp[:, :1], PTOP), PTOP + torch.cumsum(dp, 1)], 1)[..., r, r]  # one-cell ring
    psr = pr[:, -1]
    ps = torch.zeros_like(dp[:, 0])
    ps[..., r, r] = psr

    def energy():
        u, v = st["u"], st["v"]
        ua = 0.5 * (u[..., NG:NG + n, i] + u[..., NG + 1:NG + n + 1, i])
        va = 0.5 * (v[..., i, NG:NG + n] + v[..., i, NG + 1:NG + n + 1])
        return ((CP * st["pt"][..., i, i] * st["pkz"] + 0.5 * (ua * ua + va * va)) * st["delp"][..., i, i]).sum(1)

    te0 = energy()
    a4, b4 = ak.view(1, -1, 1, 1), bk.view(1, -1, 1, 1)
    for k, ax in (("u", 2), ("v", 3)):  # winds on interfaces averaged to their faces
        cut = (Ellipsis, slice(NG, NG + n + 1), i) if k == "u" else (Ellipsis, i, slice(NG, NG + n + 1))
        inner = pr[..., 1:-1] if k == "u" else pr[..., 1:-1, :]
        lo, hi = inner.narrow(ax, 0, n + 1), inner.narrow(ax, 1, n + 1)
        p1 = 0.5 * (lo + hi)
        p2 = a4 + 0.5 * b4 * (lo[:, -1:] + hi[:, -1:])
        p1, p2 = _cols(p1), _cols(p2)
        st[k][cut] = _uncols(_remap(_cols(st[k][cut]), p1, p2, _search(p1, p2), -1, 9), st[k][cut])
    p1, p2 = _interfaces(_cols(dp[..., i, i]), ak, bk)
    where = _search(p1, p2)
    new = _uncols(p2[1:] - p2[:-1], st["pkz"])
    if not c["hydro"]:
        w = st["w"][..., i, i]
        st["w"][..., i, i] = _uncols(_remap(_cols(w), p1, p2, where, -2, 9, None, st["ws"].reshape(-1)), w)
        dz = -st["delz"] / dp[..., i, i]
        st["delz"] = -_uncols(_remap(_cols(dz), p1, p2, where, 1, 9), dz) * new
    pt = st["pt"]
    st["delp"] = _exact_remap(st["q"], dp, pt, s)
    pe = pr.permute(0, 2, 1, 3).clone()  # (tile, j, level, i)
    pi = _uncols(p2, torch.empty(dp.shape[0], npz + 1, n, n))
    pe[:, 1:-1, :, 1:-1] = pi.permute(0, 2, 1, 3)
    ln = torch.log(pi)
    pk = torch.exp(KAPPA * ln)
    if c["hydro"]:
        st["pkz"] = pk.diff(dim=1) / (KAPPA * ln.diff(dim=1))
    else:
        st["pkz"] = torch.exp(KAPPA / (1 - KAPPA) * torch.log(-RD / GRAV * new / st["delz"] * pt[..., i, i]))
    if c["consv"] > 0:
        ar = m["area"][..., i, i]
        gain = c["consv"] * ((te0 * ar).sum() - (energy() * ar).sum()) / (CP * (psr[..., 1:-1, 1:-1] - PTOP) * ar).sum()
        pt[..., i, i] = pt[..., i, i] + gain / st["pkz"]
    return {**st, "pe": pe, "peln": ln.permute(0, 2, 1, 3).contiguous(), "pk": pk, "ps": ps, "te0_2d": te0}
