// fused.hip -- FP64 instantiation of the fused transport kernel and the
// device-resident advection + remap step driver.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "fused.h"
#include "fused_kernel.h"
#include "mapz_fast.h"
#include "mapz_fields.h"
#include "mapz_prep.h"

namespace fv3 {

template <int HO>
static void go64(const FusedArgs<double> &a, const KindStreams &s) {
  const dim3 b(FT_LANES * 4);
  int n[7];
  fused_grid_split(a, n);
  auto grid = [&](int k) { return dim3(fused_grid_x(a, n[k], 4), (unsigned)a.npz, (unsigned)a.ntiles); };
  if (n[0] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 0, 2>), grid(0), b, 0, s.k[0], a);
  if (n[1] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 1, 2>), grid(1), b, 0, s.k[1], a);
  if (n[2] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 2, 2>), grid(2), b, 0, s.k[2], a);
  if (n[3] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 3, 2>), grid(3), b, 0, s.k[2], a);
  if (n[4] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 4, 2>), grid(4), b, 0, s.k[3], a);
  if (n[5] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 5, 2>), grid(5), b, 0, s.k[2], a);
  if (n[6] > 0) hipLaunchKernelGGL((k_fused_tp<double, 4, 1, HO, 6, 2>), grid(6), b, 0, s.k[3], a);
}

int launch_fused_f64(const FusedArgs<double> &a, const KindStreams &s) {
  if (a.hord == 8)
    go64<8>(a, s);
  else
    go64<0>(a, s);
  FV3_HIP(hipGetLastError());
  return 0;
}

__global__ void k_nsplit_check(const int *nsplit, int npz, int cap, int *flag) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int bad = 0;
    for (int k = 0; k < npz; k++) bad |= nsplit[k] > cap || nsplit[k] < 1;
    *flag = bad;
  }
}

// The halo cells of the target thickness, which keep the source's (blockIdx.y:
// level, of every tile), unless the host will refuse the step.
__global__ void __launch_bounds__(256) k_halo_dp(const double *dp1, double *delp_out, Dims d, StepCounts counts) {
  if (!__syncthreads_or(counts.any(threadIdx.x, 256))) return;
  const int e = blockIdx.x * 256 + threadIdx.x, nj = d.je - d.js + 1, rows = NG * d.nid;
  if (e >= 2 * (rows + NG * nj)) return;
  int i, j;
  if (e < 2 * rows) {
    i = e % d.nid;
    j = e < rows ? e / d.nid : NG + nj + (e - rows) / d.nid;
  } else {
    const int m = (e - 2 * rows) % (2 * NG);
    i = m < NG ? m : d.nid - 2 * NG + m;
    j = NG + (e - 2 * rows) / (2 * NG);
  }
  const long long o = blockIdx.y * d.s2 + (long long)j * d.nid + i;
  delp_out[o] = dp1[o];
}

// The geometry, metrics and strides of a pass over nq tracers of every tile.
template <typename T>
static FusedArgs<T> fused_geometry(const Ctx &c, int nq, int hord) {
  const Dims &d = c.d;
  const int npz = c.npz, nt = c.ntiles, ni = d.ie - d.is + 1, nj = d.je - d.js + 1;
  FusedArgs<T> a{};
  a.is = d.is; a.ie = d.ie; a.js = d.js; a.je = d.je;
  a.isd = d.isd; a.ied = d.ied; a.jsd = d.jsd; a.jed = d.jed;
  a.npx = d.npx; a.npy = d.npy; a.nid = d.nid;
  a.s2 = d.s2; a.sx = d.sx; a.sy = d.sy; a.smx = d.smx; a.smy = d.smy;
  a.corners = d.bounded ? 0u : d.corners;
  a.edge = d.edge;
  a.npz = npz; a.nq = nq; a.hord = hord;
  a.ntiles = nt;
  a.tq = d.s2 * npz * nq;
  a.tcx = d.sx * npz;
  a.tcy = d.sy * npz;
  a.tmx = d.smx * npz;
  a.tmy = d.smy * npz;
  a.tdp = d.s2 * npz;
  a.nstrip = (ni + FT_BX - 1) / FT_BX;
  // interior strips: every lane's column i0-3..i0+60 lies in the compute
  // domain and, on a cube face, 3 or more cells inside the tile; their lean
  // rows lt..lb keep every input row j0-3..j0+H+2 in the domain and every
  // stencil row off the cube-edge rows, so the lean kernel needs no halo,
  // corner or cube-edge code
  {
    const bool edges = d.edge || (!d.bounded && d.corners != 0u);
    auto strip_ok = [&](int st) {
      const int i0 = d.is + st * FT_BX;
      const int lo = i0 - NG, hi = i0 - NG + FT_LANES - 1;
      return lo >= d.is && hi <= d.ie && (!edges || (lo >= 3 && hi <= d.npx - 3));
    };
    // (js + 6: the output row of the first input row, three above the first
    // lean row, is itself a domain row, so no row index of a lean block clamps)
    a.lt = std::max(d.js + 2 * NG, edges ? 8 : d.js + 2 * NG);
    a.lb = std::min(d.je - NG, edges ? d.npy - 4 : d.je - NG);
    a.s_lo = 1; a.s_hi = 0; a.nmid = 0;
    int s0 = -1, s1 = -2;
    for (int st = 0; st < a.nstrip; st++)
      if (strip_ok(st)) { if (s0 < 0) s0 = st; s1 = st; }
    const bool inner = s0 >= 0 && a.lb >= a.lt;
    const int rows = inner ? a.lb - a.lt + 1 : nj;
    // The units are the edge kinds' and FP64's workgroups of four tracers, three
    // resident per CU in FP32 and two in FP64; the FP32 lean kind, whose workgroups
    // hold 4 to 32 tracers by configuration, takes the same height, since all kinds of
    // a pass share it.  A lean block's six first rows cost about four: with 2.5, two
    // tracers on a C420 L63 tile 953 us a step and on C260 L127 827, with 4 913 and
    // 800, with 12 930 and 804; ten or more tracers the same within 0.5 %.
    const long long units = (long long)a.nstrip * npz * nt * ((nq + 3) / 4);
    a.H = c.fused_h > 0 ? c.fused_h
                        : fused_block_rows(rows, units, sizeof(T) == 4 ? 768 : 512, inner ? 4.0 : 2.0 * NG);
    a.H = std::min(nj, a.H);
    a.nvblk = (nj + a.H - 1) / a.H;
    if (inner) {
      a.s_lo = s0;
      a.s_hi = s1;
      a.nmid = (a.lb - a.lt + a.H) / a.H;
    }
  }
  const GridDev<T> &g = grid_of<T>(c);
  a.area = g.area; a.rarea = g.rarea; a.dxa = g.dxa; a.dya = g.dya;
  a.tgs2 = g.s2;
  if (sizeof(T) == 4) {
    a.gxp = (const T *)c.gfac32;
    a.gxm = a.gxp + (long long)(d.nid + 1) * d.njd;
    a.gyp = a.gxm + (long long)(d.nid + 1) * d.njd;
    a.gym = a.gyp + (long long)d.nid * (d.njd + 1);
    a.gex = a.gym + (long long)d.nid * (d.njd + 1);
    a.tgf = 2 * (long long)(d.nid + 1) * d.njd + 2 * (long long)d.nid * (d.njd + 1) + (long long)d.nid * d.njd;
  }
  return a;
}

template <typename T>
static int fused_step_t(Ctx &c, int nq, const T *q_in, T *q_out, T *pt, const double *dp1,
                        double *delp_out, const T *cx, const T *cy, const T *mfx, const T *mfy,
                        const double *ak, const double *bk, double ptop, int hord, int kord_tr,
                        int kord_tm, double t_min, int nsplit_cap, const StepArena &arena) {
  const Dims &d = c.d;
  const int npz = c.npz;
  hipStream_t s = c.stream;
  if (hord < 7 || hord > 13) return set_error("hord=%d: only the monotone orders 7..13 are implemented", hord);
  if (c.graph_safe && nsplit_cap <= 0)
    return set_error("graph-safe steps need nsplit_cap > 0 (no device-to-host read)");
  // the host-array entry points run the transport alone (c.transport_only)
  const bool remap_phase = !c.transport_only;
  const bool fast_remap = remap_phase && std::is_same<T, float>::value && c.remap_mode != 1 && npz >= 8;
  // the FP64 remap of the column tables (mapz_fields.hip), out of place too
  const bool fields = remap_phase && std::is_same<T, double>::value && npz <= FIELDS_MAX_KM;
  std::vector<int> kt(nq, kord_tr);
  if (fields && remap_orders_check(npz, nq, kt.data(), pt != nullptr, kord_tm)) return 1;
  const bool oop = fast_remap || fields;
  // the per-column remap synchronises the host with the stream, so only the
  // column-shared FP32 remap can be captured
  if (c.graph_safe && !fast_remap)
    return set_error("graph-safe steps need the FP32 form with the column-shared remap and npz >= 8");
  const bool ext = arena.base != nullptr;
  if (ext && !fast_remap)
    return set_error("the no-allocation step needs the FP32 form with the column-shared remap and npz >= 8");
  // head: cmax, frac, nsplit, flag (the context's staging arena, or the
  // front of the caller's arena)
  size_t off = 0;
  auto take = [&](size_t b) {
    size_t o = off;
    off += (b + 255) & ~(size_t)255;
    return o;
  };
  const size_t o_cmax = take(sizeof(double) * npz), o_frac = take(sizeof(T) * npz);
  const size_t o_ns = take(sizeof(int) * npz), o_flag = take(sizeof(int));
  const size_t head = off;
  const int nt = c.ntiles;
  const long long qsize = d.s2 * npz * nq * nt;  // all tiles
  const int ni = d.ie - d.is + 1, nj = d.je - d.js + 1;
  // the FP32 remap's scratch: q_tmp, the pt source copy, every tile's column data
  const size_t b_q = ((sizeof(T) * qsize) + 255) & ~(size_t)255;
  const size_t b_pt = pt ? ((sizeof(T) * d.s2 * npz * nt) + 255) & ~(size_t)255 : 0;
  const size_t b_col = fast_remap ? remap_cols_bytes(npz, (long long)ni * nj) : 0;
  if (ext && head + b_q + b_pt + b_col * nt > arena.bytes)
    return set_error("this step needs %zu bytes of scratch; the no-allocation scratch holds %zu "
                     "(fv3_step_dev allocates its own)", head + b_q + b_pt + b_col * nt, arena.bytes);
  char *base = ext ? arena.base : (char *)ctx_stage(c, head);
  if (!base) return 1;
  double *cmax = (double *)(base + o_cmax);
  T *frac = (T *)(base + o_frac);
  int *nspl = (int *)(base + o_ns), *flag = c.graph_safe ? c.step_flag : (int *)(base + o_flag);
  // FP64: the scratch (area fluxes first, which the sub-cycle counts' pass over
  // the Courant numbers also computes) is sized before the counts are known; a
  // step without the tables' remap gets its second q after them, if it has
  // sub-cycles
  T *xfx = nullptr, *yfx = nullptr, *q_tmp64 = nullptr;
  const size_t b_xf = (sizeof(T) * d.sx * npz * nt + 255) & ~(size_t)255;
  const size_t b_yf = (sizeof(T) * d.sy * npz * nt + 255) & ~(size_t)255;
  char *sc64 = nullptr;
  if constexpr (std::is_same<T, double>::value) {
    sc64 = (char *)ctx_scratch(c, b_xf + b_yf + (fields ? b_q + b_pt + coltab_bytes<T>(npz, (long long)ni * nj * nt) : 0));
    if (!sc64) return 1;
    xfx = (T *)sc64;
    yfx = (T *)(sc64 + b_xf);
    sc64 += b_xf + b_yf;
    if (fields) q_tmp64 = (T *)sc64;
  }
  // The remap runs out of place: the last transport pass of every
  // level lands in q_tmp (the caller's q_out serves as the alternate pass
  // buffer), and the remap writes q_out.
  T *q_tmp = nullptr, *pt_src = nullptr;
  char *tab = nullptr;  // the column tables
  RemapCols cols{};  // column data of the first tile
  if (fast_remap) {
    if (remap_fast_check(npz, (long long)ni * nj, d.s2, kord_tr, kord_tm, pt != nullptr)) return 1;
    char *sc = ext ? arena.base + head : (char *)ctx_scratch(c, b_q + b_pt + b_col * nt);
    if (!sc) return 1;
    q_tmp = (T *)sc;
    pt_src = pt ? (T *)(sc + b_q) : nullptr;
    cols = remap_cols_carve(sc + b_q + b_pt, npz, (long long)ni * nj);
  } else if (fields) {
    q_tmp = q_tmp64;
    pt_src = pt ? (T *)(sc64 + b_q) : nullptr;
    tab = sc64 + b_q + b_pt;
  }
  // The remap's column tables (thicknesses only) and the copy of pt that it needs
  // run on their own stream beside the host's wait for the sub-cycle counts and the
  // transport, the FP64 form's also beside the counts; the field kernel joins them
  // below.  What writes the target thickness comes after the counts and looks at
  // them (StepCounts).  In order on one stream where the caller has the target
  // thickness overwrite the source's.
  const size_t b_dp = sizeof(double) * d.s2 * npz * nt;
  const bool same_dp = reinterpret_cast<uintptr_t>(delp_out) < reinterpret_cast<uintptr_t>(dp1) + b_dp &&
                       reinterpret_cast<uintptr_t>(dp1) < reinterpret_cast<uintptr_t>(delp_out) + b_dp;
  const bool early = oop && !same_dp && c.concurrent_kinds && c.aux[3];
  hipStream_t sp = early ? c.aux[3] : s;
  const int *counts = nsplit_cap > 0 ? nullptr : nspl;
  FieldsArgs<T> fa{};
  auto remap_tables = [&]() -> int {  // FP64
    if (pt) FV3_HIP(hipMemcpyAsync(pt_src, pt, sizeof(T) * d.s2 * npz * nt, hipMemcpyDeviceToDevice, sp));
    fa.tab = coltab_carve<T>(tab, npz, (long long)ni * nj * nt);
    ColSource cs{};
    cs.ptop = ptop;
    cs.ak = ak;
    cs.bk = bk;
    cs.delp = dp1;
    return fields_prep<T>(c, fa.tab, cs, ni, nj, false, sp);
  };
  auto remap_target = [&]() -> int {  // FP32: with the tables
    if constexpr (std::is_same<T, double>::value) {
      return fields_target(c, fa.tab, dp1, delp_out, counts, sp);
    } else {
      if (delp_out != dp1) {
        hipLaunchKernelGGL(k_halo_dp, dim3((unsigned)((2 * NG * (d.nid + nj) + 255) / 256), (unsigned)(npz * nt)),
                           dim3(256), 0, sp, dp1, delp_out, d, StepCounts{counts, npz});
        FV3_HIP(hipGetLastError());
      }
      if (pt) FV3_HIP(hipMemcpyAsync(pt_src, pt, sizeof(T) * d.s2 * npz * nt, hipMemcpyDeviceToDevice, sp));
      return remap_fast_prep_f32(c, npz, ak, bk, ptop, dp1, delp_out, counts, cols, b_col, sp);
    }
  };
  if (early && fields) FV3_HIP(hipEventRecord(c.fork_ev, s));
  if (device_nsplit<T>(c, cx, cy, c.step_per_level, c.step_per_level ? 0 : c.step_q_split, cmax, nspl, frac, xfx, yfx,
                       nsplit_cap > 0 ? nullptr : c.ns_host))
    return 1;
  if (early) {
    if (fields) {
      FV3_HIP(hipStreamWaitEvent(sp, c.fork_ev, 0));
      if (remap_tables()) return 1;
    }
    FV3_HIP(hipEventRecord(c.chunk_ev, s));
    FV3_HIP(hipStreamWaitEvent(sp, c.chunk_ev, 0));
    if (remap_target()) return 1;
    FV3_HIP(hipEventRecord(c.prep_ev, sp));
  }
  int cap = nsplit_cap;
  if (cap <= 0) {
    FV3_HIP(hipStreamSynchronize(s));  // the counts are in ns_host
    const std::vector<int> h(c.ns_host, c.ns_host + npz);
    cap = *std::max_element(h.begin(), h.end());
    if (cap < 1) {
      if (early) FV3_HIP(hipStreamSynchronize(sp));  // the next call reuses the scratch
      return set_error("nsplit < 1 from a non-finite Courant number");
    }
    c.last_nsplit = h;
  }
  if (!q_tmp && cap > 1) {
    const size_t b_flux = xfx ? b_xf + b_yf : 0;
    char *sc = (char *)ctx_scratch(c, b_flux + b_q);
    if (!sc) return 1;
    q_tmp = (T *)(sc + b_flux);
    if constexpr (std::is_same<T, double>::value) {
      if (sc != (char *)xfx) {  // the scratch has grown: the fluxes once more
        xfx = (T *)sc;
        yfx = (T *)(sc + b_xf);
        if (area_fluxes(c, cx, cy, xfx, yfx)) return 1;
      }
    }
  }
  FusedArgs<T> a = fused_geometry<T>(c, nq, hord);
  a.cap = cap;
  a.nsplit = nspl;
  a.q_in = q_in;
  a.q_out = oop ? q_tmp : q_out;
  a.q_tmp = oop ? q_out : q_tmp;
  a.xfx = xfx; a.yfx = yfx;
  a.cx = cx; a.cy = cy; a.mfx = mfx; a.mfy = mfy; a.dp1 = dp1;
  const bool timing = c.timing && !c.graph_safe;
  if (timing) FV3_HIP(hipEventRecord(c.ev[0], s));
  // FP32 pipelining: the tracers go through the passes in chunks of cq, and
  // each chunk's remap runs on aux[3] (behind the column prep) while the
  // next chunk is transported; pt is remapped with the last chunk
  int cq = nq;
  if constexpr (std::is_same<T, float>::value) {
    if (early && c.pipe_chunk != 0) {
      cq = c.pipe_chunk > 0 ? c.pipe_chunk : fused32_round(c.fused_cfg);
      cq = std::max(1, std::min(cq, nq));
    }
  }
  const bool pipe = cq < nq;
  // each pass: the edge kinds fork onto auxiliary streams and join back
  // before the next pass (which reads every face's previous pass); when
  // pipelined they share two streams, so that with the remap's stream the
  // step uses four
  const bool conc = c.concurrent_kinds && c.aux[0] && c.aux[1] && c.aux[2];
  const KindStreams ks = !conc ? KindStreams{{s, s, s, s}}
                         : (pipe ? KindStreams{{s, c.aux[0], c.aux[0], c.aux[1]}}
                                 : KindStreams{{s, c.aux[0], c.aux[1], c.aux[2]}});
  const int nfork = !conc ? 0 : (pipe ? 2 : 3);
  const T *const pass_in = a.q_in;
  T *const pass_out = a.q_out, *const pass_tmp = a.q_tmp;
  const long long tq = a.tq;
  for (int q0 = 0; q0 < nq; q0 += cq) {
    const int nqc = std::min(cq, nq - q0);
    const long long qoff = (long long)q0 * npz * d.s2;
    a.nq = nqc;
    a.q_in = pass_in + qoff;
    a.q_out = pass_out + qoff;
    a.q_tmp = pass_tmp ? pass_tmp + qoff : nullptr;
    for (int it = 1; it <= cap; it++) {
      a.it = it;
      if (nfork) {
        FV3_HIP(hipEventRecord(c.fork_ev, s));
        for (int i = 0; i < nfork; i++) FV3_HIP(hipStreamWaitEvent(c.aux[i], c.fork_ev, 0));
      }
      int rc;
      if constexpr (std::is_same<T, double>::value)
        rc = launch_fused_f64(a, ks);
      else
        rc = launch_fused_f32(a, c.fused_cfg, ks);
      if (rc) return rc;
      for (int i = 0; i < nfork; i++) {
        FV3_HIP(hipEventRecord(c.join_ev[i], c.aux[i]));
        FV3_HIP(hipStreamWaitEvent(s, c.join_ev[i], 0));
      }
    }
    if constexpr (std::is_same<T, float>::value) {
      if (pipe) {
        FV3_HIP(hipEventRecord(c.chunk_ev, s));
        FV3_HIP(hipStreamWaitEvent(sp, c.chunk_ev, 0));
        const bool last = q0 + nqc >= nq;
        if (remap_fast_fields_f32(c, npz, nqc, q_tmp + qoff, q_out + qoff, last ? pt_src : nullptr,
                                  last ? pt : nullptr, kord_tr, kord_tm, t_min, cols, b_col, tq, sp))
          return 1;
      }
    }
  }
  a.nq = nq;
  if (nsplit_cap > 0) {
    hipLaunchKernelGGL(k_nsplit_check, dim3(1), dim3(1), 0, s, nspl, npz, cap, flag);
    FV3_HIP(hipGetLastError());
  }
  if (timing) FV3_HIP(hipEventRecord(c.ev[1], s));
  // remap: source thickness is dp1, target lands in delp_out; pipelined, the
  // remap phase is the wait for the last chunks' remaps
  if (pipe) {
    if (timing) FV3_HIP(hipEventRecord(c.ev[2], s));
    FV3_HIP(hipEventRecord(c.prep_ev, sp));
    FV3_HIP(hipStreamWaitEvent(s, c.prep_ev, 0));
  } else if (oop) {
    if (early)
      FV3_HIP(hipStreamWaitEvent(s, c.prep_ev, 0));
    else if ((fields && remap_tables()) || remap_target())
      return 1;
  } else if (remap_phase && delp_out != dp1) {
    FV3_HIP(hipMemcpyAsync(delp_out, dp1, b_dp, hipMemcpyDeviceToDevice, s));
  }
  if (timing && !pipe) FV3_HIP(hipEventRecord(c.ev[2], s));
  if constexpr (std::is_same<T, float>::value) {
    if (fast_remap && !pipe) {
      if (remap_fast_fields_f32(c, npz, nq, q_tmp, q_out, pt_src, pt, kord_tr, kord_tm, t_min, cols, b_col, tq, s))
        return 1;
    }
  }
  if (fields) {
    fa.set[fa.nset++] = tracer_set<T>(c, q_tmp, q_out, nq);
    for (int iq = 0; iq <= nq; iq++) fa.kord[iq] = (signed char)std::min(iq < nq ? kord_tr : kord_tm, 17);
    if (pt) {
      FieldSet<T> &x = fa.set[fa.nset++] = cell_set<T>(c, pt_src, pt, 1);
      x.use_qmin = true;
      x.qmin = (T)t_min;
    }
    if (fields_run<T>(c, fa, ni, nj)) return 1;
  } else if (!fast_remap && remap_phase) {
    if (remap_tracers_plain<T>(c, npz, nq, ak, bk, ptop, delp_out, q_out, pt, kt.data(), kord_tm,
                               t_min, 0))
      return 1;
  }
  if (timing) {
    FV3_HIP(hipEventRecord(c.ev[3], s));
    c.last_passes = cap;
    c.ev_valid = true;
  }
  if (fields) FV3_HIP(hipStreamSynchronize(s));  // FP64 steps return when they are done
  if (nsplit_cap > 0 && !c.graph_safe) {
    int hf = 0;
    FV3_HIP(hipMemcpyAsync(&hf, flag, sizeof(int), hipMemcpyDeviceToHost, s));
    FV3_HIP(hipStreamSynchronize(s));
    if (hf) return set_error("a level needs more sub-cycles than nsplit_cap=%d", nsplit_cap);
  }
  return 0;
}

int fused_pass64(Ctx &c, int nq, int hord, const double *q_in, double *q_out, const double *dp, long long tdp,
                 const double *cx, const double *cy, const double *mfx, const double *mfy, const double *xfx,
                 const double *yfx, const int *nsplit) {
  hipStream_t s = c.stream;
  FusedArgs<double> a = fused_geometry<double>(c, nq, hord);
  a.cap = 0x7fffffff;
  a.it = 1;  // reads q_in and dp as they are; every level lands in q_out
  a.nsplit = nsplit;
  a.q_in = q_in;
  a.q_out = a.q_tmp = q_out;
  a.dp1 = dp;
  if (c.ntiles > 1) a.tdp = tdp;
  a.cx = cx; a.cy = cy; a.mfx = mfx; a.mfy = mfy; a.xfx = xfx; a.yfx = yfx;
  const bool conc = c.concurrent_kinds && c.aux[0] && c.aux[1] && c.aux[2];
  const KindStreams ks = conc ? KindStreams{{s, c.aux[0], c.aux[1], c.aux[2]}} : KindStreams{{s, s, s, s}};
  if (conc) {
    FV3_HIP(hipEventRecord(c.fork_ev, s));
    for (int i = 0; i < 3; i++) FV3_HIP(hipStreamWaitEvent(c.aux[i], c.fork_ev, 0));
  }
  if (launch_fused_f64(a, ks)) return 1;
  if (conc)
    for (int i = 0; i < 3; i++) {
      FV3_HIP(hipEventRecord(c.join_ev[i], c.aux[i]));
      FV3_HIP(hipStreamWaitEvent(s, c.join_ev[i], 0));
    }
  return 0;
}

int remap_only_f32(Ctx &c, int nq, const float *q_src, float *q_dst, float *pt, const double *dp1,
                   double *delp_out, const double *ak, const double *bk, double ptop, int kord_tr,
                   int kord_tm, double t_min) {
  const Dims &d = c.d;
  const int npz = c.npz, nt = c.ntiles, ni = d.ie - d.is + 1, nj = d.je - d.js + 1;
  hipStream_t s = c.stream;
  if (remap_fast_check(npz, (long long)ni * nj, d.s2, kord_tr, kord_tm, pt != nullptr)) return 1;
  const size_t b_pt = pt ? ((sizeof(float) * d.s2 * npz * nt) + 255) & ~(size_t)255 : 0;
  const size_t b_col = remap_cols_bytes(npz, (long long)ni * nj);
  char *sc = (char *)ctx_scratch(c, b_pt + b_col * nt);
  if (!sc) return 1;
  float *pt_src = pt ? (float *)sc : nullptr;
  const long long tq = d.s2 * npz * nq, tl = d.s2 * npz;
  FV3_HIP(hipMemcpyAsync(delp_out, dp1, sizeof(double) * tl * nt, hipMemcpyDeviceToDevice, s));
  if (pt) FV3_HIP(hipMemcpyAsync(pt_src, pt, sizeof(float) * tl * nt, hipMemcpyDeviceToDevice, s));
  const RemapCols cols = remap_cols_carve(sc + b_pt, npz, (long long)ni * nj);
  if (remap_fast_prep_f32(c, npz, ak, bk, ptop, dp1, delp_out, nullptr, cols, b_col, s)) return 1;
  return remap_fast_fields_f32(c, npz, nq, q_src, q_dst, pt_src, pt, kord_tr, kord_tm, t_min, cols, b_col, tq, s);
}

int fused_step(Ctx &c, bool fp32, int nq, const void *q_in, void *q_out, void *pt,
               const double *dp1, double *delp_out, const void *cx, const void *cy,
               const void *mfx, const void *mfy, const double *ak, const double *bk, double ptop,
               int hord, int kord_tr, int kord_tm, double t_min, int nsplit_cap,
               const StepArena &arena) {
  if (fp32)
    return fused_step_t<float>(c, nq, (const float *)q_in, (float *)q_out, (float *)pt, dp1, delp_out,
                               (const float *)cx, (const float *)cy, (const float *)mfx,
                               (const float *)mfy, ak, bk, ptop, hord, kord_tr, kord_tm, t_min,
                               nsplit_cap, arena);
  return fused_step_t<double>(c, nq, (const double *)q_in, (double *)q_out, (double *)pt, dp1, delp_out,
                              (const double *)cx, (const double *)cy, (const double *)mfx,
                              (const double *)mfy, ak, bk, ptop, hord, kord_tr, kord_tm, t_min,
                              nsplit_cap, arena);
}

}  // namespace fv3
