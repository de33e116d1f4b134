// dyncore.hip -- the tracer path's inputs as dyn_core accumulates them over
// its acoustic sub-steps: the Courant numbers cx, cy, the mass fluxes mfx,
// mfy and the start thickness dp1 that fv_dynamics hands to tracer_2d_1L
// (dyn_core / d_sw live in the absent atmos_cubed_sphere submodule, reached
// from atmos_model.F90:879).  Each of n_split sub-steps of length bdt
//   - turns the sub-step's C-grid winds into Courant numbers with the upwind
//     cell width and area fluxes through the face with the upwind metric,
//   - transports delp with fv_tp_2d (no mass fluxes: the fluxes are the
//     area fluxes times the delp face values; copy_corners acts on delp),
//   - adds the delp fluxes and Courant numbers into mfx, mfy, cx, cy,
//   - updates delp by the flux divergence, and
//   - refreshes delp's six-face halo before the next sub-step.
// FV3_FORM_PLAIN64 runs every (tile, level) slab of a sub-step in one launch
// per stage (the staged transport's stage kernels, in the FP64 oracle's
// operation order); FV3_FORM_FUSED64 / FUSED32 run a whole sub-step in one
// launch that streams rows and keeps every intermediate in registers, with the
// same expressions, so both FP64 forms match the oracle bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/fv3atm_amd.h"
#include "fused_tp.h"
#include "fv3_internal.h"

namespace fv3 {

namespace {

template <typename F>
__global__ void __launch_bounds__(256) k_rect(F f, int i0, int i1, int j0, int j1) {
  const int i = i0 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int j = j0 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i <= i1 && j <= j1) f(i, j, (int)blockIdx.z);
}

template <typename F>
int launch_rect(hipStream_t s, F f, int i0, int i1, int j0, int j1, int nz) {
  if (i1 < i0 || j1 < j0 || nz <= 0) return 0;
  const dim3 b(64, 4);
  const dim3 g((unsigned)((i1 - i0 + 64) / 64), (unsigned)((j1 - j0 + 4) / 4), (unsigned)nz);
  hipLaunchKernelGGL(k_rect<F>, g, b, 0, s, f, i0, i1, j0, j1);
  FV3_HIP(hipGetLastError());
  return 0;
}

template <typename T>
struct RowQ {
  const T *p;
  int lo;
  __device__ __forceinline__ T operator()(int m) const { return p[m - lo]; }
};
template <typename T>
struct ColQ {
  const T *p;
  int lo;
  long long stride;
  __device__ __forceinline__ T operator()(int m) const { return p[(long long)(m - lo) * stride]; }
};


// ---- one acoustic sub-step in one launch ---------------------------------------
// A wave owns a strip of DYN_W columns and a block of rows of one (tile, level)
// slab, one lane per column (three more on each side), and streams over the
// rows: a row's x-side (Courant numbers and area fluxes, the inner x-sweep,
// q_j) when it is loaded, the y-faces two rows behind it (Courant numbers,
// inner and outer y-sweep, the y-fluxes), and three rows behind it q_i, the
// outer x-sweep, the x-fluxes and the delp update.  Neighbours in x come from
// the neighbouring lanes (DPP), neighbours in y from rows kept in registers, so
// that each slope, face value and cell limiter is computed once per cell and
// sweep, and nothing goes through LDS.  Each quantity is the same expression as
// in the stage kernels, so the FP64 form rounds as they do.  The next row's
// loads are issued before a row is worked on; the four waves of a workgroup
// take four levels, whose metric loads hit the same lines.  Cube edges: rows at
// the y-edges by uniform branches, columns at the x-edges in a second form of
// the row loop for the strips that hold some.  Bound by VALU issue (85% busy in
// FP32).  C384 L127, per sub-step: 345 us in FP32, 640 in FP64; 32 x 16 (FP64
// 32 x 8) blocks in LDS, each face recomputing its cell's slopes and limiter
// from there, took 940 and 1500 us.  delp is read from one buffer and written to another (a
// neighbouring wave still reads the old values as its halo); the halo cells are
// carried over, and the corner-block cells get their x-sweep (dir 1)
// copy_corners sources, as the stages leave them in place.
struct DynSubArgs {
  Dims d;
  int npz, nz, ord_in, ord_ou, first, rows;  // rows: per block
  long long gs2, gdx, gdy;
};

constexpr int DYN_W = 58;

// cells m-2 .. m+2 of a sweep line, cell m at index 2
template <typename T>
struct Win5 {
  T v[5];
  __device__ __forceinline__ T operator()(int k) const { return v[k]; }
};

// place of cell m on a sweep line: 0 inner, 1 .. 3 cells 0, 1, 2 of an edge,
// 4 .. 6 cells npx-2, npx-1, npx
__device__ __forceinline__ int edge_place(const LineGeom &g, int m) {
  if (!g.edge) return 0;
  if (g.is == 1 && m <= 2) return m == 0 ? 1 : (m == 1 ? 2 : 3);
  if (g.ie + 1 == g.npx && m >= g.npx - 2) return m == g.npx - 2 ? 4 : (m == g.npx - 1 ? 5 : 6);
  return 0;
}

// The expressions of ppm_dm, ppm_al, ppm_edge_face and ppm_cell.  Minima and
// maxima are the same compares and selects: as instructions (2.11 against 2.16 ms
// at C384 L127) they pass over a NaN, and a thickness that has gone bad spread to
// fewer cells than in the stages.
template <typename T>
__device__ __forceinline__ T slope(T qm, T q, T qp) {
  const T xt = T(0.25) * (qp - qm);
  return fsign(mn3(fabs(xt), mx3(qm, q, qp) - q, q - mn3(qm, q, qp)), xt);
}
template <typename T>
__device__ __forceinline__ T face(T ql, T q, T dml, T dm) {
  return T(0.5) * (ql + q) + K<T>::r3 * (dml - dm);
}
// the cube-edge face between cells 1 and 2 of four (their spacings: d)
template <typename T>
__device__ __forceinline__ T edge_face(T q0, T q1, T q2, T q3, T d0, T d1, T d2, T d3) {
  const T xt = T(0.5) * (((T(2) * d1 + d0) * q1 - d1 * q0) / (d0 + d1) + ((T(2) * d2 + d3) * q2 - d2 * q3) / (d2 + d3));
  return mn2(mx2(xt, mn2(mn3(q0, q1, q2), q3)), mx2(mx3(q0, q1, q2), q3));
}

// (bl, br) of an inner cell: orders 8 and 11 from its slope and its two face
// values, the others from the window
template <bool O8, typename T>
__device__ __forceinline__ void inner_cell(const Win5<T> &q, T dm, T al, T ar, int iord, T &bl, T &br) {
  if (O8 || iord == 8 || iord == 11) {
    const T xt = iord == 8 ? T(2) * dm : K<T>::ppm_fac * dm;
    bl = -fsign(mn2(fabs(xt), fabs(al - q(2))), xt);
    br = fsign(mn2(fabs(xt), fabs(ar - q(2))), xt);
  } else {
    ppm_cell<T>(q, q, 2, LineGeom{0, 0, 0, false}, iord, bl, br);
  }
}

// (bl, br) of an edge cell from its face values, the slopes beside it and the
// cells beside it
template <typename T>
__device__ __forceinline__ void edge_cell(int place, T qm, T q, T qp, T al, T ar, T dml, T dmr, T &bl, T &br) {
  bl = place == 1 ? K<T>::s14 * dml + K<T>::s11 * (qm - q) : al - q;
  br = place == 6 ? K<T>::s11 * (qp - q) - K<T>::s14 * dmr : ar - q;
  pert_ppm1(q, bl, br, 1);
}

// flux through a face between cells l and r for Courant number c
template <typename T>
__device__ __forceinline__ T upwind(T c, T ql, T bll, T brl, T qr, T blr, T brr) {
  const bool pos = c > T(0);
  const T b = pos ? bll + brl : blr + brr, a = pos ? brl : blr, q = pos ? ql : qr, s = pos ? c : -c;
  return q + (T(1) - s) * (a - s * b);
}

// One y-line per lane, a row at a time: after add(r) the window holds rows
// r-4 .. r and (bl, br) belong to row r-2, (blp, brp) to row r-3.  The face
// values next to a cube edge replace the inner ones.
template <typename T, bool O8>
struct YLine {
  Win5<T> q;
  T dm0, dm1, al, bl, br, blp, brp;  // slopes of rows r-3, r-2; face value of row r-2
  template <typename D>
  __device__ __forceinline__ void add(T v, const LineGeom &g, int r, const D &spacing, int iord) {
#pragma unroll
    for (int k = 0; k < 4; k++) q.v[k] = q.v[k + 1];
    q.v[4] = v;
    const T dm2 = slope<T>(q(2), q(3), q(4));  // of row r-1
    T ar = face<T>(q(2), q(3), dm1, dm2);      // of face r-1
    const int f = r - 1;
    int place = 0;
    if (g.edge && ((g.is == 1 && f <= 3) || (g.ie + 1 == g.npx && f >= g.npx - 1))) {
      place = edge_place(g, r - 2);
      const bool lo = g.is == 1 && f <= 3;
      if (f == (lo ? 1 : g.npx)) {
        const Win5<T> d = spacing();  // of rows r-3 .. r
        ar = edge_face<T>(q(1), q(2), q(3), q(4), d(0), d(1), d(2), d(3));
      } else if (lo && f == 2) {
        ar = K<T>::s15 * q(2) + K<T>::s11 * q(3) - K<T>::s14 * dm2;
      } else if (!lo && f == g.npx - 1) {
        ar = K<T>::s15 * q(3) + K<T>::s11 * q(2) + K<T>::s14 * dm1;
      }
    }
    blp = bl;
    brp = br;
    if (place)
      edge_cell<T>(place, q(1), q(2), q(3), al, ar, dm0, dm2, bl, br);
    else
      inner_cell<O8, T>(q, dm1, al, ar, iord, bl, br);
    dm0 = dm1;
    dm1 = dm2;
    al = ar;
  }
  __device__ __forceinline__ T flux(T c) const { return upwind<T>(c, q(1), blp, brp, q(2), bl, br); }
};

template <typename T>
struct DynRow {
  T p, u, dxa, sg0, sg2, dy, area, cx;  // row r
  T v, dx, dya, sg1, sg3, cy, mfy;      // y-faces (and cells) r-2
  T mfx, areaj, rarea;                  // row r-3
  __device__ __forceinline__ void arrived() {
    asm volatile("" : "+v"(p), "+v"(u), "+v"(dxa), "+v"(sg0), "+v"(sg2), "+v"(dy), "+v"(area), "+v"(cx));
    asm volatile("" : "+v"(v), "+v"(dx), "+v"(dya), "+v"(sg1), "+v"(sg3), "+v"(cy), "+v"(mfy));
    asm volatile("" : "+v"(mfx), "+v"(areaj), "+v"(rarea));
  }
};

template <typename T, bool O8>  // O8: both orders are 8 or 11
__global__ void __launch_bounds__(256) k_dyn_sub(const DynSubArgs a, const GridDev<T> g, T bdt,
                                                 const T *__restrict__ u, const T *__restrict__ v,
                                                 const T *__restrict__ din, T *__restrict__ dout, T *cx, T *cy, T *mfx,
                                                 T *mfy) {
  const Dims &d = a.d;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int z = (int)blockIdx.x * 4 + wave;
  if (z >= a.nz) return;  // whole wave; no barriers below
  const int tile = z / a.npz;
  const int i0 = d.is + (int)blockIdx.y * DYN_W, i1 = min(i0 + DYN_W - 1, d.ie);
  const int j0 = d.js + (int)blockIdx.z * a.rows, j1 = min(j0 + a.rows - 1, d.je);
  const int i = i0 - 3 + lane;
  const LineGeom gx{d.is, d.ie, d.npx, d.edge}, gy{d.js, d.je, d.npy, d.edge};
  // lanes past the slab repeat its last column and store nothing
  const int oc = min(i, d.ied) - d.isd, of = min(max(i, d.is), d.ie + 1) - d.is, om = min(max(i, d.is), d.ie) - d.is;
  const T *dl = din + (long long)z * d.s2;
  T *dw = dout + (long long)z * d.s2;
  const long long gt = tile * a.gs2;
  const T *dxa = g.dxa + gt, *dya = g.dya + gt, *area = g.area + gt, *rarea = g.rarea + gt;
  const T *sg = g.sin_sg + tile * 9 * a.gs2, *dx = g.dx + tile * a.gdx, *dy = g.dy + tile * a.gdy;
  const T *sg1 = sg + a.gs2, *sg2 = sg + 2 * a.gs2, *sg3 = sg + 3 * a.gs2;
  u += (long long)z * d.sx;
  v += (long long)z * d.sy;
  cx += (long long)z * d.sx;
  cy += (long long)z * d.sy;
  mfx += (long long)z * d.smx;
  mfy += (long long)z * d.smy;
  const bool first = a.first != 0;
  const bool x_edge = d.edge && ((d.is == 1 && i0 - 3 <= 2) || (d.ie + 1 == d.npx && i1 + 3 >= d.npx - 2));
  const bool corner_strip = !d.bounded && (i0 - 3 <= 0 || i1 + 3 >= d.npx);
  const int x_place = edge_place(gx, i);
  // faces next to an edge: 1 the edge's own, 2 and 3 the ones one cell inside
  const bool x_lo = d.is == 1, x_hi = d.ie + 1 == d.npx;
  const int x_face = (x_lo && i == 1) || (x_hi && i == d.npx) ? 1 : x_lo && i == 2 ? 2 : x_hi && i == d.npx - 1 ? 3 : 0;
  const bool own_x = i >= i0 && i <= i1;                                      // cells
  const bool own_xf = own_x || (i == d.ie + 1 && i1 == d.ie);                 // x-faces
  const bool own_xh = own_x || (i < d.is && i0 == d.is) || (i > d.ie && i <= d.ied && i1 == d.ie);  // with the halo
  auto left = [](T x) { return from_left(x); };
  auto right = [](T x) { return from_right(x); };

  // scalar bases and 32-bit lane offsets in bytes
  constexpr unsigned B = sizeof(T);
  const unsigned lc = (unsigned)oc * B, lf = (unsigned)of * B, lm = (unsigned)om * B;
  const unsigned rc = (unsigned)d.nid * B, rf = (unsigned)d.nix * B, rm = (unsigned)d.niy * B;
  auto at = [](const T *p, unsigned o) -> T { return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + o); };
  auto put = [](T *p, unsigned o, T x) { *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + o) = x; };
  auto load = [&](int r, DynRow<T> &w) {
    const unsigned rr = (unsigned)(min(r, d.jed) - d.jsd);
    const unsigned o = rr * rc + lc, ou = rr * rf + lf;
    w.p = at(dl, o);
    w.u = at(u, ou);
    w.dxa = at(dxa, o);
    w.sg0 = at(sg, o);
    w.sg2 = at(sg2, o);
    w.area = at(area, o);
    w.dy = at(dy, o + rr * B);
    const unsigned of2 = (unsigned)(max(r - 2, d.jsd) - d.jsd) * rc + lc;  // r-2 <= je+1
    const unsigned f = (unsigned)(min(max(r - 2, d.js), d.je + 1) - d.js), ov = f * rc + lc;
    w.v = at(v, ov);
    w.dx = at(dx, of2);
    w.dya = at(dya, of2);
    w.sg1 = at(sg1, of2);
    w.sg3 = at(sg3, of2);
    const unsigned j = (unsigned)(min(max(r - 3, d.js), d.je) - d.js), oj = (j + (unsigned)(d.js - d.jsd)) * rc + lc;
    w.areaj = at(area, oj);
    w.rarea = at(rarea, oj);
    if (!first) {
      w.cx = at(cx, ou);
      w.cy = at(cy, ov);
      w.mfy = at(mfy, f * rm + lm);
      w.mfx = at(mfx, j * rf + lf);
    }
  };
  // flux through x-face i of the row whose cells (and spacings dr) the lanes hold
  auto x_flux = [&](auto edge, T q, T c, T dr, int iord) -> T {
    constexpr bool XE = decltype(edge)::value;
    const T qm = left(q), qp = right(q), qmm = left(qm);
    const T dm = slope<T>(qm, q, qp), dml = left(dm);
    T al = face<T>(qm, q, dml, dm), bl, br;
    if constexpr (XE) {
      const T d1 = left(dr), e = edge_face<T>(qmm, qm, q, qp, left(d1), d1, dr, right(dr));
      al = x_face == 1 ? e
           : x_face == 2 ? K<T>::s15 * qm + K<T>::s11 * q - K<T>::s14 * dm
           : x_face == 3 ? K<T>::s15 * q + K<T>::s11 * qm + K<T>::s14 * dml : al;
    }
    const T ar = right(al);
    inner_cell<O8, T>(Win5<T>{{qmm, qm, q, qp, right(qp)}}, dm, al, ar, iord, bl, br);
    if constexpr (XE) {
      const T dmr = right(dm);
      if (x_place) edge_cell<T>(x_place, qm, q, qp, al, ar, dml, dmr, bl, br);
    }
    return upwind<T>(c, qm, left(bl), left(br), q, bl, br);
  };

  auto rows = [&](auto edge) {  // edge: the strip holds columns of a cube edge
    DynRow<T> w, nx;
    w.cx = w.cy = w.mfx = w.mfy = T(0);
    nx = w;
    YLine<T, O8> yp{}, yq{};                         // delp, q_j
    T c1 = T(0), c2 = T(0), c3 = T(0);               // x-Courant numbers of rows r-1, r-2, r-3
    T x1 = T(0), x2 = T(0), x3 = T(0);               // their area fluxes
    T e1 = T(0), e2 = T(0), e3 = T(0);               // their inner x-fluxes
    T d1 = T(1), d2 = T(1), d3 = T(1);               // their spacings
    T dya_m = T(0), sg3_m = T(0);                    // of cell row f-1
    T yf_m = T(0), fyi_m = T(0), fy_m = T(0);        // area flux, inner and total flux of face f-1
    load(j0 - 3, nx);
    for (int r = j0 - 3; r <= j1 + 3; r++) {
      w = nx;
      if (r < j1 + 3) load(r + 1, nx);
      // ---- row r
      T py = w.p, px = w.p;
      if (corner_strip && (r <= 0 || r >= d.npy)) {
        int si, sj;
        if (corner_src(i, r, d.npx, d.npy, 2, d.corners, si, sj)) py = dl[(sj - d.jsd) * d.nid + (si - d.isd)];
        if (corner_src(i, r, d.npx, d.npy, 1, d.corners, si, sj)) px = dl[(sj - d.jsd) * d.nid + (si - d.isd)];
      }
      const bool own_y = r >= j0 && r <= j1;
      const bool own_yh = own_y || (r < d.js && j0 == d.js) || (r > d.je && j1 == d.je);
      const bool upl = w.u > T(0);
      const T da_l = left(w.dxa), sg_l = left(w.sg2);
      const T dax = upl ? da_l : w.dxa;
      const T c0 = bdt * w.u / dax;
      const T x0 = c0 * dax * w.dy * (upl ? sg_l : w.sg0);
      const T e0 = x_flux(edge, px, c0, w.dxa, a.ord_in);
      const T fa = x0 * e0, xr = right(x0), fb = right(fa);
      const T qj = (px * w.area + fa - fb) / (w.area + x0 - xr);
      // ---- cell row r-2 of the y-lines, y-face f = r-2
      auto spacing = [&]() {
        Win5<T> s;
#pragma unroll
        for (int k = 0; k < 4; k++) s.v[k] = dya[(r - 3 + k - d.jsd) * d.nid + oc];
        s.v[4] = s.v[3];
        return s;
      };
      yp.add(py, gy, r, spacing, a.ord_in);
      yq.add(qj, gy, r, spacing, a.ord_ou);
      const int f = r - 2, j = r - 3;
      T cr = T(0), fy = T(0), fx = T(0), dp = T(0);
      if (f >= j0) {
        const bool up = w.v > T(0);
        const T day = up ? dya_m : w.dya;
        cr = bdt * w.v / day;
        const T yf = cr * day * w.dx * (up ? sg3_m : w.sg1);
        const T fyi = yp.flux(cr);
        fy = T(0.5) * (yq.flux(cr) + fyi) * yf;
        // ---- row j = r-3: q_i, the outer x-sweep, delp
        const T qi = (yp.q(1) * w.areaj + yf_m * fyi_m - yf * fyi) / (w.areaj + yf_m - yf);
        fx = T(0.5) * (x_flux(edge, qi, c3, d3, a.ord_ou) + e3) * x3;
        dp = yp.q(1) + ((fx - right(fx)) + (fy_m - fy)) * w.rarea;
        yf_m = yf;
        fyi_m = fyi;
        fy_m = fy;
      }
      dya_m = w.dya;
      sg3_m = w.sg3;
      c3 = c2;
      c2 = c1;
      c1 = c0;
      x3 = x2;
      x2 = x1;
      x1 = x0;
      e3 = e2;
      e2 = e1;
      e1 = e0;
      d3 = d2;
      d2 = d1;
      d1 = w.dxa;
      // ---- results.  The wait for the next row's loads is put here: after the
      // stores it would include them, since both are counted in order
      const T cxv = w.cx + c0, cyv = w.cy + cr, mxv = w.mfx + fx, myv = w.mfy + fy;
      nx.arrived();
      const bool own_f = f >= j0 && (f <= j1 || (f == d.je + 1 && j1 == d.je));
      if (own_yh && own_xf) put(cx, (unsigned)(r - d.jsd) * rf + lf, cxv);
      if (own_yh && own_xh && !(own_y && i >= d.is && i <= d.ie)) put(dw, (unsigned)(r - d.jsd) * rc + lc, px);
      if (own_f) {
        if (own_xh) put(cy, (unsigned)(f - d.js) * rc + lc, cyv);
        if (own_x) put(mfy, (unsigned)(f - d.js) * rm + lm, myv);
      }
      if (j >= j0) {
        if (own_xf) put(mfx, (unsigned)(j - d.js) * rf + lf, mxv);
        if (own_x) put(dw, (unsigned)(j - d.jsd) * rc + lc, dp);
      }
    }
  };
  if (x_edge)
    rows(std::true_type{});
  else
    rows(std::false_type{});
}

// Rows per block: longer blocks repeat fewer of the six rows that a block
// shares with its neighbours, shorter ones give more waves.  Waves that all fit
// at once take the time of one; beyond that the last ones to start add half a
// block's time on average.
int dyn_rows(int nj, long long lines, long long slots) {
  int best = 48;
  double least = 0.0;
  for (int rows = 48; rows >= 4; rows -= 4) {
    const double x = (double)(lines * ((nj + rows - 1) / rows)) / (double)slots;
    const double t = (rows + 6) * (x <= 1.0 ? 1.0 : x + 0.5);
    if (rows == 48 || t < least) {
      least = t;
      best = rows;
    }
  }
  return best;
}

}  // namespace

template <typename T>
static int dyn_core_fluxes(Ctx &c, int n_split, T bdt, int hord, const T *uc, const T *vc, T *delp, T *dp1,
                           T *cx, T *cy, T *mfx, T *mfy, hipStream_t s) {
  const Dims d = c.d;
  const int npz = c.npz, nt = c.ntiles, nz = npz * nt;
  const GridDev<T> g = grid_of<T>(c);
  const int ord_in = hord == 10 ? 8 : hord, ord_ou = hord;
  const long long sz = nz;
  size_t off = 0;
  auto take = [&](long long n) {
    const size_t o = off;
    off += ((size_t)n * sizeof(T) + 255) & ~(size_t)255;
    return o;
  };
  const size_t o_crx = take(d.sx * sz), o_xfx = take(d.sx * sz), o_cry = take(d.sy * sz), o_yfx = take(d.sy * sz);
  const size_t o_rax = take(d.srx * sz), o_ray = take(d.sry * sz), o_fx = take(d.smx * sz), o_fy = take(d.smy * sz);
  const size_t o_fy2 = take(d.sy * sz), o_qi = take(d.sry * sz), o_fx2 = take(d.sx * sz), o_qj = take(d.srx * sz);
  char *base = (char *)ctx_scratch(c, off);
  if (!base) return 1;
  T *crx = (T *)(base + o_crx), *xfx = (T *)(base + o_xfx), *cry = (T *)(base + o_cry), *yfx = (T *)(base + o_yfx);
  T *rax = (T *)(base + o_rax), *ray = (T *)(base + o_ray), *fx = (T *)(base + o_fx), *fy = (T *)(base + o_fy);
  T *t_fy2 = (T *)(base + o_fy2), *t_qi = (T *)(base + o_qi), *t_fx2 = (T *)(base + o_fx2), *t_qj = (T *)(base + o_qj);

  FV3_HIP(hipMemcpyAsync(dp1, delp, sizeof(T) * d.s2 * sz, hipMemcpyDeviceToDevice, s));
  const long long gs2 = g.s2, gdx = g.sdx, gdy = g.sdy;
  const T *dxa = g.dxa, *dya = g.dya, *gdxp = g.dx, *gdyp = g.dy, *sg = g.sin_sg, *area = g.area,
          *rarea = g.rarea;
  const LineGeom gx{d.is, d.ie, d.npx, d.edge}, gy{d.js, d.je, d.npy, d.edge};
  const unsigned corners = d.corners;
  auto cc = [&](int dir) {
    if (d.bounded) return 0;
    return launch_rect(s, [=] __device__(int cidx, int, int z) {
          T *w = delp + (long long)z * d.s2;
          const int blk = cidx / 9, k9 = cidx % 9;
          const int i = (blk == 0 || blk == 3 ? 1 - NG : d.npx) + k9 % 3;
          const int j = (blk == 0 || blk == 1 ? 1 - NG : d.npy) + k9 / 3;
          int si, sj;
          if (corner_src(i, j, d.npx, d.npy, dir, corners, si, sj))
            w[(long long)(j - d.jsd) * d.nid + (i - d.isd)] = w[(long long)(sj - d.jsd) * d.nid + (si - d.isd)];
        }, 0, 35, 0, 0, nz);
  };

  for (int it = 0; it < n_split; it++) {
    const T *u = uc + (long long)it * sz * d.sx, *v = vc + (long long)it * sz * d.sy;
    const bool first = it == 0;
    // Courant numbers and area fluxes with the upwind metric; cx, cy accumulate
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const long long lv = (long long)z * d.sx + (long long)(j - d.jsd) * d.nix + (i - d.is);
          const T w = u[lv];
          const int iu = w > T(0) ? i - 1 : i;
          const long long m = tile * gs2 + (long long)(j - d.jsd) * d.nid + (iu - d.isd);
          const T cr = bdt * w / dxa[m];
          crx[lv] = cr;
          xfx[lv] = cr * dxa[m] * gdyp[tile * gdy + (long long)(j - d.jsd) * (d.nid + 1) + (i - d.isd)] *
                    sg[tile * 9 * gs2 + (w > T(0) ? 2 : 0) * gs2 + (long long)(j - d.jsd) * d.nid + (iu - d.isd)];
          cx[lv] = first ? T(0) + cr : cx[lv] + cr;
        }, d.is, d.ie + 1, d.jsd, d.jed, nz))
      return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const long long lv = (long long)z * d.sy + (long long)(j - d.js) * d.nid + (i - d.isd);
          const T w = v[lv];
          const int ju = w > T(0) ? j - 1 : j;
          const long long m = tile * gs2 + (long long)(ju - d.jsd) * d.nid + (i - d.isd);
          const T cr = bdt * w / dya[m];
          cry[lv] = cr;
          yfx[lv] = cr * dya[m] * gdxp[tile * gdx + (long long)(j - d.jsd) * d.nid + (i - d.isd)] *
                    sg[tile * 9 * gs2 + (w > T(0) ? 3 : 1) * gs2 + (long long)(ju - d.jsd) * d.nid + (i - d.isd)];
          cy[lv] = first ? T(0) + cr : cy[lv] + cr;
        }, d.isd, d.ied, d.js, d.je + 1, nz))
      return 1;
    // ra_x, ra_y
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const T *xk = xfx + (long long)z * d.sx + (long long)(j - d.jsd) * d.nix;
          rax[(long long)z * d.srx + (long long)(j - d.jsd) * d.niy + (i - d.is)] =
              area[tile * gs2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)] + xk[i - d.is] - xk[i + 1 - d.is];
        }, d.is, d.ie, d.jsd, d.jed, nz))
      return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const T *yk = yfx + (long long)z * d.sy;
          ray[(long long)z * d.sry + (long long)(j - d.js) * d.nid + (i - d.isd)] =
              area[tile * gs2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)] +
              yk[(long long)(j - d.js) * d.nid + (i - d.isd)] - yk[(long long)(j + 1 - d.js) * d.nid + (i - d.isd)];
        }, d.isd, d.ied, d.js, d.je, nz))
      return 1;
    // fv_tp_2d of delp
    if (cc(2)) return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          ColQ<T> qa{delp + (long long)z * d.s2 + (i - d.isd), d.jsd, d.nid};
          ColQ<T> da{dya + tile * gs2 + (i - d.isd), d.jsd, d.nid};
          const long long lv = (long long)z * d.sy + (long long)(j - d.js) * d.nid + (i - d.isd);
          t_fy2[lv] = ppm_flux<T>(qa, da, j, cry[lv], gy, ord_in);
        }, d.isd, d.ied, d.js, d.je + 1, nz))
      return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const T *yk = yfx + (long long)z * d.sy, *f2 = t_fy2 + (long long)z * d.sy;
          const T fa = yk[(long long)(j - d.js) * d.nid + (i - d.isd)] * f2[(long long)(j - d.js) * d.nid + (i - d.isd)];
          const T fb = yk[(long long)(j + 1 - d.js) * d.nid + (i - d.isd)] * f2[(long long)(j + 1 - d.js) * d.nid + (i - d.isd)];
          t_qi[(long long)z * d.sry + (long long)(j - d.js) * d.nid + (i - d.isd)] =
              (delp[(long long)z * d.s2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)] *
                   area[tile * gs2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)] + fa - fb) /
              ray[(long long)z * d.sry + (long long)(j - d.js) * d.nid + (i - d.isd)];
        }, d.isd, d.ied, d.js, d.je, nz))
      return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          RowQ<T> qa{t_qi + (long long)z * d.sry + (long long)(j - d.js) * d.nid, d.isd};
          RowQ<T> da{dxa + tile * gs2 + (long long)(j - d.jsd) * d.nid, d.isd};
          const T cv = crx[(long long)z * d.sx + (long long)(j - d.jsd) * d.nix + (i - d.is)];
          fx[(long long)z * d.smx + (long long)(j - d.js) * d.nix + (i - d.is)] = ppm_flux<T>(qa, da, i, cv, gx, ord_ou);
        }, d.is, d.ie + 1, d.js, d.je, nz))
      return 1;
    if (cc(1)) return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          RowQ<T> qa{delp + (long long)z * d.s2 + (long long)(j - d.jsd) * d.nid, d.isd};
          RowQ<T> da{dxa + tile * gs2 + (long long)(j - d.jsd) * d.nid, d.isd};
          const long long lv = (long long)z * d.sx + (long long)(j - d.jsd) * d.nix + (i - d.is);
          t_fx2[lv] = ppm_flux<T>(qa, da, i, crx[lv], gx, ord_in);
        }, d.is, d.ie + 1, d.jsd, d.jed, nz))
      return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const T *xk = xfx + (long long)z * d.sx + (long long)(j - d.jsd) * d.nix;
          const T *f2 = t_fx2 + (long long)z * d.sx + (long long)(j - d.jsd) * d.nix;
          const T fa = xk[i - d.is] * f2[i - d.is];
          const T fb = xk[i + 1 - d.is] * f2[i + 1 - d.is];
          t_qj[(long long)z * d.srx + (long long)(j - d.jsd) * d.niy + (i - d.is)] =
              (delp[(long long)z * d.s2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)] *
                   area[tile * gs2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)] + fa - fb) /
              rax[(long long)z * d.srx + (long long)(j - d.jsd) * d.niy + (i - d.is)];
        }, d.is, d.ie, d.jsd, d.jed, nz))
      return 1;
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          ColQ<T> qa{t_qj + (long long)z * d.srx + (i - d.is), d.jsd, d.niy};
          ColQ<T> da{dya + tile * gs2 + (i - d.isd), d.jsd, d.nid};
          const T cv = cry[(long long)z * d.sy + (long long)(j - d.js) * d.nid + (i - d.isd)];
          fy[(long long)z * d.smy + (long long)(j - d.js) * d.niy + (i - d.is)] = ppm_flux<T>(qa, da, j, cv, gy, ord_ou);
        }, d.is, d.ie, d.js, d.je + 1, nz))
      return 1;
    // flux averaging with the area fluxes; mfx, mfy accumulate
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          if (i <= d.ie + 1 && j <= d.je) {
            const long long o = (long long)z * d.smx + (long long)(j - d.js) * d.nix + (i - d.is);
            const long long ox = (long long)z * d.sx + (long long)(j - d.jsd) * d.nix + (i - d.is);
            const T f = T(0.5) * (fx[o] + t_fx2[ox]) * xfx[ox];
            fx[o] = f;
            mfx[o] = first ? T(0) + f : mfx[o] + f;
          }
          if (i <= d.ie && j <= d.je + 1) {
            const long long o = (long long)z * d.smy + (long long)(j - d.js) * d.niy + (i - d.is);
            const long long oy = (long long)z * d.sy + (long long)(j - d.js) * d.nid + (i - d.isd);
            const T f = T(0.5) * (fy[o] + t_fy2[oy]) * yfx[oy];
            fy[o] = f;
            mfy[o] = first ? T(0) + f : mfy[o] + f;
          }
        }, d.is, d.ie + 1, d.js, d.je + 1, nz))
      return 1;
    // delp by the flux divergence
    if (launch_rect(s, [=] __device__(int i, int j, int z) {
          const int tile = z / npz;
          const T *fxr = fx + (long long)z * d.smx + (long long)(j - d.js) * d.nix;
          const T *fyc = fy + (long long)z * d.smy;
          T &p = delp[(long long)z * d.s2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)];
          p = p + ((fxr[i - d.is] - fxr[i + 1 - d.is]) +
                   (fyc[(long long)(j - d.js) * d.niy + (i - d.is)] - fyc[(long long)(j + 1 - d.js) * d.niy + (i - d.is)])) *
                      rarea[tile * gs2 + (long long)(j - d.jsd) * d.nid + (i - d.isd)];
        }, d.is, d.ie, d.js, d.je, nz))
      return 1;
    if (nt > 1 && it + 1 < n_split)
      if (halo_fill<T>(c, delp, (long long)npz * d.s2, nullptr, 0, npz)) return 1;
  }
  return 0;
}

// The sub-steps of dyn_core_fluxes, one launch each (plus the six-face halo
// refresh between them); delp alternates between the caller's array and a
// scratch copy and ends in the caller's.
template <typename T>
static int dyn_core_fluxes_fused(Ctx &c, int n_split, T bdt, int hord, const T *uc, const T *vc, T *delp, T *dp1,
                                 T *cx, T *cy, T *mfx, T *mfy, hipStream_t s) {
  const Dims d = c.d;
  const int npz = c.npz, nt = c.ntiles, nz = npz * nt;
  const GridDev<T> g = grid_of<T>(c);
  const long long slab = (long long)d.s2 * nz;
  T *alt = (T *)ctx_scratch(c, sizeof(T) * slab);
  if (!alt) return 1;
  FV3_HIP(hipMemcpyAsync(dp1, delp, sizeof(T) * slab, hipMemcpyDeviceToDevice, s));
  DynSubArgs a{};
  a.d = d;
  a.npz = npz;
  a.nz = nz;
  a.ord_in = hord == 10 ? 8 : hord;
  a.ord_ou = hord;
  a.gs2 = g.s2;
  a.gdx = g.sdx;
  a.gdy = g.sdy;
  const int ni = d.ie - d.is + 1, nj = d.je - d.js + 1;
  const int strips = (ni + DYN_W - 1) / DYN_W;
  // waves on the chip at once: two per SIMD by registers in FP64, four in FP32
  a.rows = dyn_rows(nj, (long long)strips * nz, 1024 * (sizeof(T) == 8 ? 2 : 4));
  const dim3 grid((unsigned)((nz + 3) / 4), (unsigned)strips, (unsigned)((nj + a.rows - 1) / a.rows));
  T *buf[2] = {delp, alt};
  for (int it = 0; it < n_split; it++) {
    a.first = it == 0;
    const T *u = uc + (long long)it * nz * d.sx, *v = vc + (long long)it * nz * d.sy;
    T *din = buf[it & 1], *dout = buf[(it + 1) & 1];
    if (hord == 8 || hord == 11)
      hipLaunchKernelGGL((k_dyn_sub<T, true>), grid, dim3(256), 0, s, a, g, bdt, u, v, din, dout, cx, cy, mfx, mfy);
    else
      hipLaunchKernelGGL((k_dyn_sub<T, false>), grid, dim3(256), 0, s, a, g, bdt, u, v, din, dout, cx, cy, mfx, mfy);
    FV3_HIP(hipGetLastError());
    if (nt > 1 && it + 1 < n_split)
      if (halo_fill<T>(c, dout, (long long)npz * d.s2, nullptr, 0, npz)) return 1;
  }
  if (n_split & 1) FV3_HIP(hipMemcpyAsync(delp, alt, sizeof(T) * slab, hipMemcpyDeviceToDevice, s));
  return 0;
}

}  // namespace fv3

using namespace fv3;

extern "C" int fv3_dyn_core_fluxes(fv3_ctx *h, int form, int n_split, double bdt, int hord_dp, const void *uc,
                                   const void *vc, void *delp, void *dp1, void *cx, void *cy, void *mfx, void *mfy,
                                   void *stream) {
  if (!h || !uc || !vc || !delp || !dp1 || !cx || !cy || !mfx || !mfy)
    return set_error("fv3_dyn_core_fluxes: NULL argument");
  if (n_split < 1) return set_error("n_split must be >= 1 (got %d)", n_split);
  if (hord_dp < 7 || hord_dp > 13) return set_error("hord_dp=%d: only the monotone orders 7..13 are implemented", hord_dp);
  if (!(bdt > 0.0)) return set_error("bdt must be > 0 (got %g)", bdt);
  if (delp == dp1) return set_error("fv3_dyn_core_fluxes: delp and dp1 must be distinct arrays");
  Ctx &c = h->c;
  std::lock_guard<std::mutex> lk(c.mu);
  if (!c.grid_set) return set_error("grid metrics not set (fv3_ctx_set_grid)");
  // the context's stream for the call: halo_fill launches there
  hipStream_t saved = c.stream;
  if (stream) c.stream = (hipStream_t)stream;
  hipStream_t s = c.stream;
  int rc;
  if (form == FV3_FORM_PLAIN64)
    rc = dyn_core_fluxes<double>(c, n_split, bdt, hord_dp, (const double *)uc, (const double *)vc, (double *)delp,
                                 (double *)dp1, (double *)cx, (double *)cy, (double *)mfx, (double *)mfy, s);
  else if (form == FV3_FORM_FUSED64)
    rc = dyn_core_fluxes_fused<double>(c, n_split, bdt, hord_dp, (const double *)uc, (const double *)vc,
                                       (double *)delp, (double *)dp1, (double *)cx, (double *)cy, (double *)mfx,
                                       (double *)mfy, s);
  else if (form == FV3_FORM_FUSED32)
    rc = dyn_core_fluxes_fused<float>(c, n_split, (float)bdt, hord_dp, (const float *)uc, (const float *)vc,
                                      (float *)delp, (float *)dp1, (float *)cx, (float *)cy, (float *)mfx,
                                      (float *)mfy, s);
  else
    rc = set_error("form %d: the dyn_core fluxes run FV3_FORM_PLAIN64 or FV3_FORM_FUSED64 (double), "
                   "FV3_FORM_FUSED32 (float)", form);
  c.stream = saved;
  if (rc) return 1;
  FV3_HIP(hipStreamSynchronize(s));
  return 0;
}
