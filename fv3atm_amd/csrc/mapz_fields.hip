// mapz_fields.hip -- vertical remap (upstream fv_mapz.F90: cs_profile /
// scalar_profile, cs_limiters, and the layer integrals of map1_ppm, map1_q2,
// map_scalar and mapn_tracer) in upstream evaluation order, for the FP64
// forms, the full Lagrangian_to_Eulerian and the tangent-linear step.
//
// What depends on a column's pressures alone -- the elimination factors of
// the interface solve, the source layers and fractions of every target
// interface -- is the same for every field of the column: k_fields_prep
// computes it once per column into [level][column] tables, and k_fields runs
// one thread per (column, field).  The solve, the limiters and the layer
// sums of a column are sequential in upstream's order, so that FP64 results
// equal a CPU FP64 evaluation bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fv3_internal.h"
#include "mapz_fields.h"
#include "mapz_prep.h"
#include "quot.h"

namespace fv3 {

namespace {

struct PrepGeo {
  int km, ni, nj, ncb, is, js, isd, jsd, nid, cni;  // cni: cells along i (the pe array's rows are cni + 2)
  long long ncol, ncols, s2, spe;
};

// One workgroup per 64 columns.  Every level's thickness is loaded at once and
// the interfaces are kept in LDS; then wave 0 runs the elimination's chain
// (the quotients off the chain four levels at a time) while the other waves
// take the target layers, each independent of the others: the source layer of
// an interface is the first that ends at or below it, walked to from the layer
// of its own number.  A column whose interfaces are out of order (its flag is
// set in passing) keeps upstream's search from the last layer found instead,
// on one lane.  Against one wave for the chain and one for the search in
// sequence: C384 L127 FP64 759 -> 451 us, the four tables of a C192 L127 FP32
// full remap 999 -> 413 us.
template <typename R>
__global__ void __launch_bounds__(64 * PREP_WAVES) k_fields_prep(const PrepGeo g, const ColSource s,
                                                                 const ColTab<R> tab, const bool iv2) {
  extern __shared__ double pe1_lds[];  // [km + 1][64]
  __shared__ int bad[64], win;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = (int)blockIdx.x / g.ncb, cb = (int)blockIdx.x % g.ncb;
  const int km = g.km;  // at most FIELDS_MAX_KM: 64 columns fit
  const long long c0 = (long long)cb * 64 + lane;
  const bool act = c0 < g.ncol;
  const long long lc = act ? c0 : g.ncol - 1;  // lanes past the last column repeat it and store nothing
  const int ii = (int)((unsigned)lc % (unsigned)g.ni), jj = (int)((unsigned)lc / (unsigned)g.ni);
  const int i = g.is + ii, j = g.js + jj;
  const long long cell = (long long)(j - g.jsd) * g.nid + (i - g.isd);
  const long long col = tile * g.ncol + lc, nc = g.ncols;
  const ColPe P{pe1_lds + lane, 64};
  if (wave == 0) {
    bad[lane] = 0;
    win = 0;
  }
  double psl = 0.0;  // kinds 1, 2: the sum of the two cells' surface pressures
  if (s.kind == 0) {
    stage_interfaces(P, km, s.ptop, s.delp + (long long)tile * km * g.s2 + cell, g.s2, wave);
  } else {
    const double *pe = s.pe + tile * g.spe, *ps = s.ps + tile * g.s2;
    const int w = g.cni + 2;
    auto at = [&](int a, int k, int b) {
      return pe[((long long)(b - (g.js - 1)) * (km + 1) + (k - 1)) * w + (a - (g.is - 1))];
    };
    const int di = s.kind == 2 ? 1 : 0, dj = 1 - di;
    for (int k = 1 + wave; k <= km + 1; k += PREP_WAVES) P(k) = 0.5 * (at(i - di, k, j - dj) + at(i, k, j));
    psl = ps[cell - (di ? 1 : g.nid)] + ps[cell];
  }
  __syncthreads();
  const double pbot = P(km + 1);
  auto PE2 = [&](int k) -> double {
    if (s.kind == 0) return k == 1 ? s.ptop : (k == km + 1 ? pbot : s.ak[k - 1] + s.bk[k - 1] * pbot);
    return s.ak[k - 1] + 0.5 * s.bk[k - 1] * psl;
  };
  // columns in order: pe1 increasing, pe2 not decreasing and within pe1
  {
    bool b = false;
    for (int k = 1 + wave; k <= km; k += PREP_WAVES) b = b || !(P(k + 1) > P(k)) || !(PE2(k + 1) >= PE2(k));
    b = b || !(PE2(1) >= P(1)) || !(PE2(km + 1) <= pbot);
    if (b) bad[lane] = 1;
  }
  __syncthreads();
  if (wave == 0) {
    // the interface solve's factors
    auto put = [&](int k, R d, R bt, R gg) {
      if (act) tab.el[(long long)(k - 1) * nc + col] = Elim<R>{d, bt, R(1) / bt, gg};
    };
    double dprev = P(2) - P(1);
    if (act) tab.d1[col] = dprev;
    R gp, bot0 = R(0), bot1 = R(0), bot2 = R(1);
    if (iv2) {
      gp = R(0.5);  // G(2)
      put(1, R(0), R(1), gp);
    } else {
      const R grat = R((P(3) - P(2)) / dprev);
      const R bet = grat * (grat + R(0.5));
      gp = (R(1) + grat * (grat + R(1.5))) / bet;
      put(1, (grat + grat) * (grat + R(1)), bet, gp);
    }
    R d4 = R(0);
    for (int k4 = 2; k4 <= km; k4 += 4) {
      double dk[4];
      R rat[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int k = min(k4 + m, km);
        dk[m] = P(k + 1) - P(k);
        rat[m] = R((m == 0 ? dprev : dk[m - 1]) / dk[m]);
      }
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int k = k4 + m;
        if (k > km) break;
        if (act) tab.d1[(long long)(k - 1) * nc + col] = dk[m];
        d4 = rat[m];
        const R bt = R(2) + d4 + d4 - gp;
        gp = d4 / bt;
        put(k, iv2 ? R(1) : d4, bt, iv2 && k == km ? R(0) : gp);
      }
      dprev = dk[3];
    }
    if (iv2) {
      bot0 = d4;
    } else {
      const R a_bot = R(1) + d4 * (d4 + R(1.5));
      bot0 = R(2) * d4 * (d4 + R(1));
      bot1 = a_bot;
      bot2 = d4 * (d4 + R(0.5)) - a_bot * gp;
    }
    if (act) {
      tab.bot[col] = bot0;
      tab.bot[nc + col] = bot1;
      tab.bot[2 * nc + col] = bot2;
    }
  }
  // the target layers
  double *dout = s.delp_out ? s.delp_out + (long long)tile * km * g.s2 + cell : nullptr;
  auto put = [&](int k, int lt, int lb, bool one, double pl, double pr, double dt, double db, double den) {
    if (!act) return;
    const long long o = (long long)(k - 1) * nc + col;
    tab.r0[o] = make_double2(pl, pr);
    tab.r1[o] = make_double2(dt, db);
    tab.r2[o] = make_double2(den, 1.0 / den);
    tab.rc[o] = lt | lb << 12 | (one ? 1 << 24 : 0);
    if (dout) dout[(long long)(k - 1) * g.s2] = den;
  };
  if (wave > 0 && !bad[lane]) {
    int w = 0;  // source layers that one target layer of the block's columns takes in, at most
    for (int k = wave; k <= km; k += PREP_WAVES - 1) {
      const double pa = PE2(k), pb = PE2(k + 1);
      const int lt = P.layer_of(pa, k, km), lb = P.layer_of(pb, k, km);
      const double a = P(lt), b = P(lt + 1), c = P(lb);
      const bool one = lt == lb;
      const double db = pb - c;
      put(k, lt, lb, one, (pa - a) / (b - a), db / (P(lb + 1) - c), one ? 0.0 : b - pa, one ? 0.0 : db, pb - pa);
      int lo = __builtin_amdgcn_readfirstlane(lt), hi = __builtin_amdgcn_readfirstlane(lb);
      for (unsigned long long m; (m = __ballot(lt < lo)) != 0;) lo = __builtin_amdgcn_readlane(lt, __builtin_ctzll(m));
      for (unsigned long long m; (m = __ballot(lb > hi)) != 0;) hi = __builtin_amdgcn_readlane(lb, __builtin_ctzll(m));
      w = max(w, hi - lo + 1);
    }
    atomicMax(&win, w);
  } else if (wave > 0) {
    atomicMax(&win, NO_WINDOW);
  }
  if (wave == 1 && bad[lane]) {  // upstream's search
    int k0 = 1;
    double pa = PE2(1);
    for (int k = 1; k <= km; k++) {
      const double pb = PE2(k + 1);
      int lt = 0, lb = km + 1;
      bool one = false;
      double pl = 0.0, pr = 0.0, dt = 0.0, db = 0.0;
      for (int l = k0; l <= km; l++) {
        const double a = P(l), b = P(l + 1);
        if (pa >= a && pa <= b) {
          lt = l;
          pl = (pa - a) / (b - a);
          if (pb <= b) {
            one = true;
            pr = (pb - a) / (b - a);
            k0 = lb = l;
            break;
          }
          dt = b - pa;
          for (int m = l + 1; m <= km; m++)
            if (!(pb > P(m + 1))) {
              db = pb - P(m);
              pr = db / (P(m + 1) - P(m));
              k0 = lb = m;
              break;
            }
          break;
        }
      }
      put(k, lt, lb, one, pl, pr, dt, db, pb - pa);
      pa = pb;
    }
  }
  __syncthreads();
  if (wave == 0 && act) tab.win[col] = win;
}

// The target thickness from the tables, one thread per cell and level, by itself: a
// step submits it behind the tables, which need not wait for the counts (with the
// tables behind the counts a C96 L64 FP64 step took 525 us against 436).
__global__ void __launch_bounds__(256) k_fields_target(const double2 *r2, const double *dp1, double *out, Dims d, int km,
                                                       long long ncols, StepCounts counts) {
  if (!__syncthreads_or(counts.any(threadIdx.x, 256))) return;
  const int c = (int)(blockIdx.x * 256 + threadIdx.x), i = c % d.nid + d.isd, j = c / d.nid + d.jsd;
  if (j > d.jed) return;
  const int k = blockIdx.y, tile = blockIdx.z, ni = d.ie - d.is + 1, nj = d.je - d.js + 1;
  const long long o = ((long long)tile * km + k) * d.s2 + c;
  if (i < d.is || i > d.ie || j < d.js || j > d.je)
    out[o] = dp1[o];
  else
    out[o] = r2[k * ncols + (long long)tile * ni * nj + (long long)(j - d.js) * ni + (i - d.is)].x;
}

// ---- the field kernel
constexpr int FD_B = 8;      // levels per regenerated block
constexpr int FD_WAVES = 4;  // fields per workgroup (one per wave)
// source cells kept in LDS for the targets: over 64 neighbouring columns a target
// took in three to five, at most, where thicknesses vary by 5 % in waves and 10 %
// from cell to cell, and a sixth cell would cost 1.5 KB more per FP64 wave; a block
// that needs more walks column by column.  Fewer for (value, tangent) pairs, whose
// cells are twice as large.
template <typename T>
constexpr int FD_RING = sizeof(T) > 8 ? 4 : 5;
// LDS rows of 64 values per wave: block ends, a block's interface values, and
// three coefficients per kept cell
template <typename T>
__host__ __device__ constexpr int fd_rows(int nb) {
  return nb + FD_B + 3 * FD_RING<T>;
}

struct TargetRec {
  double2 r0, r1, r2;
  int rc;
};

// One wave: 64 columns of one field.  Three passes over the levels:
//   down  the elimination; the entry value of every FD_B-level block to LDS;
//   up    each block's eliminated values again from its entry value, then
//         the back substitution; the block's exit value replaces the entry
//         value in LDS;
//   down  the eliminated values once more (their chain is carried), the block's
//         interface values by back substitution from its exit value, into LDS,
//         then level by level the interface limits, extremum flags, cell
//         limiters and layer integrals over a window of six cell means.
// The columns of a wave go through the target layers in lockstep: a cell's
// three coefficients go to a ring of FD_RING cells in LDS, and once the cell is
// done in which the target's bottom lies in every column, each column takes its
// pieces from the ring.  Records are loaded and results stored a whole level at
// a time.  A block where one target takes in more cells than the ring holds
// (tab.win) runs column by column instead, each with a target of its own: its
// scattered records and stores, and loops of several turns per level, were most
// of the time (C384 L127, 9 tracers + pt in FP64: 4.86 ms in that form, 3.75 in
// lockstep, 3.53 with the levels walked by adding to scalar bases and the waves
// dealt to (column block, field) pairs without gaps, 3.58 with sums divided for any
// operands; the full remap of C192 L127 in FP32, 13 fields: 1.85, 1.65, 1.44 ms).
// Only the block ends, one block and the ring are kept (20 KB of LDS per wave
// in FP64 at 127 levels: two waves per SIMD); the field's second and third
// reads come from cache.  The divisions by the field-independent pivots use
// their stored reciprocals (quot).  Bound by dependent FP64 operations at two
// waves per SIMD (VALU a third busy).  One thread per column looping over its
// fields with every work array in HBM (at C96 144 waves on 1024 SIMDs) took
// 18.7 ms for the C384 case, tables included (now 3.58 + 0.45), 1.79 ms for C96
// L64 4 tracers + pt (0.125 + 0.027), 12.4 ms for the FP32 remap (1.44 + 0.44).
template <typename T>
__global__ void __launch_bounds__(64 * FD_WAVES, sizeof(T) > 8 ? 1 : 2) k_fields(const FieldsArgs<T> a) {
  using R = typename RealOf<T>::type;
  extern __shared__ __align__(16) char fd_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // blocks are dealt round-robin to the 8 XCDs: renumber so that the fields
  // of one column block run on one XCD, one after another
  const unsigned bid = blockIdx.x, nx = 8, q8 = a.nwg / nx, r8 = a.nwg % nx;
  const unsigned xcd = bid % nx, idx = bid / nx;
  const unsigned logical = xcd < r8 ? xcd * (q8 + 1) + idx : r8 * (q8 + 1) + (xcd - r8) * q8 + idx;
  const unsigned job = logical * FD_WAVES + wave;
  const int cblk = (int)(job / (unsigned)a.nf), f = (int)(job % (unsigned)a.nf);
  if (cblk >= a.ncb * a.ntiles) return;  // whole wave; no barriers below
  int si = 0, fi = f;
  while (si + 1 < a.nset && fi >= a.set[si].count) fi -= a.set[si++].count;
  const FieldSet<T> &S = a.set[si];
  const int iv = S.iv, kord = a.kord[f], akord = kord < 0 ? -kord : kord;
  const bool use_qmin = S.use_qmin, mapn = S.mapn;
  const R qmin = S.qmin;
  const int tile = cblk / a.ncb, cb = cblk % a.ncb;
  const long long c0 = (long long)cb * 64 + lane;
  const bool act = c0 < a.ncol;
  const long long lc = act ? c0 : a.ncol - 1;
  const long long nc = a.ncols, col = tile * a.ncol + lc;
  const int km = a.km, nb = (km + FD_B - 1) / FD_B;
  const unsigned cell = (unsigned)((lc / a.ni) * S.ld + lc % a.ni);
  const long long fbase = fi * S.fstride + tile * S.tstride, sbase = fi * S.sfstride + tile * S.ststride;
  const R *src = S.src + sbase, *src_t = nullptr;
  if constexpr (sizeof(T) != sizeof(R)) src_t = S.src_t + sbase;
  const long long lev = S.lev;
  const unsigned cbyte = cell * (unsigned)sizeof(R);
  // scalar level bases, lane byte offsets; levels are walked by adding to the
  // bases (a 64-bit product per load was half of the scalar work)
  const long long levb = lev * (long long)sizeof(R), elb = nc * (long long)sizeof(Elim<R>);
  auto ldat = [&](long long o) -> T {  // o: (k - 1) levb
    const R v = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(src) + o + cbyte);
    if constexpr (sizeof(T) == sizeof(R)) {
      return v;
    } else {
      T r(v);
      r.d[0] = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(src_t) + o + cbyte);
      return r;
    }
  };
  auto ld = [&](int k) -> T { return ldat((k - 1) * levb); };
  const long long colu = tile * a.ncol + (long long)cb * 64;  // the block's first column
  const unsigned cl = (unsigned)(lc - (long long)cb * 64), ebyte = cl * (unsigned)sizeof(Elim<R>);
  T *lds = reinterpret_cast<T *>(fd_lds) + (size_t)wave * fd_rows<T>(nb) * 64 + lane;
  auto CP = [&](int b) -> T & { return lds[b * 64]; };
  auto BQ = [&](int j) -> T & { return lds[(nb + j) * 64]; };
  constexpr int NR = FD_RING<T>;
  T *ring = lds + (nb + FD_B) * 64;  // [NR][3][64]
  const bool iv2 = iv == -2;
  const T qs = iv2 ? T(S.qs[tile * a.ncol + lc]) : T(R(0));
  const R bot0 = a.tab.bot[col], bot1 = a.tab.bot[nc + col], bot2 = a.tab.bot[2 * nc + col];

  struct Blk {
    T av[FD_B + 1];  // a(k0-1 .. k0+B-1)
    Elim<R> e[FD_B];
  };
  auto fetch = [&](int b, Blk &x) {
    const int k0 = b * FD_B + 1;
    const char *e = reinterpret_cast<const char *>(a.tab.el + colu) + (k0 - 1) * elb;
    long long o = (k0 - 1) * levb;
    x.av[0] = ldat(b > 0 ? o - levb : o);
    if (k0 + FD_B - 1 <= km) {
#pragma unroll
      for (int j = 0; j < FD_B; j++) {
        x.av[j + 1] = ldat(o);
        x.e[j] = *reinterpret_cast<const Elim<R> *>(e + ebyte);
        o += levb;
        e += elb;
      }
    } else {
#pragma unroll
      for (int j = 0; j < FD_B; j++) {
        x.av[j + 1] = ldat(o);
        x.e[j] = *reinterpret_cast<const Elim<R> *>(e + ebyte);
        if (k0 + j < km) {
          o += levb;
          e += elb;
        }
      }
    }
  };
  // the eliminated values of block b from the one above it
  auto eliminate = [&](int b, const Blk &x, T q, T (&qv)[FD_B], const T &a2nd) {
    const int k0 = b * FD_B + 1;
    if (b > 0 && k0 + FD_B - 1 < km) {
#pragma unroll
      for (int j = 0; j < FD_B; j++)
        qv[j] = q = quot(R(3) * (x.av[j] + x.e[j].d4 * x.av[j + 1]) - q, x.e[j].bt, x.e[j].y);
      return q;
    }
#pragma unroll
    for (int j = 0; j < FD_B; j++) {
      const int k = k0 + j;
      if (k <= km) {
        if (k == 1) {
          q = iv2 ? R(1.5) * x.av[1] : quot(x.e[0].d4 * x.av[1] + a2nd, x.e[0].bt, x.e[0].y);
        } else {
          T n = R(3) * (x.av[j] + x.e[j].d4 * x.av[j + 1]);
          if (iv2 && k == km) {
            q = (n - bot0 * qs - q) / x.e[j].bt;  // the division: an infinite value reaches the rows above
          } else {
            q = quot(n - q, x.e[j].bt, x.e[j].y);
          }
        }
      }
      qv[j] = q;
    }
    return q;
  };
  // block b's interface values from the one below it: put(j, value)
  auto substitute = [&](int b, const Blk &x, T q, const T (&qv)[FD_B], auto put) {
    const int k0 = b * FD_B + 1;
    if (k0 + FD_B - 1 <= km) {
#pragma unroll
      for (int j = FD_B - 1; j >= 0; j--) put(j, q = qv[j] - x.e[j].g * q);
    } else {
#pragma unroll
      for (int j = FD_B - 1; j >= 0; j--)
        if (k0 + j <= km) put(j, q = qv[j] - x.e[j].g * q);
    }
    return q;
  };
  const T a2nd = ld(2);

  // ---- down: elimination
  T q = T(R(0));
  {
    Blk cur, nxt;
    fetch(0, cur);
    for (int b = 0; b < nb; b++) {
      if (b + 1 < nb) fetch(b + 1, nxt);
      CP(b) = q;
      T qv[FD_B];
      q = eliminate(b, cur, q, qv, a2nd);
      cur = nxt;
    }
  }
  const T qbot = iv2 ? qs : T((bot0 * ld(km) + ld(km - 1) - bot1 * q) / bot2);

  // ---- up: the value below every block
  {
    Blk cur, nxt;
    fetch(nb - 1, cur);
    q = iv2 ? T(R(0)) : qbot;  // iv = -2: the last row has no value below it (its factor is 0)
    for (int b = nb - 1; b >= 0; b--) {
      if (b > 0) fetch(b - 1, nxt);
      const T entry = CP(b);
      CP(b) = q;
      if (b > 0) {
        T qv[FD_B];
        eliminate(b, cur, entry, qv, a2nd);
        q = substitute(b, cur, q, qv, [](int, const T &) {});
      }
      cur = nxt;
    }
  }

  // ---- down: limits, cells, layer integrals
  const bool lim = akord <= 16;
  const T zero = T(R(0));
  T A_4 = zero, A_3 = zero, A_2 = zero, A_1 = zero, A_0 = zero, A_p = ld(1), A_n = a2nd;  // a(p-4 .. p+2)
  T L_2 = zero, L_1 = zero, L_0 = zero;                                      // limited Q(p-2 .. p)
  int E_3 = 0, E_2 = 0, E_1 = 0;                                             // flags of cells p-3 .. p-1
  auto recat = [&](long long o) -> TargetRec {  // o: 4 (k - 1) nc
    auto r = [&](const double2 *p) {
      return *reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(p + colu) + 4 * o + cl * 16);
    };
    return TargetRec{r(a.tab.r0), r(a.tab.r1), r(a.tab.r2),
                     *reinterpret_cast<const int *>(reinterpret_cast<const char *>(a.tab.rc + colu) + o + cl * 4)};
  };
  const long long nc4 = 4 * nc;
  auto rec = [&](int k) -> TargetRec { return recat((min(k, km) - 1) * nc4); };
  TargetRec tr = rec(1), tn = rec(2);  // the next two targets'
  using SumT = typename std::conditional<sizeof(T) == sizeof(R), double, D1>::type;  // sums in FP64
  auto wide = [](const T &v) -> SumT { return (SumT)v; };
  auto narrow = [](const SumT &v) -> T {
    if constexpr (sizeof(T) == sizeof(R)) return T(v);
    else return v;
  };
  auto ldd = [&](long long o) -> double {  // o: 8 (k - 1) nc
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a.tab.d1 + colu) + o + cl * 8);
  };
  double d1n = ldd(0);  // thickness of the next cell
  const double r3 = 1.0 / 3.0, r23 = 2.0 / 3.0;
  // pieces of a target in a cell's parabola: within one cell, from pl to the
  // cell's bottom, from its top to esl
  auto within = [&](const T &a2, const T &a3, const T &a4, double pl, double pr) -> T {
    const double z = pr * (pr + pl) + pl * pl;
    const T tail = mapn ? T(a4 * R(r3 * z)) : T(a4 * R(r3) * R(z));
    return a2 + (a4 + a3 - a2) * R(0.5 * (pr + pl)) - tail;
  };
  auto top_piece = [&](const T &a2, const T &a3, const T &a4, double pl, double dp) -> SumT {
    return dp * wide(a2 + (a4 + a3 - a2) * R(0.5 * (1.0 + pl)) - a4 * R(r3 * (1.0 + pl * (1.0 + pl))));
  };
  auto bottom_piece = [&](const T &a2, const T &a3, const T &a4, double esl, double dp) -> SumT {
    return dp * wide(a2 + R(0.5 * esl) * (a3 - a2 + a4 * R(1.0 - r23 * esl)));
  };
  char *dst = reinterpret_cast<char *>(S.dst + fbase), *dst_t = nullptr;
  if constexpr (sizeof(T) != sizeof(R)) dst_t = reinterpret_cast<char *>(S.dst_t + fbase);
  auto store = [&](char *at, char *at_t, const T &v) {
    if constexpr (sizeof(T) == sizeof(R)) {
      *reinterpret_cast<R *>(at) = v;
    } else {
      *reinterpret_cast<R *>(at) = v.v;
      *reinterpret_cast<R *>(at_t) = v.d[0];
    }
  };

  auto sweep = [&](auto lockstep) {
  int kt = 1;  // the target in hand: the wave's in lockstep, else the lane's
  // in lockstep: slot of cell c; thickness times mean of cells c-1 ..
  int cs = NR - 1;
  long long ro = (min(3, km) - 1) * nc4;  // of the record to be loaded next
  char *du = dst, *du_t = dst_t;          // of the target in hand
  SumT M[NR - 1];
#pragma unroll
  for (int m = 0; m < NR - 1; m++) M[m] = SumT(0.0);
  // lane by lane: the open target's sum
  bool open = false;
  SumT acc(0.0);
  char *dl = dst + cbyte, *dl_t = dst_t + cbyte;
  auto emit = [&](const T &v) {
    if (act) store(dl, dl_t, v);
    dl += levb;
    dl_t += levb;
    kt++;
    tr = tn;
    tn = rec(kt + 1);
  };

  long long ao = (min(3, km) - 1) * levb, dof = 0;  // of the next mean, of the next cell's thickness
  T chain = zero;  // the eliminated value above the block
  Blk cur, nxt;
  fetch(0, cur);
  for (int b = 0; b < nb; b++) {
    const int k0 = b * FD_B + 1;
    {
      T qv[FD_B];
      chain = eliminate(b, cur, chain, qv, a2nd);
      substitute(b, cur, CP(b), qv, [&](int j, const T &v) { BQ(j) = v; });
    }
    const bool last = b + 1 == nb;
    if (!last) fetch(b + 1, nxt);
    const int pend = last ? km + 2 : k0 + FD_B - 1;
    auto step = [&](int p, auto inner) {  // inner: 5 <= p < km, no special cells
      constexpr bool IN = decltype(inner)::value;
      A_4 = A_3;
      A_3 = A_2;
      A_2 = A_1;
      A_1 = A_0;
      A_0 = A_p;
      A_p = A_n;
      A_n = ldat(ao);
      if (p + 2 < km) ao += levb;
      L_2 = L_1;
      L_1 = L_0;
      if (IN || p <= km) L_0 = BQ(p - k0);
      else if (p == km + 1) L_0 = qbot;
      // interface p lies between cells p-1 (A_1) and p (A_0)
      if (lim && (IN || (p >= 2 && p <= km))) {
        const T lo = mn2(A_1, A_0), hi = mx2(A_1, A_0);
        if (!IN && (p == 2 || p == km)) {
          L_0 = mx2(mn2(L_0, hi), lo);
        } else {
          const T glo = A_1 - A_2, ghi = A_p - A_0;
          const T dn = mn2(L_0, hi);
          T v;
          if (glo * ghi > zero) {
            v = mx2(dn, lo);
          } else if (glo > zero) {
            v = mx2(L_0, lo);
          } else {
            v = iv == 0 ? mx2(zero, dn) : dn;
          }
          L_0 = v;
        }
      }
      E_3 = E_2;
      E_2 = E_1;
      // flags of cell p-1: 1 extm, 2 ext5, 4 ext6
      if (lim && (IN || (p >= 2 && p <= km + 1))) {
        const int e = p - 1;
        const bool em = !IN && (e == 1 || e == km) ? (L_1 - A_1) * (L_0 - A_1) > zero
                                          : (A_1 - A_2) * (A_0 - A_1) < zero;
        E_1 = em ? 1 : 0;
        if (akord > 9) {
          const T x0 = R(2) * A_1 - (L_1 + L_0), x1 = fabs(L_1 - L_0);
          E_1 |= (fabs(x0) > x1 ? 2 : 0) | (fabs(R(3) * x0) > x1 ? 4 : 0);
        }
      }
      const int c = p - 2;
      if (!IN && c < 1) return;
      // ---- cell c = p-2: a(c) is A_2, its interface values L_2, L_1
      T a1 = A_2, a2 = L_2, a3 = L_1, a4;
      if (!lim) {
        a4 = R(3) * (R(2) * a1 - (a2 + a3));
      } else if (!IN && (c == 1 || c == 2 || c >= km - 1)) {
        if (c == 1) {
          if (iv == 0) {
            a2 = mx2(zero, a2);
          } else if (iv == -1) {
            if (a2 * a1 <= zero) a2 = zero;
          }
        } else if (c == km) {
          if (iv == 0) {
            a3 = mx2(zero, a3);
          } else if (iv == -1) {
            if (a3 * a1 <= zero) a3 = zero;
          }
        }
        a4 = R(3) * (R(2) * a1 - (a2 + a3));
        cs_lim1(a1, a2, a3, a4, (E_2 & 1) != 0, c == 1 || c == km ? 1 : 2);
      } else {
        const T gk = A_2 - A_3, gk1 = A_1 - A_2, gk2 = A_0 - A_1, gkm1 = A_3 - A_4;
        const bool low = use_qmin && a1 < T(qmin);
        if (akord < 9) {
          huynh2(a1, a2, a3, gk, gk1, gk2, gkm1);
          a4 = R(3) * (R(2) * a1 - (a2 + a3));
        } else if (akord == 9) {
          if ((E_2 & 1) && ((E_3 & 1) || (E_1 & 1) || low)) {
            a2 = a1;
            a3 = a1;
            a4 = zero;
          } else {
            a4 = R(6) * a1 - R(3) * (a2 + a3);
            if (fabs(a4) > fabs(a2 - a3)) {
              huynh2(a1, a2, a3, gk, gk1, gk2, gkm1);
              a4 = R(6) * a1 - R(3) * (a2 + a3);
            }
          }
        } else {
          if (E_2 & 2) {
            if ((E_3 & 2) || (E_1 & 2) || low) {
              a2 = a1;
              a3 = a1;
            } else if ((E_3 & 4) || (E_1 & 4)) {
              huynh2(a1, a2, a3, gk, gk1, gk2, gkm1);
            }
          } else if (E_2 & 4) {
            if ((E_3 & 2) || (E_1 & 2)) huynh2(a1, a2, a3, gk, gk1, gk2, gkm1);
          }
          a4 = R(3) * (R(2) * a1 - (a2 + a3));
        }
        if (iv == 0) cs_lim1(a1, a2, a3, a4, (E_2 & 1) != 0, 0);
      }
      const double d1c = d1n;
      if (IN || c < km) dof += 2 * nc4;
      d1n = ldd(dof);
      if constexpr (decltype(lockstep)::value) {
        // ---- the targets whose last cell, over the wave's columns, is c
        cs = cs + 1 == NR ? 0 : cs + 1;
        T *slot = ring + cs * 192;
        slot[0] = a2;
        slot[64] = a3;
        slot[128] = a4;
#pragma unroll
        for (int m = NR - 2; m > 0; m--) M[m] = M[m - 1];
        M[0] = d1c * wide(A_2);  // c's own; M[m]: cell c-m's
        while (kt <= km && __ballot(((tr.rc >> 12) & 0xfff) > c) == 0) {
          const TargetRec t = tr;
          tr = tn;
          tn = recat(ro);
          if (kt + 2 < km) ro += nc4;
          const int lt = t.rc & 0xfff, lb = (t.rc >> 12) & 0xfff;
          auto at = [&](int l) -> const T * {
            const int s = cs - (c - l);
            return ring + (s < 0 ? s + NR : s) * 192;
          };
          const T *x = at(lt);
          const T x2 = x[0], x3 = x[64], x4 = x[128];
          T v;
          if (t.rc >> 24) {
            v = within(x2, x3, x4, t.r0.x, t.r0.y);
          } else {
            const T *y = at(lb);
            const T y2 = y[0], y3 = y[64], y4 = y[128];
            SumT sum = top_piece(x2, x3, x4, t.r0.x, t.r1.x);
#pragma unroll
            for (int m = NR - 2; m > 0; m--)
              if (lt < c - m && c - m < lb) sum = sum + M[m];
            sum = sum + bottom_piece(y2, y3, y4, t.r0.y, t.r1.y);
            v = narrow(quot_any(sum, t.r2.x, t.r2.y));
          }
          if (act) store(du + cbyte, du_t + cbyte, v);
          du += levb;
          du_t += levb;
          kt++;
        }
      } else {
        // ---- the target layers that end, lie or begin in source layer c
        while (kt <= km) {
          const int lt = tr.rc & 0xfff, lb = (tr.rc >> 12) & 0xfff;
          if (open) {
            if (lb != c) {
              acc = acc + d1c * wide(A_2);
              break;
            }
            acc = acc + bottom_piece(a2, a3, a4, tr.r0.y, tr.r1.y);
            emit(narrow(quot_any(acc, tr.r2.x, tr.r2.y)));
            open = false;
          } else if (lt == 0) {
            emit(narrow(SumT(0.0) / tr.r2.x));
          } else if (lt > c) {
            break;
          } else if (tr.rc >> 24) {
            emit(within(a2, a3, a4, tr.r0.x, tr.r0.y));
          } else {
            acc = top_piece(a2, a3, a4, tr.r0.x, tr.r1.x);
            open = true;
            break;
          }
        }
      }
    };
    for (int p = k0; p <= pend; p++) {
      if (decltype(lockstep)::value && p >= 5 && p < km)
        step(p, std::true_type{});
      else
        step(p, std::false_type{});
    }
    cur = nxt;
  }
  if constexpr (!decltype(lockstep)::value)
    // a target that ends below the source, and those no layer holds
    while (kt <= km) {
      emit(narrow(open ? quot_any(acc, tr.r2.x, tr.r2.y) : SumT(0.0) / tr.r2.x));
      open = false;
    }
  };
  if (__builtin_amdgcn_readfirstlane(a.tab.win[col]) <= NR)
    sweep(std::true_type{});
  else
    sweep(std::false_type{});
}

template <typename T>
size_t fields_lds(int km) {
  const int nb = (km + FD_B - 1) / FD_B;
  return sizeof(T) * FD_WAVES * (size_t)fd_rows<T>(nb) * 64;
}

}  // namespace

template <typename R>
size_t coltab_bytes(int km, long long ncols) {
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t n = (size_t)km * ncols;
  return al(sizeof(Elim<R>) * n) + al(sizeof(double) * n) + 3 * al(sizeof(double2) * n) + al(sizeof(int) * n) +
         al(sizeof(R) * 3 * (size_t)ncols) + al(sizeof(int) * (size_t)ncols);
}

template <typename R>
ColTab<R> coltab_carve(void *base, int km, long long ncols) {
  ColTab<R> t{};
  char *p = (char *)base;
  auto take = [&](size_t b) {
    char *r = p;
    p += (b + 255) & ~(size_t)255;
    return r;
  };
  const size_t n = (size_t)km * ncols;
  t.el = (Elim<R> *)take(sizeof(Elim<R>) * n);
  t.d1 = (double *)take(sizeof(double) * n);
  t.r0 = (double2 *)take(sizeof(double2) * n);
  t.r1 = (double2 *)take(sizeof(double2) * n);
  t.r2 = (double2 *)take(sizeof(double2) * n);
  t.rc = (int *)take(sizeof(int) * n);
  t.bot = (R *)take(sizeof(R) * 3 * (size_t)ncols);
  t.win = (int *)take(sizeof(int) * (size_t)ncols);
  return t;
}

// More than 64 KB of dynamic LDS per workgroup must be allowed per kernel.
int fields_setup() {
  static DeviceOnce once;
  FV3_HIP(once([] {
    hipError_t err = hipSuccess;
    auto allow = [&](const void *fn, size_t b) {
      if (err == hipSuccess) err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)b);
    };
    allow(reinterpret_cast<const void *>(&k_fields_prep<float>), prep_lds(FIELDS_MAX_KM));
    allow(reinterpret_cast<const void *>(&k_fields_prep<double>), prep_lds(FIELDS_MAX_KM));
    allow(reinterpret_cast<const void *>(&k_fields<float>), fields_lds<float>(FIELDS_MAX_KM));
    allow(reinterpret_cast<const void *>(&k_fields<double>), fields_lds<double>(FIELDS_MAX_KM));
    allow(reinterpret_cast<const void *>(&k_fields<D1>), std::min<size_t>(fields_lds<D1>(FIELDS_MAX_KM), 160 * 1024));
    return err;
  }));
  return 0;
}

template <typename R>
int fields_prep(Ctx &c, const ColTab<R> &tab, const ColSource &src, int ni, int nj, bool iv2, hipStream_t s) {
  const Dims &d = c.d;
  if (c.npz > FIELDS_MAX_KM) return set_error("column tables support km <= %d (got %d)", FIELDS_MAX_KM, c.npz);
  if (fields_setup()) return 1;
  PrepGeo g{};
  g.km = c.npz; g.ni = ni; g.nj = nj; g.is = d.is; g.js = d.js; g.isd = d.isd; g.jsd = d.jsd; g.nid = d.nid;
  g.cni = d.ie - d.is + 1;
  g.ncol = (long long)ni * nj;
  g.ncols = g.ncol * c.ntiles;
  g.s2 = d.s2;
  g.spe = (long long)(g.cni + 2) * (g.km + 1) * (d.je - d.js + 3);
  g.ncb = (int)((g.ncol + 63) / 64);
  hipLaunchKernelGGL(k_fields_prep<R>, dim3((unsigned)g.ncb * (unsigned)c.ntiles), dim3(64 * PREP_WAVES), prep_lds(g.km),
                     s, g, src, tab, iv2);
  FV3_HIP(hipGetLastError());
  return 0;
}

int fields_target(Ctx &c, const ColTab<double> &tab, const double *dp1, double *out, const int *counts, hipStream_t s) {
  const Dims &d = c.d;
  const long long ncols = (long long)(d.ie - d.is + 1) * (d.je - d.js + 1) * c.ntiles;
  hipLaunchKernelGGL(k_fields_target, dim3((unsigned)((d.s2 + 255) / 256), (unsigned)c.npz, (unsigned)c.ntiles), dim3(256),
                     0, s, tab.r2, dp1, out, d, c.npz, ncols, StepCounts{counts, c.npz});
  FV3_HIP(hipGetLastError());
  return 0;
}

template <typename T>
int fields_run(Ctx &c, FieldsArgs<T> &a, int ni, int nj) {
  a.km = c.npz;
  a.ni = ni;
  a.ncol = (long long)ni * nj;
  a.ncols = a.ncol * c.ntiles;
  a.ncb = (int)((a.ncol + 63) / 64);
  a.nf = 0;
  for (int s = 0; s < a.nset; s++) a.nf += a.set[s].count;
  if (a.nf == 0) return 0;
  if (fields_lds<T>(a.km) > 160 * 1024) return set_error("remap of %d levels does not fit in LDS", a.km);
  a.ntiles = c.ntiles;
  const long long nwg = ((long long)a.ncb * c.ntiles * a.nf + FD_WAVES - 1) / FD_WAVES;
  if (nwg > 0x7fffffffLL / FD_WAVES) return set_error("remap grid too large");
  a.nwg = (unsigned)nwg;
  hipLaunchKernelGGL(k_fields<T>, dim3(a.nwg), dim3(64 * FD_WAVES), fields_lds<T>(a.km), c.stream, a);
  FV3_HIP(hipGetLastError());
  return 0;
}

template <typename T>
FieldSet<T> cell_set(const Ctx &c, const T *src, T *dst, int iv) {
  const Dims &d = c.d;
  const long long o0 = (long long)(d.js - d.jsd) * d.nid + (d.is - d.isd);
  FieldSet<T> f{};
  f.src = src + o0;
  f.dst = dst + o0;
  f.lev = d.s2;
  f.ld = d.nid;
  f.fstride = f.tstride = f.sfstride = f.ststride = d.s2 * c.npz;
  f.count = 1;
  f.iv = iv;
  return f;
}

template <typename T>
FieldSet<T> tracer_set(const Ctx &c, const T *src, T *dst, int nq) {
  FieldSet<T> f = cell_set(c, src, dst, 0);
  f.tstride = f.ststride = f.fstride * nq;
  f.count = nq;
  f.use_qmin = true;
  f.mapn = nq > 5;  // mapn_tracer, else map1_q2
  return f;
}

#define FV3_FIELDS(T)                                                                                            \
  template size_t coltab_bytes<T>(int, long long);                                                               \
  template ColTab<T> coltab_carve<T>(void *, int, long long);                                                    \
  template int fields_prep<T>(Ctx &, const ColTab<T> &, const ColSource &, int, int, bool, hipStream_t);         \
  template int fields_run<T>(Ctx &, FieldsArgs<T> &, int, int);                                                  \
  template FieldSet<T> cell_set<T>(const Ctx &, const T *, T *, int);                                            \
  template FieldSet<T> tracer_set<T>(const Ctx &, const T *, T *, int);
FV3_FIELDS(double)
FV3_FIELDS(float)
template int fields_run<D1>(Ctx &, FieldsArgs<D1> &, int, int);
#undef FV3_FIELDS

}  // namespace fv3
