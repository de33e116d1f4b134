// mapz_fields.h -- the vertical remap in upstream evaluation order, one thread
// per (column, field), over column tables shared by every field of a column
// (host-side internal interface; kernels in mapz_fields.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "dual.h"
#include "mapz_column.h"

namespace fv3 {

struct Ctx;

// the real type a value type is stored in: float, double, or double for
// (value, tangent) pairs kept in two arrays
template <typename T>
struct RealOf {
  using type = T;
};
template <>
struct RealOf<D1> {
  using type = double;
};

// elimination factors of one interface: Q'(k) = (3 (a(k-1) + d4 a(k)) -
// Q'(k-1)) / bt, Q(k) = Q'(k) - g Q(k+1); y = 1 / bt
template <typename R>
struct alignas(4 * sizeof(R)) Elim {
  R d4, bt, y, g;
};

// Column tables, [level][column] over the columns of every tile:
//   el   elimination factors (level 1 holds the top row's)
//   d1   source layer thickness
//   r0   per target layer: pl, pr -- the fraction within its source layer of
//        the target's top interface and of its bottom one
//   r1   pressure widths of its top and bottom pieces
//   r2   its thickness and that one's reciprocal
//   rc   its source layers: top | bottom << 12 | (both in one layer) << 24
//        (top 0: no layer holds it; bottom km + 1: it ends below the source)
//   bot  [3][column] bottom-row factors
//   win  [column] how many source layers one target layer takes in over the 64
//        columns of a block together, at most (a block with a column whose
//        interfaces are out of order: NO_WINDOW)
constexpr int NO_WINDOW = 1 << 20;
template <typename R>
struct ColTab {
  Elim<R> *el;
  double *d1;
  double2 *r0, *r1, *r2;
  int *rc;
  R *bot;
  int *win;
};

template <typename R>
size_t coltab_bytes(int km, long long ncols);
template <typename R>
ColTab<R> coltab_carve(void *base, int km, long long ncols);

// Largest km the kernels take (the column's interfaces are staged in LDS).
constexpr int FIELDS_MAX_KM = 255;
// ... and for (value, tangent) pairs, whose block ends are twice as large
constexpr int FIELDS_MAX_KM_TL = 160;

// What the tables are made from: cell columns of delp (kind 0: pe1 = ptop +
// running sum, pe2 = ak + bk ps; delp_out, when given, receives the target
// thickness and may be delp itself), or the interfaces of the D-grid winds'
// columns (kind 1: u, averages of cells j-1, j; kind 2: v, of i-1, i) from pe
// (is-1:ie+1, km+1, js-1:je+1) and ps (isd:ied, jsd:jed).
struct ColSource {
  int kind;
  double ptop;
  const double *ak, *bk;
  const double *delp;
  double *delp_out;
  const double *pe, *ps;
};

// fields sharing a layout: src, dst at the first column of tile 0; fstride
// between fields, tstride between tiles (sfstride, ststride: the source's),
// lev between levels, ld between rows.  qs: surface values (iv = -2), (column)
// per tile.
template <typename T>
struct FieldSet {
  using R = typename RealOf<T>::type;
  const R *src, *src_t;
  R *dst, *dst_t;
  long long fstride, tstride, sfstride, ststride, lev;
  int ld, count, iv;
  bool use_qmin, mapn;
  R qmin;
  const R *qs;
};

constexpr int FIELDS_MAX_SETS = 3;

template <typename T>
struct FieldsArgs {
  using R = typename RealOf<T>::type;
  int km, ni, ncb, ntiles, nf, nset;
  unsigned nwg;
  long long ncol, ncols;  // columns per tile, of every tile
  ColTab<R> tab;
  FieldSet<T> set[FIELDS_MAX_SETS];
  signed char kord[REMAP_MAX_NQ + FIELDS_MAX_SETS];  // by field
};

// once per device, before any capture: the kernels' LDS limits
int fields_setup();
// tables of the columns (ni x nj per tile, every tile of c); iv2: factors of
// the iv = -2 solve (bottom value given)
template <typename R>
int fields_prep(Ctx &c, const ColTab<R> &tab, const ColSource &src, int ni, int nj, bool iv2, hipStream_t s);
// the target thickness of the cell columns from their tables (halo cells as dp1's;
// out may be dp1; counts: StepCounts, or NULL)
int fields_target(Ctx &c, const ColTab<double> &tab, const double *dp1, double *out, const int *counts, hipStream_t s);
// remap every field of the sets; sources and destinations must not overlap
template <typename T>
int fields_run(Ctx &c, FieldsArgs<T> &a, int ni, int nj);

// sets for tracers (iv = 0, floor 0; q (isd:ied, jsd:jed, km, nq) per tile) and
// for one field on cell columns with a halo
template <typename T>
FieldSet<T> tracer_set(const Ctx &c, const T *src, T *dst, int nq);
template <typename T>
FieldSet<T> cell_set(const Ctx &c, const T *src, T *dst, int iv);

// tracers, pt and delz (any may be absent) of Lagrangian_to_Eulerian in place
// over the cell columns, delp to its target thickness; stream-ordered
template <typename T>
int remap_cells_inplace(Ctx &c, int km, int nq, const double *ak, const double *bk, double ptop, double *delp, T *q,
                        T *pt, T *dz, const int *kord_tr, int kord_tm, int kord_dz, double t_min, int fill);
int remap_orders_check(int km, int nq, const int *kord_tr, bool with_pt, int kord_tm);

}  // namespace fv3
