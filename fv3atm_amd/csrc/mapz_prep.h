// mapz_prep.h -- a workgroup's columns of Lagrangian interfaces in LDS, shared
// by the kernels that tabulate what a remap's columns have in common.
#pragma once
#include <hip/hip_runtime.h>

namespace fv3 {

// The sub-cycle counts (n of them) of a step whose remap launches are submitted
// before the host knows them: where none is at least 1 the host refuses the step,
// and a kernel may not write the target thickness.  No counts (NULL): it may.
struct StepCounts {
  const int *ns;
  int n;
  // whether the calling thread's share of the counts lets the step go on
  __device__ __forceinline__ bool any(int tid, int threads) const {
    bool a = ns == nullptr;
    if (ns)
      for (int k = tid; k < n; k += threads) a = a || ns[k] >= 1;
    return a;
  }
};

constexpr int PREP_WAVES = 8;

// Columns per workgroup: one per lane, or per two lanes (which then do the
// same) where 64 columns of interfaces do not fit in LDS; at most 129 KB up to
// 512 levels.
__host__ __device__ constexpr int prep_cols(int km) { return km <= 255 ? 64 : 32; }
constexpr int PREP_MAX_KM = 512;  // what the one-thread-per-column field kernel takes (64 KB of LDS)
__host__ __device__ constexpr size_t prep_lds(int km) { return sizeof(double) * (size_t)(km + 1) * prep_cols(km); }

// interface k (1-based) of the lane's column: [km + 1][columns] doubles
struct ColPe {
  double *p;
  int cols;
  __device__ __forceinline__ double &operator()(int k) const { return p[(k - 1) * cols]; }
  // the first layer whose lower interface is at or below pressure v (the
  // column in order, v within it), walking from layer l
  __device__ __forceinline__ int layer_of(double v, int l, int km) const {
    while (l < km && v > (*this)(l + 1)) l++;
    while (l > 1 && !(v > (*this)(l))) l--;
    return l;
  }
};

// the column's interfaces by running sums from ptop: every wave loads its
// share of the thicknesses (level k at dl[(k-1) s2]), then wave 0 adds them up.
// The caller synchronises before reading.
__device__ __forceinline__ void stage_interfaces(const ColPe &P, int km, double ptop, const double *dl, long long s2,
                                                 int wave) {
  int k = 1 + wave;
  for (; k + 3 * PREP_WAVES <= km; k += 4 * PREP_WAVES) {
    double v[4];
#pragma unroll
    for (int m = 0; m < 4; m++) v[m] = dl[(long long)(k + m * PREP_WAVES - 1) * s2];
#pragma unroll
    for (int m = 0; m < 4; m++) P(k + m * PREP_WAVES + 1) = v[m];
  }
  for (; k <= km; k += PREP_WAVES) P(k + 1) = dl[(long long)(k - 1) * s2];
  __syncthreads();
  if (wave == 0) {
    double p = ptop;
    P(1) = p;
    int q = 1;
    for (; q + 7 <= km; q += 8) {
      double v[8];
#pragma unroll
      for (int m = 0; m < 8; m++) v[m] = P(q + m + 1);
#pragma unroll
      for (int m = 0; m < 8; m++) P(q + m + 1) = p = p + v[m];
    }
    for (; q <= km; q++) P(q + 1) = p = p + P(q + 1);
  }
}

}  // namespace fv3
