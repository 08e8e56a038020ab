// rows.h -- rows of the SBP 4-8 operators on operands staged in LDS, shared by the kernels
// that run a whole RK stage (fused2d.hip, line1d.hip).
#pragma once
#include "device.h"

namespace mgd {

// A pointer that comes out of a descriptor in memory (group kernels) is generic to the
// compiler: flat accesses, which count as LDS and as global ones at once.  This says that it
// points to global memory.
template <class T>
using global_ptr = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ global_ptr<T> glob(T* p) {
  return (global_ptr<T>)p;
}

// The patch tables: no kernel writes them, so they are read through scalar loads, also behind
// a barrier or a store.
using ConstPatches = const __attribute__((address_space(4))) Patches;
using ConstPatch = const __attribute__((address_space(4))) DPatch;

// The dense closure rows (BD x BW) of operator `slot` into LDS, one value per thread and
// turn: the left end's, then the right end's (row m: the m-th point from that end).
template <int NT, int BD, int BW>
__device__ __forceinline__ void stage_rows(const Geo& g, int slot, double* tab) {
  const Op& op = g.ops[slot];
  for (int e = threadIdx.x; e < 2 * BD * BW; e += NT) {
    const int m = e / BW % BD, c = e % BW;
    tab[e] = e < BD * BW ? op.b1[m][c] : op.b2[m][c];
  }
}

// A closure row on the BW operands f(j, k) of the components j, in the order of the grid
// index; four columns of LDS reads at a time (more would spill registers).
template <int NV, int BW, class F>
__device__ __forceinline__ void closure_row(const double* row, F&& f, double* out) {
#pragma unroll
  for (int j = 0; j < NV; ++j) out[j] = 0.0;
#pragma unroll
  for (int k = 0; k < BW; ++k) {
    const double b = row[k];
#pragma unroll
    for (int j = 0; j < NV; ++j) out[j] += b * f(j, k);
    if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
}

// Place of index i on a non-periodic direction: m the distance from the nearer end, right
// which end that is; m is large on a periodic direction.
struct EdgePlace {
  int m;
  bool right;
};
__device__ __forceinline__ EdgePlace edge_place(const Dir& dd, int i) {
  const int r = dd.len - 1 - i;
  return {dd.periodic ? 1 << 30 : min(i, r), r < i};
}

__device__ __forceinline__ double skew_sum(const double* p, const double* m, const double* c) {
  double s = c[1] * (p[0] - m[0]);
#pragma unroll
  for (int k = 2; k <= 4; ++k) s += c[k] * (p[k - 1] - m[k - 1]);
  return s;
}

// Interior row of D4 (and of D4^T) on the window w[0..4].  The products with 1 and -4 are
// exact, so the fused form rounds as the plain sum does.
__device__ __forceinline__ double d4_row(const double* w) {
  return __fma_rn(kD4[1], w[3] + w[1], w[4] + w[0]) + kD4[0] * w[2];
}

// D4^T (-arc D4 x) of the two-level dissipation at one point from the nine operands about it
// (the metric is constant along a line of a rectilinear grid): the five intermediates that
// the point's row needs are formed again by each thread, 35 operations instead of a pass of
// the intermediates through LDS with two more barriers.
__device__ __forceinline__ double two_level(const double* w, double marc) {
  double z[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) z[k] = marc * d4_row(w + k);
  return d4_row(z);
}

// The same on a line with ends: w holds the nine operands of the window that starts at index
// clamp(i - 4, 0, len - 9), b the weights of the point's closure row.  The first two
// rows of D4 repeat the stencil of the third one, summed in the order of the index; D4^T has 5
// closure rows of 7 columns.
__device__ __forceinline__ double two_level_edge(const double* w, double marc, EdgePlace e,
                                                 const double* b) {
  double z[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) z[k] = marc * d4_row(w + k);
  if (e.m >= 5) return d4_row(z);
  const int o = e.right ? 4 : 0;
  double first = 0.0, s = 0.0;
#pragma unroll
  for (int k = 0; k < 5; ++k) first += kD4[k < 2 ? 2 - k : k - 2] * (o ? w[k + 4] : w[k]);
  first = marc * first;
  if (!e.right) {
    s += b[0] * first;
    s += b[1] * first;
#pragma unroll
    for (int k = 0; k < 5; ++k) s += b[k + 2] * z[k];
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) s += b[k] * z[k];
    s += b[5] * first;
    s += b[6] * first;
  }
  return s;
}

// The weights of the closure row of D4^T at a point (of some row where it has none).
__device__ __forceinline__ void closure_weights(const double* rows, EdgePlace e, double* b) {
  const double* r = rows + (e.right ? 35 : 0) + 7 * min(e.m, 4);
#pragma unroll
  for (int c = 0; c < 7; ++c) b[c] = r[c];
}

}  // namespace mgd
