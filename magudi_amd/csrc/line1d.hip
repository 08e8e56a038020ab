// line1d.hip -- whole RK4 steps of 1-D inviscid regions in one launch.
//
// A line of a few thousand points keeps a handful of CUs busy for a microsecond per stage; with
// a launch per operator (eight to ten per stage) the runs were launches and nothing else.  Here
// a work-group owns a piece of the line and carries it through up to four time steps: it loads
// its points with a halo of four points per stage on either side, and each stage computes the
// points whose stencils still hold, four fewer on a side that is not an end of the line.  One
// thread per point; its state, the RK levels and the patch constants stay in registers, the
// operand and the flux pass through LDS (two buffers in turn: one barrier per stage).
//
// The halo work is repeated by the neighbours: 256 threads own 96 points of a four-step launch.
// That is the price of one exchange through memory instead of sixteen, paid by CUs that would
// idle; line_steps() takes fewer steps per launch where the line fills the chip.
//
// What bounds it: the latency of a stage inside the work-group (2 us: LDS write, barrier, 35 LDS
// reads, 200 dependent FP64 operations on one wave per SIMD).  A line of 2048 points, forward /
// adjoint, us per step: 97 / 140 with a launch per operator, 8.3 / 11 here; 400000 points
// 198 / 362 -> 36 / 162; 512 lines of 2048 350 / 726 -> 86 / 420.
//
// Every sum is formed in the order of the per-operator kernels (kernels.hip), so the states and
// gradients are theirs bit for bit.
#include "line1d.h"
#include "rows.h"

namespace mgd {

constexpr int kLT = 256;              // threads, and points with halo, of a work-group
constexpr int kLN = 3;                // components
constexpr int kLW = kLT + 8;          // LDS row: four points of padding on either side
constexpr int kEnd = 16;              // columns that the closure rows of either end reach

// The piece of work-group b: owned points [x0, x0 + sx), staged points [e0, e0 + count) (indices
// of a periodic line wrap), and whether the staged points begin / end with the line.
struct Piece {
  int x0, sx, e0, count;
  bool first, last;
};
__device__ __forceinline__ Piece line_piece(const Dir& d, int nb, int halo, int b) {
  Piece c;
  const int q = d.len / nb, m = d.len % nb;
  c.x0 = b * q + min(b, m);
  c.sx = q + (b < m ? 1 : 0);
  int lo = c.x0 - halo, hi = c.x0 + c.sx + halo;
  c.first = !d.periodic && lo < kEnd;
  c.last = !d.periodic && hi > d.len - kEnd;
  if (c.first) lo = 0;
  if (c.last) hi = d.len;
  c.e0 = lo;
  c.count = hi - lo;
  return c;
}

// The point of this thread: staged position e, grid index gi, distances from the ends, the
// patches that hold it.
struct LinePoint {
  int e, gi;
  bool own;
  EdgePlace edge;
  unsigned patches;
};
__device__ __forceinline__ LinePoint line_point(const Dir& d, const Piece& c, ConstPatches* P) {
  LinePoint t;
  t.e = threadIdx.x;
  int gi = c.e0 + min(t.e, c.count - 1);
  if (d.periodic) {
    gi %= d.len;
    if (gi < 0) gi += d.len;
  }
  t.gi = gi;
  t.own = t.e >= c.x0 - c.e0 && t.e < c.x0 - c.e0 + c.sx;
  t.edge = edge_place(d, gi);
  t.patches = 0;
  const int n = P->count;
  for (int ip = 0; ip < n; ++ip)
    if (gi >= P->p[ip].lo[0] && gi <= P->p[ip].hi[0]) t.patches |= 1u << ip;
  return t;
}

// Whether stage j of the launch still computes position e.
__device__ __forceinline__ bool holds(const Piece& c, int e, int j) {
  const int m = 4 * (j + 1);
  return e >= (c.first ? 0 : m) && e < c.count - (c.last ? 0 : m);
}

// Derivative row of the point on one component x (its place in a staged row) of operator rows
// `tab` (BD x BW left, then right); c: interior coefficients.
template <int BD, int BW>
__device__ __forceinline__ void line_derivative(const double (*s)[kLW], const LinePoint& t,
                                                const Piece& c, const Dir& d, const double* tab,
                                                const double* cf, double* out) {
  if (t.edge.m < BD) {
    const int col = 4 + (t.edge.right ? d.len - BW - c.e0 : 0);
    closure_row<kLN, BW>(tab + BW * t.edge.m + (t.edge.right ? BD * BW : 0),
                         [&](int l, int k) { return s[l][col + k]; }, out);
    return;
  }
#pragma unroll
  for (int l = 0; l < kLN; ++l) {
    const double* x = &s[l][t.e + 4];
    const double p[4] = {x[1], x[2], x[3], x[4]}, m[4] = {x[-1], x[-2], x[-3], x[-4]};
    out[l] = skew_sum(p, m, cf);
  }
}

// r += amount * dissipation of the staged operand s at the point (addDissipation).
__device__ __forceinline__ void line_dissipation(const Geo& g, const double (*s)[kLW],
                                                 const LinePoint& t, const Piece& c,
                                                 const double* tab, double hw, double amount,
                                                 double* r) {
  const Dir& d = g.dir[0];
  if (g.composite) {
    double v[kLN];
    if (t.edge.m < 8) {
      const int col = 4 + (t.edge.right ? d.len - 12 - c.e0 : 0);
      closure_row<kLN, 12>(tab + 12 * t.edge.m + (t.edge.right ? 96 : 0),
                           [&](int l, int k) { return s[l][col + k]; }, v);
    } else {
      const double* k = g.ops[SLOT_DISS].c + kMaxHW;
#pragma unroll
      for (int l = 0; l < kLN; ++l) {
        const double* x = &s[l][t.e + 4];
        double a = 0.0;
#pragma unroll
        for (int i = 1; i <= 4; ++i) a += k[i] * (x[i] + x[-i]);
        v[l] = a + k[0] * x[0];
      }
    }
#pragma unroll
    for (int l = 0; l < kLN; ++l) r[l] = r[l] + amount * v[l];
    return;
  }
  const int m = t.edge.m;
  const int col = t.e + 4 - 4 + (m < 4 ? (t.edge.right ? m - 4 : 4 - m) : 0);
  double b[7];
  closure_weights(tab, t.edge, b);
#pragma unroll
  for (int l = 0; l < kLN; ++l) {
    double w[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) w[k] = s[l][col + k];
    double v = two_level_edge(w, -1.0, t.edge, b);    // the metric of a line is 1
    if (hw != 1.0) v = v / hw;       // 1 away from the first / last boundary rows
    r[l] = r[l] + amount * v;
  }
}

// Closure rows of the dissipation of a non-periodic line.
__device__ __forceinline__ void stage_diss_rows(const Geo& g, double* tab) {
  if (!g.dissipation) return;
  if (g.composite) stage_rows<kLT, 8, 12>(g, SLOT_DISS, tab);
  else stage_rows<kLT, 5, 7>(g, SLOT_DISS_T, tab);
}

// -------------------------------------------------------------------------- forward
__global__ void __launch_bounds__(kLT) k_line_forward(Geo g, const Patches* patches, int nb,
                                                      LineForward a) {
  __shared__ double sq[2][kLN][kLW], sf[2][kLN][kLW], tab[192 + 192];
  ConstPatches* P = (ConstPatches*)patches;
  const Dir d = g.dir[0];
  const Piece c = line_piece(d, nb, 4 * a.nstages, blockIdx.x);
  const LinePoint t = line_point(d, c, P);
  const long inst = blockIdx.y, N = g.N;
  double v[kLN], q0[kLN], b2[kLN];
#pragma unroll
  for (int l = 0; l < kLN; ++l) {
    v[l] = glob(a.in)[(inst * kLN + l) * N + t.gi];
    q0[l] = b2[l] = 0.0;
  }
  const double h = glob(g.h[0])[t.gi], hw = glob(g.hw[0])[t.gi], x = glob(g.x[0])[t.gi];
  const double jac = 1.0 / h;
  double d1[5];
#pragma unroll
  for (int k = 1; k <= 4; ++k) d1[k] = g.ops[SLOT_FIRST].c[kMaxHW + k];
  if (!d.periodic) {
    stage_rows<kLT, 8, 12>(g, SLOT_FIRST, tab);
    stage_diss_rows(g, tab + 192);
  }
  // constants of the actuator and the cost target at the point
  const bool act = a.control && a.ip_act >= 0 && ((t.patches >> a.ip_act) & 1u);
  const bool cost = a.jpartial && a.ip_cost >= 0 && t.own && ((t.patches >> a.ip_cost) & 1u);
  int ka = 0, kc = 0;
  double ma = 0.0, pb = 0.0, mo = 0.0;
  if (act) {
    ka = t.gi - P->p[a.ip_act].lo[0];
    ma = glob(P->p[a.ip_act].strength)[ka];
  }
  if (cost) {
    kc = t.gi - P->p[a.ip_cost].lo[0];
    pb = glob(P->p[a.ip_cost].aplus)[kc];
    mo = glob(P->p[a.ip_cost].strength)[kc];
  }
  unsigned point_patches = t.patches;
  if (a.ip_cost >= 0) point_patches &= ~(1u << a.ip_cost);
  if (a.ip_act >= 0 && !act) point_patches &= ~(1u << a.ip_act);
  double e0 = 0.0;                    // Gaussian of the first source
  if (a.nsrc > 0) {
    const double dx = x - glob(a.src)[0].loc[0];
    e0 = exp(-glob(a.src)[0].gfac * (0.0 + dx * dx));
  }
#pragma unroll 1
  for (int j = 0; j < a.nstages; ++j) {
    const int stage = (j & 3) + 1, buf = j & 1;
    double ctl = 0.0;
    if (act) ctl = glob(a.control)[(long)j * a.na + inst * a.control_stride + ka];
    {
      const Prim<1> s = prim<1>(v, g.gamma);
      double f[kLN];
      inviscid_flux<1>(v, s, 0, f);
#pragma unroll
      for (int l = 0; l < kLN; ++l) {
        sq[buf][l][t.e + 4] = v[l];
        sf[buf][l][t.e + 4] = f[l];
      }
    }
    __syncthreads();
    if (!holds(c, t.e, j)) continue;
    double r[kLN];
    line_derivative<8, 12>(sf[buf], t, c, d, tab, d1, r);
#pragma unroll
    for (int l = 0; l < kLN; ++l) r[l] = 0.0 - r[l];
    if (g.dissipation) line_dissipation(g, sq[buf], t, c, tab + 192, hw, g.diss_amount, r);
#pragma unroll
    for (int l = 0; l < kLN; ++l) r[l] = r[l] * jac;
    for (unsigned m = point_patches; m; m &= m - 1) {
      const DPatch& pt = patches->p[__ffs(m) - 1];
      const int k = t.gi - pt.lo[0];
      switch (pt.type) {
        case MGD_PATCH_FAR_FIELD: {
          const double* A = pt.aplus + (long)k * 9;
          const double* qt = pt.aplus + (long)pt.np * 9 + (long)k * 3;
          const double sj = pt.sigma_inv * jac;
#pragma unroll
          for (int i = 0; i < kLN; ++i) {
            double s = 0.0;
#pragma unroll
            for (int l = 0; l < kLN; ++l) s += A[l * 3 + i] * (v[l] - qt[l]);
            r[i] = r[i] - sj * s;
          }
          break;
        }
        case MGD_PATCH_SPONGE: {
          const double sp = pt.strength[k];
          const double* qt = pt.aplus + (long)k * 3;
#pragma unroll
          for (int l = 0; l < kLN; ++l) r[l] = r[l] - sp * (v[l] - qt[l]);
          break;
        }
        case MGD_PATCH_ACTUATOR:
          r[2] = r[2] + ma * ctl;
          break;
        case MGD_PATCH_KOLMOGOROV:
          r[1] = r[1] + v[0] * pt.strength[k];
          break;
        default:
          break;
      }
    }
    for (int s = 0; s < a.nsrc; ++s) {
      const double amp = glob(a.src_amp)[(long)j * a.nsrc + inst * a.src_inst_stride + s];
      double e = e0;
      if (s > 0) {
        const double dx = x - glob(a.src)[s].loc[0];
        e = exp(-glob(a.src)[s].gfac * (0.0 + dx * dx));
      }
      r[2] = r[2] + amp * e;
    }
    // RK4 stage update (substepForwardRK4, src/RK4IntegratorImpl.f90:115-156)
    const double dt = a.dt;
#pragma unroll
    for (int l = 0; l < kLN; ++l) {
      if (stage == 1) {
        q0[l] = v[l];
        b2[l] = v[l] + div6(dt * r[l]);
        v[l] = v[l] + dt * r[l] / 2.0;
      } else if (stage == 4) {
        v[l] = b2[l] + div6(dt * r[l]);
      } else {
        b2[l] = b2[l] + div3(dt * r[l]);
        v[l] = stage == 2 ? q0[l] + dt * r[l] / 2.0 : q0[l] + dt * r[l];
      }
    }
    if (!t.own) continue;
    double* const k1 = a.keep[j];
    double* const k2 = stage == 4 ? a.keep2[j >> 2] : nullptr;
#pragma unroll
    for (int l = 0; l < kLN; ++l) {
      if (k1) glob(k1)[(inst * kLN + l) * N + t.gi] = v[l];
      if (k2) glob(k2)[(inst * kLN + l) * N + t.gi] = v[l];
    }
    if (cost) {
      const Prim<1> s = prim<1>(v, g.gamma);
      const double F = s.p - pb;
      const double gn = (hw * 1.0) * h;     // gnorm<1>
      glob(a.jpartial)[(inst * a.nslots + a.slot + j) * a.npts + kc] = 1.0 * gn * (F * F * mo);
    }
  }
  if (a.out && t.own) {
#pragma unroll
    for (int l = 0; l < kLN; ++l) glob(a.out)[(inst * kLN + l) * N + t.gi] = v[l];
  }
}

// -------------------------------------------------------------------------- adjoint
__global__ void __launch_bounds__(kLT) k_line_adjoint(Geo g, const Patches* patches, int nb,
                                                      LineAdjoint a) {
  __shared__ double sl[2][kLN][kLW], tab[384 + 192];
  ConstPatches* P = (ConstPatches*)patches;
  const Dir d = g.dir[0];
  const Piece c = line_piece(d, nb, 4 * a.nstages, blockIdx.x);
  const LinePoint t = line_point(d, c, P);
  const long inst = blockIdx.y, N = g.N;
  double v[kLN], l0[kLN], b2[kLN], qn[kLN];
#pragma unroll
  for (int l = 0; l < kLN; ++l) {
    v[l] = glob(a.in)[(inst * kLN + l) * N + t.gi];
    qn[l] = glob(a.q[0])[(inst * kLN + l) * N + t.gi];
    l0[l] = b2[l] = 0.0;
  }
  const double h = glob(g.h[0])[t.gi], hw = glob(g.hw[0])[t.gi];
  const double jac = 1.0 / h;
  double d1[5];
#pragma unroll
  for (int k = 1; k <= 4; ++k) d1[k] = g.ops[SLOT_ADJ].c[kMaxHW + k];
  if (!d.periodic) {
    stage_rows<kLT, 12, 16>(g, SLOT_ADJ, tab);
    stage_diss_rows(g, tab + 384);
  }
  const bool act = a.ip_act >= 0 && t.own && ((t.patches >> a.ip_act) & 1u);
  const bool cost = a.ip_cost >= 0 && ((t.patches >> a.ip_cost) & 1u);
  int ka = 0;
  double ma = 0.0, pb = 0.0, mo = 0.0;
  if (act) {
    ka = t.gi - P->p[a.ip_act].lo[0];
    ma = glob(P->p[a.ip_act].strength)[ka];
  }
  if (cost) {
    const int kc = t.gi - P->p[a.ip_cost].lo[0];
    pb = glob(P->p[a.ip_cost].aplus)[kc];
    mo = glob(P->p[a.ip_cost].strength)[kc];
  }
  unsigned point_patches = t.patches;
  if (a.ip_act >= 0) point_patches &= ~(1u << a.ip_act);
#pragma unroll 1
  for (int j = 0; j < a.nstages; ++j) {
    const int stage = 4 - (j & 3), buf = j & 1;
    const int jn = min(j + 1, a.nstages - 1);
    double q[kLN];
#pragma unroll
    for (int l = 0; l < kLN; ++l) {
      q[l] = qn[l];
      qn[l] = glob(a.q[jn])[(inst * kLN + l) * N + t.gi];   // for the next stage
      sl[buf][l][t.e + 4] = v[l];
    }
    __syncthreads();
    if (!holds(c, t.e, j)) continue;
    if (act) {
      // ThermalActuator gradient and sensitivity on the pre-update adjoint state
      if (a.grad) glob(a.grad)[inst * a.grad_stride - (long)j * a.na + ka] = v[2] * (ma * 1.0);
      if (a.spartial) {
        const double F = v[2] * ma * 1.0;
        const double gn = (hw * 1.0) * h;   // gnorm<1>
        glob(a.spartial)[(inst * a.nslots + a.slot - j) * a.npts + ka] = 1.0 * gn * (F * F);
      }
    }
    double T[kLN], r[kLN], A[9];
    line_derivative<12, 16>(sl[buf], t, c, d, tab, d1, T);
    const Prim<1> s = prim<1>(q, g.gamma);
    const double m1[1] = {1.0};
    inviscid_jacobian<1>(m1, s, g.gamma, A);
#pragma unroll
    for (int i = 0; i < kLN; ++i) {
      double w = 0.0;
#pragma unroll
      for (int k = 0; k < kLN; ++k) w += A[i * 3 + k] * T[k];
      r[i] = 0.0 + w;
    }
    if (g.dissipation) line_dissipation(g, sl[buf], t, c, tab + 384, hw, -g.diss_amount, r);
#pragma unroll
    for (int l = 0; l < kLN; ++l) r[l] = r[l] * jac;
    for (unsigned m = point_patches; m; m &= m - 1) {
      const DPatch& pt = patches->p[__ffs(m) - 1];
      const int k = t.gi - pt.lo[0];
      switch (pt.type) {
        case MGD_PATCH_FAR_FIELD: {
          const double* Ap = pt.aplus + (long)k * 9;
          const double sj = pt.sigma_inv * jac;
#pragma unroll
          for (int i = 0; i < kLN; ++i) {
            double w = 0.0;
#pragma unroll
            for (int l = 0; l < kLN; ++l) w += Ap[i * 3 + l] * v[l];
            r[i] = r[i] + sj * w;
          }
          break;
        }
        case MGD_PATCH_SPONGE: {
          const double sp = pt.strength[k];
#pragma unroll
          for (int l = 0; l < kLN; ++l) r[l] = r[l] + sp * v[l];
          break;
        }
        case MGD_PATCH_COST_TARGET: {
          // acoustic-noise adjoint forcing from the forward state (none at the last stage of
          // the run), scaled by the stage factor
          if (a.t1 - (j >> 2) == 0 && stage == 1) break;
          const double factor = stage == 4 ? 2.0 : (stage == 2 ? 0.5 : 1.0);
          const double F = -2.0 * mo * 1.0 * (g.gamma - 1.0) * (s.p - pb);
          const double ke = 0.0 + s.u[0] * s.u[0];
          r[0] = r[0] + factor * (0.5 * ke * F);
          r[1] = r[1] + factor * (-s.u[0] * F);
          r[2] = r[2] + factor * F;
          break;
        }
        case MGD_PATCH_KOLMOGOROV:
          r[0] = r[0] - v[1] * pt.strength[k];
          break;
        default:
          break;
      }
    }
    // RK4 adjoint stage update (substepAdjointRK4, src/RK4IntegratorImpl.f90:215-261)
    const double dt = a.dt;
#pragma unroll
    for (int l = 0; l < kLN; ++l) {
      if (stage == 4) {
        l0[l] = v[l];
        b2[l] = v[l] - div6(dt * r[l]);
        v[l] = v[l] - dt * r[l] / 2.0;
      } else if (stage == 1) {
        v[l] = b2[l] - div6(dt * r[l]);
      } else {
        b2[l] = b2[l] - div3(dt * r[l]);
        v[l] = stage == 3 ? l0[l] - dt * r[l] / 2.0 : l0[l] - dt * r[l];
      }
    }
  }
  if (t.own) {
#pragma unroll
    for (int l = 0; l < kLN; ++l) glob(a.out)[(inst * kLN + l) * N + t.gi] = v[l];
  }
}

// ------------------------------------------------------------------------ host side
// Work-groups of a launch of nstages stages: a piece, its halos and the columns of the ends that
// lie just beyond them fit the threads.
static int line_blocks(const Geo& g, int nstages) {
  const int own = kLT - 8 * nstages - 2 * kEnd;
  return (g.dir[0].len + own - 1) / own;
}

// Four steps per launch while the work-groups are few (up to some 2.5 per CU): a launch is then
// latency, and its halo work is done by CUs that would idle.  Forward us per step, four against
// one: 209 groups 8.4 / 11.3, 418: 9.6 / 11.3, 836: 13.4 / 13.1, 1672: 22.1 / 18.6, 4169 (one
// line of 400000): 49 / 36.
int line_steps(const Geo& g) {
  return (long)line_blocks(g, kLineStages) * g.ninst <= 640 ? kLineSteps : 1;
}

void launch_line_forward(const Geo& g, const Patches* P, const LineForward& a, hipStream_t st) {
  const int nb = line_blocks(g, a.nstages);
  k_line_forward<<<dim3(nb, g.ninst), kLT, 0, st>>>(g, P, nb, a);
}

void launch_line_adjoint(const Geo& g, const Patches* P, const LineAdjoint& a, hipStream_t st) {
  const int nb = line_blocks(g, a.nstages);
  k_line_adjoint<<<dim3(nb, g.ninst), kLT, 0, st>>>(g, P, nb, a);
}

}  // namespace mgd
