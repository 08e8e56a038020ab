// fused2d.hip -- one-launch-per-RK-stage kernels for 2-D inviscid flows on gfx950.
//
// A work-group owns one tile of at most TX x TY grid points of one instance.  It
// stages the operand (q for a forward stage, lambda for an adjoint stage) with a
// 4-point halo in LDS, forms the contravariant fluxes once per staged point, and
// computes for its points: the SBP 4-8 flux divergence in x and y, the artificial
// dissipation D4^T diag(-arc) D4 (or the composite operator) in x and y, the Jacobian
// scaling, the patch terms (far-field SAT, sponge, actuator, cost target, Kolmogorov),
// the acoustic source and the RK4 stage update -- each RK stage reads its operands
// once and writes its outputs once.
//
// Tiles come from a balanced partition of each direction (host side), so on a
// non-periodic direction the first and last tiles hold at least 12 points: every
// boundary-closure row then lies in one tile and its closure stencil (up to 16 wide
// for the adjoint operator) reads staged LDS data like the interior stencil does.
// Each tile carries a bit mask of the patches that intersect it.
//
// The functional / sensitivity quadrature terms are written per patch point and stage
// and reduced by a fixed-order tree, so J and the sensitivity are deterministic and
// independent of the tile shape and of scheduling.
#include "fused2d.h"
#include "rows.h"

namespace mgd {

constexpr int HX = 4, HY = 4;     // halo of the staged operand
constexpr int NV2 = 4;
constexpr int kMinEdgeTile = 12;    // closure depth of the adjoint 4-8 operator
constexpr int kRedThreads = 256;    // block size of the reduction kernels
constexpr int kFarPoints = 32;      // far-field points of one patch that a tile forms ahead

// Tile shape: TX x TY points, one thread per point.  A thread beyond a partial tile loads and
// stages clamped points and stores nothing.  LDS (doubles): the staged operand q[4][EY][EX];
// forward, the contravariant fluxes of the tile rows (x) and columns (y); the boundary closure
// rows of an edge tile; the far-field terms.
template <int TX_, int TY_>
struct Shape {
  static constexpr int TX = TX_, TY = TY_, NT = TX * TY;
  static_assert(NT % 64 == 0, "whole waves");
  static constexpr int EX = TX + 2 * HX, EY = TY + 2 * HY;
  // halo points (the corners are never read): x-halo columns, then y-halo rows
  static constexpr int kHalo = 2 * HX * TY + 2 * HY * TX;
  static constexpr int kHaloIters = (kHalo + NT - 1) / NT;
  static constexpr int SQ = NV2 * EY * EX, SFX = NV2 * TY * EX, SFY = NV2 * EY * TX;
  static constexpr int kFar = 2 * 4 * kFarPoints;
  // closure rows of both ends: first derivative 8 x 12 and composite 8 x 12 (or dissipation
  // transpose 5 x 7); adjoint derivative 12 x 16 and dissipation 8 x 12
  static constexpr int kTabF = 2 * 96 + 2 * 96, kTabA = 2 * 192 + 2 * 96;
  static constexpr int kFwdLds = SQ + SFX + SFY + kTabF + kFar;
  static constexpr int kAdjLds = SQ + kTabA + kFar;
  static constexpr int kDualLds = kFwdLds > kAdjLds ? kFwdLds : kAdjLds;
  // waves per SIMD that the LDS use allows (160 KiB per CU), the register budget: at most 4
  static constexpr int waves(int lds) {
    const int w = (160 * 1024) / (8 * lds) * NT / 64 / 4;
    return w < 1 ? 1 : w > 4 ? 4 : w;
  }
  // the tile splits into blocks of 8 x 8 points, one wave each (thread_point)
  static constexpr bool kQuads = TX % 8 == 0 && TY % 8 == 0;
};

struct TileGeo {
  int x0, y0, sx, sy;   // origin and size of the tile
  bool bx, by;          // at a non-periodic x / y boundary (closure rows in the tile)
};

// Tile of this launch block (XCD band map), or -1; its geometry from the balanced
// partition, with no memory access.
__device__ __forceinline__ int block_tile(const Tiling& T, int b) {
  const int tile = (b % kNumXcd) * T.band + b / kNumXcd;
  return tile < T.nbx * T.nby ? tile : -1;
}

__device__ __forceinline__ TileGeo tile_geo(const Geo& g, const Tiling& T, int tile) {
  const int bx = tile % T.nbx, by = tile / T.nbx;
  TileGeo t;
  t.x0 = bx * T.qx + min(bx, T.lx) + max(0, bx - (T.nbx - T.rx));
  t.sx = T.qx + (bx < T.lx || bx >= T.nbx - T.rx ? 1 : 0);
  t.y0 = by * T.qy + min(by, T.ly) + max(0, by - (T.nby - T.ry));
  t.sy = T.qy + (by < T.ly || by >= T.nby - T.ry ? 1 : 0);
  t.bx = !g.dir[0].periodic && (bx == 0 || bx == T.nbx - 1);
  t.by = !g.dir[1].periodic && (by == 0 || by == T.nby - 1);
  return t;
}

// Tile column tx and row ty of this thread.  Row-major in general; in a tile on a non-periodic
// x boundary each wave covers 8 x 8 points, so that the 8 closure columns of the first
// derivative fill whole waves (a wave with both kinds of columns runs both paths): the last
// block of columns ends with the tile (its closure columns on the right boundary), the others
// start from its left.  False: the thread has no point of its own.
template <class S>
__device__ __forceinline__ bool thread_point(const TileGeo& t, int* tx, int* ty) {
  const int e = threadIdx.x;
  if (S::kQuads && t.bx) {
    const int l = e & 63, w = e >> 6;
    constexpr int QX = S::TX / 8;
    const int cb = w % QX, c = l & 7;
    *ty = (l >> 3) + 8 * (w / QX);
    *tx = cb == QX - 1 ? t.sx - 8 + c : 8 * cb + c;
    return *ty < t.sy && (cb == QX - 1 || *tx < t.sx - 8);
  }
  *tx = e % S::TX;
  *ty = e / S::TX;
  return *tx < t.sx && *ty < t.sy;
}

// global index of an extended (halo) index, or -1 outside a non-periodic domain
__device__ __forceinline__ int ext_index(const Dir& dd, int gi) {
  if (gi >= 0 && gi < dd.len) return gi;
  if (!dd.periodic) return -1;
  return gi < 0 ? gi + dd.len - dd.off : gi - dd.len + dd.off;
}

// One halo point of this thread: its place (ex, ey) in the staged tile, grid indices and
// which halo it is (1 x, 2 y, 0 none: then (gi, gj) is a point of the tile).
struct HaloSlot {
  int ex, ey, gi, gj, kind;
};
template <class S>
__device__ __forceinline__ HaloSlot halo_slot(const Geo& g, const TileGeo& t, int it) {
  const int e = threadIdx.x + it * S::NT;
  HaloSlot h;
  bool in;
  if (e < 2 * HX * S::TY) {
    const int c = e % 8, r = e / 8;
    h.ex = c < 4 ? c : t.sx + c;
    h.ey = HY + r;
    in = r < t.sy;
    h.kind = 1;
  } else {
    const int e2 = e - 2 * HX * S::TY, r = e2 / S::TX, c = e2 % S::TX;
    h.ex = HX + c;
    h.ey = r < 4 ? r : t.sy + r;
    in = r < 8 && c < t.sx;
    h.kind = 2;
  }
  h.gi = ext_index(g.dir[0], t.x0 - HX + h.ex);
  h.gj = ext_index(g.dir[1], t.y0 - HY + h.ey);
  if (!in || h.gi < 0 || h.gj < 0) {
    h.kind = 0;
    h.gi = t.x0;
    h.gj = t.y0;
  }
  return h;
}

// Row of the 9-point symmetric operator c_0..c_4 about x, whose coefficients sum to zero:
// sum_k c_k (x_k - x).
__device__ __forceinline__ double sym9(double x, const double* p, const double* m, const double* c) {
  double s = c[1] * ((p[0] - x) + (m[0] - x));
#pragma unroll
  for (int k = 2; k <= 4; ++k) s = __fma_rn(c[k], (p[k - 1] - x) + (m[k - 1] - x), s);
  return s;
}

// Scale of the one-level (9-point) dissipation sum of the adjoint stage along a direction:
// amount H^-1 (-arc) of the two-level operator, amount of the composite one.
__device__ __forceinline__ double diss_scale(const Geo& g, double amount, double arc, double hw) {
  if (g.composite) return amount;
  double s = amount * -arc;
  if (hw != 1.0) s = s / hw;    // 1 away from the first / last boundary rows
  return s;
}

// The Jacobian part of the adjoint rhs for 2-D Euler (computeRhsAdjoint): r = sum_d A_d^T t_d
// with the flux Jacobians A_d of the Cartesian directions and t_d = metric_d T1[d].  The
// products are formed through the enthalpy, not through the entries of A_d (most of which
// are multiples of one another): 46 operations instead of some 170.
__device__ __forceinline__ void adj_jacobian_rows(const double* mx, const Prim<2>& s, double gamma,
                                                  const double (*T1)[NV2], double* r) {
  double t[NV2], w[NV2];
#pragma unroll
  for (int c = 0; c < NV2; ++c) {
    t[c] = mx[0] * T1[0][c];
    w[c] = mx[1] * T1[1][c];
  }
  const double u = s.u[0], v = s.u[1], ke = 0.5 * (u * u + v * v), H = s.T + ke;
  const double a = u * t[1] + v * t[2], b = u * w[1] + v * w[2];
  const double e = u * t[3] + v * w[3];
  const double z = (gamma - 1.0) * ((t[1] + w[2]) + e);
  r[0] = (ke * z - H * e) - (u * a + v * b);
  r[1] = ((t[0] + a) + H * t[3]) + ((u * t[1] + v * w[1]) - u * z);
  r[2] = ((w[0] + b) + H * w[3]) + ((u * t[2] + v * w[2]) - v * z);
  r[3] = z + e;
}

__device__ __forceinline__ bool in_patch(ConstPatch& pt, int i, int j) {
  return i >= pt.lo[0] && i <= pt.hi[0] && j >= pt.lo[1] && j <= pt.hi[1];
}

// The far-field terms of a tile formed ahead of the stencil work, while its operand loads are
// in flight: of the first two far-field patches in the tile with at most kFarPoints of its
// points, thread 4 k + i forms component i of point k -- sum_c A+[c][i] (q_c - qt_c)
// forward, sum_c A+[i][c] lambda_c adjoint -- into LDS, where the point's thread finds it
// (a chain of loads per patch at the end of the kernel otherwise, on the slowest tiles).
struct FarAhead {
  int ip[2];       // patch, or -1
  int i0[2], j0[2], w[2];
};
template <class S, bool ADJ>
__device__ __forceinline__ FarAhead far_ahead(const Geo& g, ConstPatches* P,
                                              const TileGeo& t, unsigned m, global_ptr<const double> x,
                                              double* ff) {
  FarAhead f;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    f.ip[s] = -1;
    f.i0[s] = f.j0[s] = f.w[s] = 0;
    if (!m) continue;
    const int ip = __ffs(m) - 1;
    m &= m - 1;
    ConstPatch& pt = P->p[ip];
    const int i0 = max(pt.lo[0], t.x0), i1 = min(pt.hi[0], t.x0 + t.sx - 1);
    const int j0 = max(pt.lo[1], t.y0), j1 = min(pt.hi[1], t.y0 + t.sy - 1);
    const int w = i1 - i0 + 1, n = w * (j1 - j0 + 1);
    if (n <= 0 || n > kFarPoints) continue;
    f.ip[s] = ip;
    f.i0[s] = i0;
    f.j0[s] = j0;
    f.w[s] = w;
    for (int e = threadIdx.x; e < 4 * n; e += S::NT) {
      const int k = e >> 2, i = e & 3;
      const int gi = i0 + k % w, gj = j0 + k / w;
      const long p = gi + (long)g.n[0] * gj;
      const int kp = (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]);
      const global_ptr<const double> A = glob(pt.aplus) + (long)kp * 16;
      double v = 0.0;
      if (ADJ) {
#pragma unroll
        for (int c = 0; c < NV2; ++c) v += A[i * 4 + c] * x[c * g.N + p];
      } else {
        const global_ptr<const double> qt = glob(pt.aplus) + (long)pt.np * 16 + (long)kp * 4;
#pragma unroll
        for (int c = 0; c < NV2; ++c) v += A[c * 4 + i] * (x[c * g.N + p] - qt[c]);
      }
      ff[s * 4 * kFarPoints + e] = v;
    }
  }
  return f;
}

// The terms of patch ip (one of those formed ahead) at grid point (gi, gj).
__device__ __forceinline__ void far_formed(const FarAhead& f, int ip, const double* ff, int gi,
                                           int gj, double* out) {
  const int s = ip == f.ip[0] ? 0 : 1;
  const double* x = ff + s * 4 * kFarPoints + 4 * ((gi - f.i0[s]) + f.w[s] * (gj - f.j0[s]));
#pragma unroll
  for (int l = 0; l < NV2; ++l) out[l] = x[l];
}

// -------------------------------------------------------------------------- forward
// What bounds the stage: on small grids (a few blocks per CU) the chain load - LDS - stencils -
// store of one block, so there is one barrier, and every operand is asked for before it; on
// batches the 160 bytes per point and stage (0.09 ms for 20 instances of 401 x 401 at the rate
// of a copy) beside 0.07 ms of FP64 issue and 0.06 ms of LDS reads, which overlap in part.
// Plain stores: the rows of a tile end inside cache lines that the neighbour completes, and
// non-temporal stores sent them to memory in pieces (8 x 273^2: 39.3 against 36.9 us).
// Against the stage with the dissipation's intermediates in LDS (three barriers, every patch
// read at the end): 401^2 15.2 -> 13.3 us, 201^2 10.8 -> 10.1, 20 x 401^2 191 -> 173.
// One forward stage on tile block `blk` of instance `inst` (uniform per work-group).
template <class S>
__device__ __forceinline__ void fwd_stage_body(const Geo& g, const Patches* patches,
                                               const Tiling& T, const FwdStage& a, int blk,
                                               long inst, double* lds) {
  constexpr int TX = S::TX, TY = S::TY, EX = S::EX, EY = S::EY, HS = S::kHaloIters;
  double* sq = lds;
  double* sfx = sq + S::SQ;
  double* sfy = sfx + S::SFX;
  double* tab = sfy + S::SFY;
  double* ff = tab + S::kTabF;
  const int tile = block_tile(T, blk);
  ConstPatches* P = (ConstPatches*)patches;
  if (tile < 0) return;   // block beyond the tiles of its XCD (uniform per block)
  const TileGeo t = tile_geo(g, T, tile);
  const long NVN = (long)NV2 * g.N;
  const global_ptr<const double> qi = glob(a.qin) + inst * NVN;
  const unsigned pmask = glob(T.pmask)[tile];
  int tx, ty;
  const bool mine = thread_point<S>(t, &tx, &ty);
  const int gi = t.x0 + (mine ? tx : 0), gj = t.y0 + (mine ? ty : 0);
  const long p = gi + (long)g.n[0] * gj;
  // the operand: own point and halo points, then everything else the thread will need, in
  // the order of use (a wait for a load waits for those issued before it)
  double v[NV2], hv[HS][NV2], hm[HS];
#pragma unroll
  for (int l = 0; l < NV2; ++l) v[l] = qi[l * g.N + p];
#pragma unroll
  for (int it = 0; it < HS; ++it) {
    const HaloSlot h = halo_slot<S>(g, t, it);
    const long pp = h.gi + (long)g.n[0] * h.gj;
#pragma unroll
    for (int l = 0; l < NV2; ++l) hv[it][l] = qi[l * g.N + pp];
    hm[it] = h.kind == 2 ? glob(g.h[0])[h.gi] : glob(g.h[1])[h.gj];   // metric<2> of the halo's direction
  }
  const double h0 = glob(g.h[0])[gi], hw0 = glob(g.hw[0])[gi], h1 = glob(g.h[1])[gj], hw1 = glob(g.hw[1])[gj];
  double d1[5];                     // interior coefficients
#pragma unroll
  for (int k = 1; k <= 4; ++k) d1[k] = g.ops[SLOT_FIRST].c[kMaxHW + k];
  const FarAhead far = far_ahead<S, false>(g, P, t, pmask & P->far_mask, qi, ff);
  if (t.bx || t.by) {
    stage_rows<S::NT, 8, 12>(g, SLOT_FIRST, tab);
    if (g.dissipation) {
      if (g.composite) stage_rows<S::NT, 8, 12>(g, SLOT_DISS, tab + 192);
      else stage_rows<S::NT, 5, 7>(g, SLOT_DISS_T, tab + 192);
    }
  }
  // stage the operand and the fluxes
  if (mine) {
    const Prim<2> s = prim<2>(v, g.gamma);
    double f0[NV2], f1[NV2];
    inviscid_flux<2>(v, s, 0, f0);
    inviscid_flux<2>(v, s, 1, f1);
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      sq[(l * EY + ty + HY) * EX + tx + HX] = v[l];
      sfx[(l * TY + ty) * EX + tx + HX] = h1 * f0[l];
      sfy[(l * EY + ty + HY) * TX + tx] = h0 * f1[l];
    }
  }
#pragma unroll
  for (int it = 0; it < HS; ++it) {
    const HaloSlot h = halo_slot<S>(g, t, it);
    if (h.kind == 0) continue;
    const Prim<2> s = prim<2>(hv[it], g.gamma);
    double f[NV2];
    if (h.kind == 1) {
      inviscid_flux<2>(hv[it], s, 0, f);
#pragma unroll
      for (int l = 0; l < NV2; ++l) sfx[(l * TY + h.ey - HY) * EX + h.ex] = hm[it] * f[l];
    } else {
      inviscid_flux<2>(hv[it], s, 1, f);
#pragma unroll
      for (int l = 0; l < NV2; ++l) sfy[(l * EY + h.ey) * TX + h.ex - HX] = hm[it] * f[l];
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) sq[(l * EY + h.ey) * EX + h.ex] = hv[it][l];
  }
  // RK operands, sponge, source and cost-target values, fetched while the stencils run
  const bool sponge = (pmask & P->sponge_mask) != 0;            // uniform per block
  const bool cost = a.jpartial && a.ip_cost >= 0 && ((pmask >> a.ip_cost) & 1u);
  double q0[NV2], b2[NV2], qt[NV2], damp = 0.0, sx0 = 0.0, sy0 = 0.0, pb = 0.0, mo = 0.0;
#pragma unroll
  for (int l = 0; l < NV2; ++l) {
    const long o = inst * NVN + l * g.N + p;
    q0[l] = a.stage == 2 || a.stage == 3 ? glob(a.q0)[o] : 0.0;
    b2[l] = a.stage >= 2 ? glob(a.b2)[o] : 0.0;
    qt[l] = 0.0;
  }
  if (sponge) {
    damp = glob(P->damp)[p];
#pragma unroll
    for (int l = 0; l < NV2; ++l) qt[l] = glob(P->qtarget)[l * g.N + p];
  }
  if (a.nsrc > 0) {
    sx0 = glob(P->srcx)[gi];
    sy0 = glob(P->srcy)[gj];
  }
  bool jin = false;
  int kj = 0;
  if (cost) {
    ConstPatch& pt = P->p[a.ip_cost];
    jin = mine && in_patch(pt, gi, gj);
    kj = jin ? (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]) : 0;
    pb = glob(pt.aplus)[kj];
    mo = glob(pt.strength)[kj];
  }
  __syncthreads();
  // r = 0 - (D_x F_x + D_y F_y) and the dissipation in x and y
  double r[NV2];
  const double ax = -fabs(h1), ay = -fabs(h0);          // -arc length along x, y
  const double* fx = sfx + ty * EX + tx + HX;           // the point in the staged arrays
  const double* fy = sfy + (ty + HY) * TX + tx;
  const double* qc = sq + (ty + HY) * EX + tx + HX;
  if (!mine) {
    // nothing: no point of its own
  } else if (!t.bx && !t.by) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      double xp[4], xm[4], yp[4], ym[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        xp[k] = fx[l * TY * EX + k + 1];
        xm[k] = fx[l * TY * EX - (k + 1)];
        yp[k] = fy[(l * EY + k + 1) * TX];
        ym[k] = fy[(l * EY - (k + 1)) * TX];
      }
      __builtin_amdgcn_sched_barrier(0);   // one batch of LDS reads, one wait
      r[l] = 0.0 - (skew_sum(xp, xm, d1) + skew_sum(yp, ym, d1));
    }
  } else {
    const EdgePlace ex = edge_place(g.dir[0], gi), ey = edge_place(g.dir[1], gj);
    double dx[NV2], dy[NV2];
    if (t.bx && ex.m < 8) {
      const double* b = sfx + ty * EX + HX + (ex.right ? t.sx - 12 : 0);
      closure_row<NV2, 12>(tab + 12 * ex.m + (ex.right ? 96 : 0),
                      [&](int j, int k) { return b[j * TY * EX + k]; }, dx);
    } else {
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        const double* x = fx + l * TY * EX;
        const double xp[4] = {x[1], x[2], x[3], x[4]}, xm[4] = {x[-1], x[-2], x[-3], x[-4]};
        dx[l] = skew_sum(xp, xm, d1);
      }
    }
    if (t.by && ey.m < 8) {
      const double* b = sfy + (HY + (ey.right ? t.sy - 12 : 0)) * TX + tx;
      closure_row<NV2, 12>(tab + 12 * ey.m + (ey.right ? 96 : 0),
                      [&](int j, int k) { return b[(j * EY + k) * TX]; }, dy);
    } else {
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        const double* c = fy + l * EY * TX;
        const double yp[4] = {c[TX], c[2 * TX], c[3 * TX], c[4 * TX]};
        const double ym[4] = {c[-TX], c[-2 * TX], c[-3 * TX], c[-4 * TX]};
        dy[l] = skew_sum(yp, ym, d1);
      }
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = 0.0 - (dx[l] + dy[l]);
  }
  if (g.dissipation && mine) {
    if (g.composite) {
      const EdgePlace ex = edge_place(g.dir[0], gi), ey = edge_place(g.dir[1], gj);
#pragma unroll 1
      for (int d = 0; d < 2; ++d) {
        const EdgePlace e = d == 0 ? ex : ey;
        const int step = d == 0 ? 1 : EX;
        double dv[NV2];
        if (e.m < 8) {
          const double* b = d == 0 ? sq + (ty + HY) * EX + HX + (e.right ? t.sx - 12 : 0)
                                   : sq + (HY + (e.right ? t.sy - 12 : 0)) * EX + tx + HX;
          closure_row<NV2, 12>(tab + 192 + 12 * e.m + (e.right ? 96 : 0),
                          [&](int j, int k) { return b[j * EY * EX + k * step]; }, dv);
        } else {
#pragma unroll
          for (int l = 0; l < NV2; ++l) {
            const double* x = qc + l * EY * EX;
            double s = 0.0;
#pragma unroll
            for (int k = 1; k <= 4; ++k)
              s += g.ops[SLOT_DISS].c[kMaxHW + k] * (x[k * step] + x[-k * step]);
            dv[l] = s + g.ops[SLOT_DISS].c[kMaxHW] * x[0];
          }
        }
#pragma unroll
        for (int l = 0; l < NV2; ++l) r[l] = r[l] + g.diss_amount * dv[l];
      }
    } else if (!t.bx && !t.by) {
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        double w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = k == 4 ? v[l] : qc[l * EY * EX + k - 4];
        __builtin_amdgcn_sched_barrier(0);
        r[l] = r[l] + g.diss_amount * two_level(w, ax);
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = k == 4 ? v[l] : qc[(l * EY + k - 4) * EX];
        __builtin_amdgcn_sched_barrier(0);
        r[l] = r[l] + g.diss_amount * two_level(w, ay);
      }
    } else {
      const EdgePlace ex = edge_place(g.dir[0], gi), ey = edge_place(g.dir[1], gj);
      // the windows of nine operands, moved inside the domain at its ends
      const double* bx = qc - 4 + (ex.m < 4 ? (ex.right ? ex.m - 4 : 4 - ex.m) : 0);
      const double* by = qc + (-4 + (ey.m < 4 ? (ey.right ? ey.m - 4 : 4 - ey.m) : 0)) * EX;
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        double w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = bx[l * EY * EX + k];
        double dv = two_level_edge(w, ax, ex, tab + 192);
        if (hw0 != 1.0) dv = dv / hw0;   // 1 away from the first / last boundary rows
        r[l] = r[l] + g.diss_amount * dv;
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = by[(l * EY + k) * EX];
        dv = two_level_edge(w, ay, ey, tab + 192);
        if (hw1 != 1.0) dv = dv / hw1;
        r[l] = r[l] + g.diss_amount * dv;
      }
    }
  }
  if (!mine) return;
  // point terms, RK4 stage update (substepForwardRK4, src/RK4IntegratorImpl.f90:115-156) and
  // the functional term of the new stage state
  const double dt = a.dt;
  const double jac = 1.0 / (h0 * h1);   // jacobian<2>
#pragma unroll
  for (int l = 0; l < NV2; ++l) r[l] = r[l] * jac;
  // far fields, then sponges, then the other patches, each in the order of the patches
  for (unsigned m = pmask & P->far_mask; m; m &= m - 1) {
    const int ip = __ffs(m) - 1;
    ConstPatch& pt = P->p[ip];
    if (!in_patch(pt, gi, gj)) continue;
    const double sj = pt.sigma_inv * jac;
    double f[NV2];
    if (ip == far.ip[0] || ip == far.ip[1]) {
      far_formed(far, ip, ff, gi, gj, f);
    } else {
      const int kp = (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]);
      const global_ptr<const double> A = glob(pt.aplus) + (long)kp * 16;
      const global_ptr<const double> qf = glob(pt.aplus) + (long)pt.np * 16 + (long)kp * 4;
#pragma unroll
      for (int i = 0; i < NV2; ++i) {
        f[i] = 0.0;
#pragma unroll
        for (int c = 0; c < NV2; ++c) f[i] += A[c * 4 + i] * (v[c] - qf[c]);
      }
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] - sj * f[l];
  }
  if (damp != 0.0) {      // 0 outside the sponges, whatever the target holds there
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] - damp * (v[l] - qt[l]);
  }
  unsigned rest = pmask & ~(P->sponge_mask | P->far_mask);
  if (a.ip_cost >= 0) rest &= ~(1u << a.ip_cost);
  while (rest) {
    const int ip = __ffs(rest) - 1;
    rest &= rest - 1;
    ConstPatch& pt = P->p[ip];
    if (!in_patch(pt, gi, gj)) continue;
    const int kp = (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]);
    switch (pt.type) {
      case MGD_PATCH_ACTUATOR:
        if (a.control) r[3] = r[3] + glob(pt.strength)[kp] * glob(a.control)[inst * a.control_stride + kp];
        break;
      case MGD_PATCH_KOLMOGOROV:
        r[1] = r[1] + v[0] * glob(pt.strength)[kp];
        break;
      default:
        break;
    }
  }
  // Gaussian sources: exp(-g (dx^2 + dy^2)) as the product of its 1-D factors
  if (a.nsrc > 0) r[3] = r[3] + glob(a.src_amp)[inst * a.src_inst_stride] * (sx0 * sy0);
  for (int s = 1; s < a.nsrc; ++s)
    r[3] = r[3] + glob(a.src_amp)[inst * a.src_inst_stride + s] *
                      (glob(P->srcx)[(long)s * g.n[0] + gi] * glob(P->srcy)[(long)s * g.n[1] + gj]);
  double qn[NV2];
#pragma unroll
  for (int l = 0; l < NV2; ++l) {
    const long o = inst * NVN + l * g.N + p;
    const double rl = r[l];
    if (a.stage == 1) {
      glob(a.b2)[o] = v[l] + div6(dt * rl);
      qn[l] = v[l] + dt * rl / 2.0;
    } else if (a.stage == 2) {
      glob(a.b2)[o] = b2[l] + div3(dt * rl);
      qn[l] = q0[l] + dt * rl / 2.0;
    } else if (a.stage == 3) {
      glob(a.b2)[o] = b2[l] + div3(dt * rl);
      qn[l] = q0[l] + dt * rl;
    } else {
      qn[l] = b2[l] + div6(dt * rl);
    }
    glob(a.qout)[o] = qn[l];
    if (a.rhs_out) glob(a.rhs_out)[o] = rl;
  }
  if (cost && jin) {
    const Prim<2> s = prim<2>(qn, g.gamma);
    const double F = s.p - pb;
    const double gn = (hw1 * (hw0 * 1.0)) * (h0 * h1);   // gnorm<2>
    glob(a.jpartial)[(inst * a.nslots + a.slot) * a.npts + kj] = 1.0 * gn * (F * F * mo);
  }
}

// -------------------------------------------------------------------------- adjoint
// Bounded as the forward stage is (192 bytes per point and stage: 0.11 ms for 20 x 401^2).
// Both directions' dissipation is one 9-point operator (SLOT_DISS2) on the staged values that
// D+ reads anyway, and the Jacobian products go through the enthalpy.  The RK operands are
// loaded behind the stencils: held across them, they cost 100 bytes of scratch per thread and
// 0.1 ms (20 x 401^2: 252 against 162 us; with the edge tiles' closures kept from spilling the
// last 20 bytes, 141).  Before: 401^2 15.1 -> 12.1 us, 201^2 10.8 -> 9.4, 20 x 401^2 170 -> 142.
// One adjoint stage on tile block `blk` of instance `inst` (uniform per work-group).
template <class S>
__device__ __forceinline__ void adj_stage_body(const Geo& g, const Patches* patches,
                                               const Tiling& T, const AdjStage& a, int blk,
                                               long inst, double* lds) {
  constexpr int EX = S::EX, EY = S::EY, HS = S::kHaloIters;
  double* sq = lds;
  double* tab = sq + S::SQ;
  double* ff = tab + S::kTabA;
  const int tile = block_tile(T, blk);
  ConstPatches* P = (ConstPatches*)patches;
  if (tile < 0) return;   // block beyond the tiles of its XCD (uniform per block)
  const TileGeo t = tile_geo(g, T, tile);
  const long NVN = (long)NV2 * g.N;
  const global_ptr<const double> li = glob(a.lam) + inst * NVN;
  const global_ptr<const double> qi = glob(a.q) + inst * NVN;
  const unsigned pmask = glob(T.pmask)[tile];
  int tx, ty;
  const bool mine = thread_point<S>(t, &tx, &ty);
  const int gi = t.x0 + (mine ? tx : 0), gj = t.y0 + (mine ? ty : 0);
  const long p = gi + (long)g.n[0] * gj;
  double v[NV2], hv[HS][NV2], q[NV2];
#pragma unroll
  for (int l = 0; l < NV2; ++l) v[l] = li[l * g.N + p];
#pragma unroll
  for (int it = 0; it < HS; ++it) {
    const HaloSlot h = halo_slot<S>(g, t, it);
    const long pp = h.gi + (long)g.n[0] * h.gj;
#pragma unroll
    for (int l = 0; l < NV2; ++l) hv[it][l] = li[l * g.N + pp];
  }
  double d1[5], ds[5];              // interior coefficients
#pragma unroll
  for (int k = 0; k <= 4; ++k) {
    d1[k] = g.ops[SLOT_ADJ].c[kMaxHW + k];
    ds[k] = g.ops[SLOT_DISS2].c[kMaxHW + k];
  }
  const FarAhead far = far_ahead<S, true>(g, P, t, pmask & P->far_mask, li, ff);
  if (t.bx || t.by) {
    stage_rows<S::NT, 12, 16>(g, SLOT_ADJ, tab);
    if (g.dissipation) stage_rows<S::NT, 8, 12>(g, SLOT_DISS2, tab + 384);
  }
  if (mine) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) sq[(l * EY + ty + HY) * EX + tx + HX] = v[l];
  }
#pragma unroll
  for (int it = 0; it < HS; ++it) {
    const HaloSlot h = halo_slot<S>(g, t, it);
    if (h.kind == 0) continue;
#pragma unroll
    for (int l = 0; l < NV2; ++l) sq[(l * EY + h.ey) * EX + h.ex] = hv[it][l];
  }
  // the forward stage state at the point and the grid values, fetched while the stencils run
#pragma unroll
  for (int l = 0; l < NV2; ++l) q[l] = qi[l * g.N + p];
  const double h0 = glob(g.h[0])[gi], hw0 = glob(g.hw[0])[gi], h1 = glob(g.h[1])[gj], hw1 = glob(g.hw[1])[gj];
  __syncthreads();
  if (!mine) return;
  // D+ lambda along x and y (T1) and the dissipation (w), from the same staged values
  double T1[2][NV2], w[NV2], l0[NV2], b2[NV2];
  const double* lc = sq + (ty + HY) * EX + tx + HX;   // the point in the staged tile
  const double sx = diss_scale(g, -g.diss_amount, fabs(h1), hw0);
  const double sy = diss_scale(g, -g.diss_amount, fabs(h0), hw1);
  if (!t.bx && !t.by) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      double xp[4], xm[4], yp[4], ym[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        xp[k] = lc[l * EY * EX + k + 1];
        xm[k] = lc[l * EY * EX - (k + 1)];
        yp[k] = lc[(l * EY + k + 1) * EX];
        ym[k] = lc[(l * EY - (k + 1)) * EX];
      }
      __builtin_amdgcn_sched_barrier(0);   // one batch of LDS reads, one wait
      T1[0][l] = skew_sum(xp, xm, d1);
      T1[1][l] = skew_sum(yp, ym, d1);
      w[l] = sx * sym9(v[l], xp, xm, ds) + sy * sym9(v[l], yp, ym, ds);
    }
  } else {
    const EdgePlace ex = edge_place(g.dir[0], gi), ey = edge_place(g.dir[1], gj);
    // the 16 (12) staged values at the end of the line
    const int ox = ex.right ? t.sx - 1 : 0, oy = ey.right ? t.sy - 1 : 0;
    const double* bx = sq + (ty + HY) * EX + HX + ox;
    const double* by = sq + (HY + oy) * EX + tx + HX;
    const int rx = ex.right ? 15 : 0, ry = ey.right ? 15 : 0;
    const int qx = ex.right ? 11 : 0, qy = ey.right ? 11 : 0;
    const bool cx = t.bx && ex.m < 12, cy = t.by && ey.m < 12;
    double dv[NV2];
    if (cx)
      closure_row<NV2, 16>(tab + 16 * ex.m + (ex.right ? 192 : 0),
                      [&](int j, int k) { return bx[j * EY * EX + k - rx]; }, T1[0]);
    if (t.bx && ex.m < 8) {
      if (g.dissipation)
        closure_row<NV2, 12>(tab + 384 + 12 * ex.m + (ex.right ? 96 : 0),
                        [&](int j, int k) { return bx[j * EY * EX + k - qx] - v[j]; }, dv);
    } else {
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        const double* x = lc + l * EY * EX;
        const double xp[4] = {x[1], x[2], x[3], x[4]}, xm[4] = {x[-1], x[-2], x[-3], x[-4]};
        if (!cx) T1[0][l] = skew_sum(xp, xm, d1);
        dv[l] = sym9(v[l], xp, xm, ds);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) w[l] = sx * dv[l];
    if (cy)
      closure_row<NV2, 16>(tab + 16 * ey.m + (ey.right ? 192 : 0),
                      [&](int j, int k) { return by[(j * EY + k - ry) * EX]; }, T1[1]);
    if (t.by && ey.m < 8) {
      if (g.dissipation)
        closure_row<NV2, 12>(tab + 384 + 12 * ey.m + (ey.right ? 96 : 0),
                        [&](int j, int k) { return by[(j * EY + k - qy) * EX] - v[j]; }, dv);
    } else {
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        const double* c = lc + l * EY * EX;
        const double yp[4] = {c[EX], c[2 * EX], c[3 * EX], c[4 * EX]};
        const double ym[4] = {c[-EX], c[-2 * EX], c[-3 * EX], c[-4 * EX]};
        if (!cy) T1[1][l] = skew_sum(yp, ym, d1);
        dv[l] = sym9(v[l], yp, ym, ds);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) w[l] = w[l] + sy * dv[l];
  }
  // here, not before: the closure rows need the registers
  const bool sponge = (pmask & P->sponge_mask) != 0;            // uniform per block
  const double damp = sponge ? glob(P->damp)[p] : 0.0;
#pragma unroll
  for (int l = 0; l < NV2; ++l) {
    const long o = inst * NVN + l * g.N + p;
    l0[l] = a.stage == 3 || a.stage == 2 ? glob(a.l0)[o] : 0.0;
    b2[l] = a.stage <= 3 ? glob(a.b2)[o] : 0.0;
  }
  const Prim<2> s = prim<2>(q, g.gamma);
  double r[NV2];
  const double mx[2] = {h1, h0};   // metric<2>(g, 0, .), metric<2>(g, 1, .)
  adj_jacobian_rows(mx, s, g.gamma, T1, r);
  const double jac = 1.0 / (h0 * h1);   // jacobian<2>
#pragma unroll
  for (int l = 0; l < NV2; ++l) r[l] = (g.dissipation ? r[l] + w[l] : r[l]) * jac;
  // far fields, then sponges, then the other patches, each in the order of the patches
  for (unsigned m = pmask & P->far_mask; m; m &= m - 1) {
    const int ip = __ffs(m) - 1;
    ConstPatch& pt = P->p[ip];
    if (!in_patch(pt, gi, gj)) continue;
    const double sj = pt.sigma_inv * jac;
    double f[NV2];
    if (ip == far.ip[0] || ip == far.ip[1]) {
      far_formed(far, ip, ff, gi, gj, f);
    } else {
      const int kp = (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]);
      const global_ptr<const double> A = glob(pt.aplus) + (long)kp * 16;
#pragma unroll
      for (int i = 0; i < NV2; ++i) {
        f[i] = 0.0;
#pragma unroll
        for (int c = 0; c < NV2; ++c) f[i] += A[i * 4 + c] * v[c];
      }
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] + sj * f[l];
  }
  if (sponge) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] + damp * v[l];
  }
  unsigned rest = pmask & ~(P->sponge_mask | P->far_mask);
  while (rest) {
    const int ip = __ffs(rest) - 1;
    rest &= rest - 1;
    ConstPatch& pt = P->p[ip];
    if (!in_patch(pt, gi, gj)) continue;
    const int kp = (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]);
    switch (pt.type) {
      case MGD_PATCH_COST_TARGET: {
        // acoustic-noise adjoint forcing from the forward state at this point
        // (src/AcousticNoiseImpl.f90:208-280), scaled by the stage factor
        if (a.zero_forcing) break;
        const double F = -2.0 * glob(pt.strength)[kp] * 1.0 * (g.gamma - 1.0) * (s.p - glob(pt.aplus)[kp]);
        const double ke = s.u[0] * s.u[0] + s.u[1] * s.u[1];
        r[0] = r[0] + a.forcing_factor * (0.5 * ke * F);
        r[1] = r[1] + a.forcing_factor * (-s.u[0] * F);
        r[2] = r[2] + a.forcing_factor * (-s.u[1] * F);
        r[3] = r[3] + a.forcing_factor * F;
        break;
      }
      case MGD_PATCH_ACTUATOR: {
        // ThermalActuator gradient and sensitivity on the pre-update adjoint state
        if (a.grad) glob(a.grad)[inst * a.grad_stride + kp] = v[3] * (glob(pt.strength)[kp] * 1.0);
        if (a.spartial) {
          const double F = v[3] * glob(pt.strength)[kp] * 1.0;
          const double gn = (glob(g.hw[1])[gj] * (glob(g.hw[0])[gi] * 1.0)) * (h0 * h1);   // gnorm<2>
          glob(a.spartial)[(inst * a.nslots + a.slot) * a.npts + kp] = 1.0 * gn * (F * F);
        }
        break;
      }
      case MGD_PATCH_KOLMOGOROV:
        r[0] = r[0] - v[1] * glob(pt.strength)[kp];
        break;
      default:
        break;
    }
  }
  // RK4 adjoint stage update (substepAdjointRK4, src/RK4IntegratorImpl.f90:215-261)
  const double dt = a.dt;
#pragma unroll
  for (int l = 0; l < NV2; ++l) {
    const long o = inst * NVN + l * g.N + p;
    const double rl = r[l];
    double ln;
    if (a.stage == 4) {
      glob(a.b2)[o] = v[l] - div6(dt * rl);
      ln = v[l] - dt * rl / 2.0;
    } else if (a.stage == 3) {
      glob(a.b2)[o] = b2[l] - div3(dt * rl);
      ln = l0[l] - dt * rl / 2.0;
    } else if (a.stage == 2) {
      glob(a.b2)[o] = b2[l] - div3(dt * rl);
      ln = l0[l] - dt * rl;
    } else {
      ln = b2[l] - div6(dt * rl);
    }
    glob(a.lout)[o] = ln;
    if (a.rhs_out) glob(a.rhs_out)[o] = rl;
  }
}

template <class S>
__global__ void __launch_bounds__(S::NT, S::waves(S::kFwdLds)) k_fwd_stage2d(Geo g, const Patches* __restrict__ P,
                                                       Tiling T, FwdStage a) {
  __shared__ double lds[S::kFwdLds];
  fwd_stage_body<S>(g, P, T, a, blockIdx.x, blockIdx.y, lds);
}

template <class S>
__global__ void __launch_bounds__(S::NT, S::waves(S::kAdjLds)) k_adj_stage2d(Geo g, const Patches* __restrict__ P,
                                                       Tiling T, AdjStage a) {
  __shared__ double lds[S::kAdjLds];
  adj_stage_body<S>(g, P, T, a, blockIdx.x, blockIdx.y, lds);
}

// One adjoint stage and one forward stage of the same region in one launch: blocks
// [0, nblk) run the adjoint stage's tiles, blocks [nblk, 2 nblk) the forward stage's (the
// window recompute beside the adjoint of the next window: independent states, so the
// same values as two launches).  nblk is a multiple of 8, so a block's XCD -- its index
// mod 8 -- is the one its tile is dealt to either way.
template <class S>
__global__ void __launch_bounds__(S::NT, S::waves(S::kDualLds)) k_dual_stage2d(Geo g, const Patches* __restrict__ P,
                                                        Tiling T, AdjStage a, FwdStage f) {
  __shared__ double lds[S::kDualLds];
  if ((int)blockIdx.x < T.nblk) adj_stage_body<S>(g, P, T, a, blockIdx.x, blockIdx.y, lds);
  else fwd_stage_body<S>(g, P, T, f, (int)blockIdx.x - T.nblk, blockIdx.y, lds);
}

// Block sum: wave-level shuffles, then one LDS exchange of the per-wave sums.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  __syncthreads();   // retire earlier readers of the scratch space
  const int w = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int k = 0; k < NT / 64; ++k) s += red[k];
  return s;
}

// Several regions in one launch: launch block k belongs to the member m with
// mem[m].block0 <= k < mem[m + 1].block0 (members in block order), which sees it as tile
// block (k - block0) mod nblk of instance (k - block0) / nblk.  args[m]: the stage of m.
__device__ __forceinline__ int group_member(const GroupMember* mem, int nmem, int* blk,
                                            long* inst) {
  int m = 0;
  while (m + 1 < nmem && (int)blockIdx.x >= mem[m + 1].block0) ++m;
  const int lb = (int)blockIdx.x - mem[m].block0;
  *blk = lb % mem[m].T.nblk;
  *inst = lb / mem[m].T.nblk;
  return m;
}

template <class S>
__global__ void __launch_bounds__(S::NT, S::waves(S::kFwdLds))
    k_fwd_stage2d_group(const GroupMember* __restrict__ mem, int nmem, const FwdStage* __restrict__ args) {
  __shared__ double lds[S::kFwdLds];
  int blk;
  long inst;
  const int m = group_member(mem, nmem, &blk, &inst);
  const GroupMember& gm = mem[m];
  fwd_stage_body<S>(gm.g, gm.P, gm.T, args[m], blk, inst, lds);
}

template <class S>
__global__ void __launch_bounds__(S::NT, 3)   // the descriptors in scalar registers leave fewer for addresses
    k_adj_stage2d_group(const GroupMember* __restrict__ mem, int nmem, const AdjStage* __restrict__ args) {
  __shared__ double lds[S::kAdjLds];
  int blk;
  long inst;
  const int m = group_member(mem, nmem, &blk, &inst);
  const GroupMember& gm = mem[m];
  adj_stage_body<S>(gm.g, gm.P, gm.T, args[m], blk, inst, lds);
}

// Stage sums of the per-point quadrature terms of one chunk of stages: one block of
// kSumThreads per (stage, instance), a fixed-order tree over the points.
constexpr int kSumThreads = 1024;
__global__ void __launch_bounds__(kSumThreads) k_stage_sums(const double* __restrict__ partial,
                                                            int nslots, int npts,
                                                            double* __restrict__ sums,
                                                            int nstages, int base) {
  __shared__ double red[kSumThreads / 64];
  const int s = blockIdx.x;
  const long inst = blockIdx.y;
  const double* src = partial + (inst * nslots + s) * (long)npts;
  double v = 0.0;
  for (int k = threadIdx.x; k < npts; k += kSumThreads) v += src[k];
  const double sum = block_sum<kSumThreads>(v, red);
  if (threadIdx.x == 0) sums[inst * nstages + base + s] = sum;
}

// acc[inst] += w[s] * sums[s] over the stages in time-marching order (the running time
// quadrature of Solver%runForward / runAdjoint); reverse = adjoint order.  One block
// per instance: the products are formed in parallel into LDS, one chunk at a time, and
// added by one thread in stage order (the order of the running sum).
__global__ void __launch_bounds__(kRedThreads) k_stage_accumulate(
    const double* __restrict__ sums, int nstages, const double* __restrict__ w,
    double* __restrict__ acc, int reverse) {
  constexpr int kChunk = 2048;
  __shared__ double prod[kChunk];
  const long inst = blockIdx.x;
  double total = acc[inst];
  for (int c0 = 0; c0 < nstages; c0 += kChunk) {
    const int n = min(kChunk, nstages - c0);
    __syncthreads();
    for (int k = threadIdx.x; k < n; k += kRedThreads) {
      const int s = reverse ? nstages - 1 - (c0 + k) : c0 + k;
      prod[k] = w[s] * sums[inst * nstages + s];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll 8
      for (int k = 0; k < n; ++k) total = total + prod[k];
    }
  }
  if (threadIdx.x == 0) acc[inst] = total;
}

// ------------------------------------------------------------------------ host side
using S32x16 = Shape<32, 16>;
using S16x32 = Shape<16, 32>;
using S16x16 = Shape<16, 16>;
using S24x16 = Shape<24, 16>;
using S16x24 = Shape<16, 24>;
using S16x12 = Shape<16, 12>;

static const int kShapeDims[kNumTileShapes][2] = {{32, 16}, {16, 32}, {16, 16}, {24, 16},
                                                  {16, 24}, {16, 12}};

int fused2d_shape_dims(int shape, int* tx, int* ty) {
  if (shape < 0 || shape >= kNumTileShapes) return MGD_ERR_ARG;
  *tx = kShapeDims[shape][0];
  *ty = kShapeDims[shape][1];
  return MGD_OK;
}

// Balanced partition of len points into n = ceil(len / T) tiles of q or q + 1 points,
// the larger ones at both ends (l leading, r trailing: the edge tiles are the largest,
// as the boundary closures need): tile b holds q + (b < l || b >= n - r) points.
static void balanced(int len, int T, std::vector<int>& org, std::vector<int>& size, int* q,
                     int* l, int* r) {
  const int n = (len + T - 1) / T;
  const int extra = len % n;
  *q = len / n;
  *l = (extra + 1) / 2;
  *r = extra / 2;
  int o = 0;
  for (int b = 0; b < n; ++b) {
    const int sz = *q + (b < *l || b >= n - *r ? 1 : 0);
    org.push_back(o);
    size.push_back(sz);
    o += sz;
  }
}

int fused2d_make_tiling(const Geo& g, const Patches& hp, int shape, HostTiling* out) {
  int tx, ty;
  if (fused2d_shape_dims(shape, &tx, &ty) != MGD_OK) return MGD_ERR_ARG;
  out->shape = shape;
  out->org.clear();
  out->size.clear();
  balanced(g.n[0], tx, out->org, out->size, &out->qx, &out->lx, &out->rx);
  out->nbx = (int)out->org.size();
  balanced(g.n[1], ty, out->org, out->size, &out->qy, &out->ly, &out->ry);
  out->nby = (int)out->org.size() - out->nbx;
  for (int d = 0; d < 2; ++d) {
    if (g.dir[d].periodic) continue;
    const int first = d == 0 ? 0 : out->nbx;
    const int last = d == 0 ? out->nbx - 1 : out->nbx + out->nby - 1;
    if (out->size[first] < kMinEdgeTile || out->size[last] < kMinEdgeTile) return MGD_ERR_UNSUPPORTED;
  }
  out->pmask.assign((size_t)out->nbx * out->nby, 0u);
  for (int by = 0; by < out->nby; ++by)
    for (int bx = 0; bx < out->nbx; ++bx) {
      const int xa = out->org[bx], xb = xa + out->size[bx] - 1;
      const int ya = out->org[out->nbx + by], yb = ya + out->size[out->nbx + by] - 1;
      unsigned m = 0;
      for (int ip = 0; ip < hp.count; ++ip) {
        const DPatch& pt = hp.p[ip];
        if (xb < pt.lo[0] || xa > pt.hi[0] || yb < pt.lo[1] || ya > pt.hi[1]) continue;
        m |= 1u << ip;
      }
      out->pmask[(size_t)by * out->nbx + bx] = m;
    }
  // XCD-aware block -> tile map.  Work-groups are dealt to the XCDs round-robin by
  // linear block index, and each XCD has its own L2: XCD x receives blocks x, x + 8, ...
  // which are mapped to one contiguous band of tiles (row-major), so neighbouring tiles
  // -- whose halos overlap -- share an L2.  Bands hold ceil(ntiles / 8) tiles; the spare
  // blocks of the last band map to -1 and exit at once.
  const int ntiles = out->nbx * out->nby;
  const int band = (ntiles + kNumXcd - 1) / kNumXcd;
  out->band = band;
  out->nblk = band * kNumXcd;
  out->tile_of_block.assign((size_t)out->nblk, -1);
  for (int b = 0; b < out->nblk; ++b) {
    const int pos = (b % kNumXcd) * band + b / kNumXcd;
    out->tile_of_block[(size_t)b] = pos < ntiles ? pos : -1;
  }
  return MGD_OK;
}

template <class S>
static void fwd_group_launch(const GroupMember* mem, int nmem, int nblocks, const FwdStage* args,
                             hipStream_t st) {
  k_fwd_stage2d_group<S><<<nblocks, S::NT, 0, st>>>(mem, nmem, args);
}

template <class S>
static void adj_group_launch(const GroupMember* mem, int nmem, int nblocks, const AdjStage* args,
                             hipStream_t st) {
  k_adj_stage2d_group<S><<<nblocks, S::NT, 0, st>>>(mem, nmem, args);
}

template <class S>
static void fwd_launch(const Geo& g, const Patches* P, const Tiling& T, const FwdStage& a,
                       hipStream_t st) {
  k_fwd_stage2d<S><<<dim3(T.nblk, g.ninst), S::NT, 0, st>>>(g, P, T, a);
}

template <class S>
static void adj_launch(const Geo& g, const Patches* P, const Tiling& T, const AdjStage& a,
                       hipStream_t st) {
  k_adj_stage2d<S><<<dim3(T.nblk, g.ninst), S::NT, 0, st>>>(g, P, T, a);
}

template <class S>
static void dual_launch(const Geo& g, const Patches* P, const Tiling& T, const AdjStage& a,
                        const FwdStage& f, hipStream_t st) {
  k_dual_stage2d<S><<<dim3(2 * T.nblk, g.ninst), S::NT, 0, st>>>(g, P, T, a, f);
}

void launch_dual_stage2d(const Geo& g, const Patches* P, const Tiling& T, const AdjStage& a,
                         const FwdStage& f, hipStream_t st) {
  switch (T.shape) {
    case 0: dual_launch<S32x16>(g, P, T, a, f, st); break;
    case 1: dual_launch<S16x32>(g, P, T, a, f, st); break;
    case 2: dual_launch<S16x16>(g, P, T, a, f, st); break;
    case 3: dual_launch<S24x16>(g, P, T, a, f, st); break;
    case 4: dual_launch<S16x24>(g, P, T, a, f, st); break;
    default: dual_launch<S16x12>(g, P, T, a, f, st); break;
  }
}

void launch_fwd_stage2d(const Geo& g, const Patches* P, const Tiling& T, const FwdStage& a,
                        hipStream_t st) {
  switch (T.shape) {
    case 0: fwd_launch<S32x16>(g, P, T, a, st); break;
    case 1: fwd_launch<S16x32>(g, P, T, a, st); break;
    case 2: fwd_launch<S16x16>(g, P, T, a, st); break;
    case 3: fwd_launch<S24x16>(g, P, T, a, st); break;
    case 4: fwd_launch<S16x24>(g, P, T, a, st); break;
    default: fwd_launch<S16x12>(g, P, T, a, st); break;
  }
}

void launch_adj_stage2d(const Geo& g, const Patches* P, const Tiling& T, const AdjStage& a,
                        hipStream_t st) {
  switch (T.shape) {
    case 0: adj_launch<S32x16>(g, P, T, a, st); break;
    case 1: adj_launch<S16x32>(g, P, T, a, st); break;
    case 2: adj_launch<S16x16>(g, P, T, a, st); break;
    case 3: adj_launch<S24x16>(g, P, T, a, st); break;
    case 4: adj_launch<S16x24>(g, P, T, a, st); break;
    default: adj_launch<S16x12>(g, P, T, a, st); break;
  }
}

int launch_fwd_stage2d_group(int shape, const GroupMember* mem, int nmem, int nblocks,
                             const FwdStage* args, hipStream_t st) {
  if (shape != kGroupShape) return MGD_ERR_UNSUPPORTED;
  fwd_group_launch<S16x16>(mem, nmem, nblocks, args, st);
  return MGD_OK;
}

int launch_adj_stage2d_group(int shape, const GroupMember* mem, int nmem, int nblocks,
                             const AdjStage* args, hipStream_t st) {
  if (shape != kGroupShape) return MGD_ERR_UNSUPPORTED;
  adj_group_launch<S16x16>(mem, nmem, nblocks, args, st);
  return MGD_OK;
}

void launch_stage_reduce(const double* partial, int nslots, int nfill, int npts, double* sums,
                         int nstages, int base, int ninst, hipStream_t st) {
  if (nfill <= 0 || npts <= 0) return;
  k_stage_sums<<<dim3(nfill, ninst), kSumThreads, 0, st>>>(partial, nslots, npts, sums, nstages,
                                                           base);
}

void launch_stage_accumulate(const double* sums, int nstages, const double* w, double* acc,
                             int ninst, int reverse, hipStream_t st) {
  if (nstages <= 0) return;
  k_stage_accumulate<<<ninst, kRedThreads, 0, st>>>(sums, nstages, w, acc, reverse);
}

}  // namespace mgd
