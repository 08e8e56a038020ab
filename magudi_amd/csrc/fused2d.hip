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

// Tile shape: TX x TY points.  D = 1: one thread per point.  D = 2: two, one group of threads
// for each direction -- half the chain of a thread, for launches that leave the chip idle: the
// first group stages the points and does the x lines and the end of the stage, the second the
// halo and the y lines, whose sums it hands over through LDS.  A thread beyond a partial tile
// loads and stages clamped points and stores nothing.  LDS (doubles): the staged operand
// q[4][EY][EX]; forward, the contravariant fluxes of the tile rows (x) and columns (y); the
// boundary closure rows of an edge tile; the far-field terms; the sums handed over.
template <int TX_, int TY_, int D_>
struct Shape {
  static constexpr int TX = TX_, TY = TY_, D = D_, NP = TX * TY, NT = NP * D;
  static_assert(NP % 64 == 0, "whole waves");
  static constexpr int EX = TX + 2 * HX, EY = TY + 2 * HY;
  // halo points (the corners are never read): x-halo columns, then y-halo rows
  static constexpr int kHalo = 2 * HX * TY + 2 * HY * TX;
  static constexpr int kHaloIters = (kHalo + NP - 1) / NP;
  static constexpr int SQ = NV2 * EY * EX, SFX = NV2 * TY * EX, SFY = NV2 * EY * TX;
  static constexpr int kFar = 2 * 4 * kFarPoints, kSums = D == 2 ? 2 * NV2 * NP : 0;
  // closure rows of both ends: first derivative 8 x 12 and composite 8 x 12 (or dissipation
  // transpose 5 x 7); adjoint derivative 12 x 16 and dissipation 8 x 12
  static constexpr int kTabF = 2 * 96 + 2 * 96, kTabA = 2 * 192 + 2 * 96;
  static constexpr int kFwdLds = SQ + SFX + SFY + kTabF + kFar + kSums;
  static constexpr int kAdjLds = SQ + kTabA + kFar + kSums;
  static constexpr int kDualLds = kFwdLds > kAdjLds ? kFwdLds : kAdjLds;
  // waves per SIMD that the LDS use allows (160 KiB per CU), the register budget: at most 4
  static constexpr int waves(int lds) {
    const int w = (160 * 1024) / (8 * lds) * NT / 64 / 4;
    return w < 1 ? 1 : w > 4 ? 4 : w;
  }
  // the tile splits into blocks of 8 x 8 points, one wave each (thread_point)
  static constexpr bool kQuads = TX % 8 == 0 && TY % 8 == 0;
  // components whose LDS reads go out together, as the register budget allows
  static constexpr int kBatchF = waves(kFwdLds) <= 3 ? 2 : 1, kBatchA = D;
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
  // by = tile / nbx: the product is that or one less
  int by = (int)__umulhi((unsigned)tile, T.inv_nbx);
  if (tile - by * T.nbx >= T.nbx) ++by;
  const int bx = tile - by * T.nbx;
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
  const int e = threadIdx.x % S::NP;
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
  const int e = threadIdx.x % S::NP + it * S::NP;
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

// The staged line through a point: c the point (components CS apart, neighbours STEP), pos its
// place in the tile of `size` points along the line, edge whether the tile is at an end of the
// line, e the point's place there.
struct StagedLine {
  const double* c;
  int pos, size;
  bool edge;
  EdgePlace e;
};

// Skew derivative with closure rows BD x BW (tab) and interior coefficients cf on the line.
template <int STEP, int CS, int NB>
__device__ __forceinline__ void line_derivative(const StagedLine& t, const double* tab,
                                                const double* cf, double* out) {
  if (t.edge && t.e.m < 8) {
    const double* b = t.c + ((t.e.right ? t.size - 12 : 0) - t.pos) * STEP;
    closure_row<NV2, 12>(tab + 12 * t.e.m + (t.e.right ? 96 : 0),
                         [&](int l, int k) { return b[l * CS + k * STEP]; }, out);
    return;
  }
#pragma unroll
  for (int l0 = 0; l0 < NV2; l0 += NB) {
    double p[NB][4], m[NB][4];
#pragma unroll
    for (int l = 0; l < NB; ++l)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        p[l][k] = t.c[(l0 + l) * CS + (k + 1) * STEP];
        m[l][k] = t.c[(l0 + l) * CS - (k + 1) * STEP];
      }
    __builtin_amdgcn_sched_barrier(0);   // one batch of LDS reads, one wait
#pragma unroll
    for (int l = 0; l < NB; ++l) out[l0 + l] = skew_sum(p[l], m[l], cf);
  }
}

// H^-1 times the dissipation of the operand on the line (-arc: marc).
template <int STEP, int CS, int NB>
__device__ __forceinline__ void line_dissipation(const Geo& g, const StagedLine& t, double marc,
                                                 double hw, const double* tab, double* out) {
  if (g.composite) {
    if (t.e.m < 8) {
      const double* b = t.c + ((t.e.right ? t.size - 12 : 0) - t.pos) * STEP;
      closure_row<NV2, 12>(tab + 12 * t.e.m + (t.e.right ? 96 : 0),
                           [&](int l, int k) { return b[l * CS + k * STEP]; }, out);
      return;
    }
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      const double* x = t.c + l * CS;
      double s = 0.0;
#pragma unroll
      for (int k = 1; k <= 4; ++k)
        s += g.ops[SLOT_DISS].c[kMaxHW + k] * (x[k * STEP] + x[-k * STEP]);
      out[l] = s + g.ops[SLOT_DISS].c[kMaxHW] * x[0];
    }
    return;
  }
  // the window of nine operands, moved inside the domain at its ends
  const int m = t.e.m;
  const int move = t.edge && m < 4 ? (t.e.right ? m - 4 : 4 - m) : 0;
  const double* b = t.c + (move - 4) * STEP;
  // a point's closure weights: held, or read again for each component where registers are short
  double cw[7];
  if (NB > 1 && t.edge) closure_weights(tab, t.e, cw);
  const double* rows = tab + (t.e.right ? 35 : 0) + 7 * min(t.e.m, 4);
#pragma unroll
  for (int l0 = 0; l0 < NV2; l0 += NB) {
    double w[NB][9];
#pragma unroll
    for (int l = 0; l < NB; ++l)
#pragma unroll
      for (int k = 0; k < 9; ++k) w[l][k] = b[(l0 + l) * CS + k * STEP];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int l = 0; l < NB; ++l) {
      if (!t.edge) {
        out[l0 + l] = two_level(w[l], marc);
      } else {
        const double v = two_level_edge(w[l], marc, t.e, NB > 1 ? cw : rows);
        out[l0 + l] = hw != 1.0 ? v / hw : v;   // 1 away from the first / last boundary rows
      }
    }
  }
}

// D+ of the staged adjoint state (T) and the sum of its 9-point dissipation (w) on the line; v:
// the state at the point.
template <int STEP, int CS, int NB>
__device__ __forceinline__ void line_adjoint(const Geo& g, const StagedLine& t, const double* v,
                                             const double* tab, const double* cf, const double* ds,
                                             double* T, double* w) {
  const bool closure = t.edge && t.e.m < 12;
  // the last (first) of the 16 and 12 staged values that the closure rows of an end reach
  const double* b = t.c + ((t.e.right ? t.size - 1 : 0) - t.pos) * STEP;
  if (closure) {
    const double* b16 = b - (t.e.right ? 15 * STEP : 0);
    closure_row<NV2, 16>(tab + 16 * t.e.m + (t.e.right ? 192 : 0),
                         [&](int l, int k) { return b16[l * CS + k * STEP]; }, T);
  }
  if (t.edge && t.e.m < 8) {
    if (!g.dissipation) return;
    const double* b12 = b - (t.e.right ? 11 * STEP : 0);
    closure_row<NV2, 12>(tab + 384 + 12 * t.e.m + (t.e.right ? 96 : 0),
                         [&](int l, int k) { return b12[l * CS + k * STEP] - v[l]; }, w);
    return;
  }
#pragma unroll
  for (int l0 = 0; l0 < NV2; l0 += NB) {
    double p[NB][4], m[NB][4];
#pragma unroll
    for (int l = 0; l < NB; ++l)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        p[l][k] = t.c[(l0 + l) * CS + (k + 1) * STEP];
        m[l][k] = t.c[(l0 + l) * CS - (k + 1) * STEP];
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int l = 0; l < NB; ++l) {
      if (!closure) T[l0 + l] = skew_sum(p[l], m[l], cf);
      w[l0 + l] = sym9(v[l0 + l], p[l], m[l], ds);
    }
  }
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
// in flight (a chain of loads per patch at the end of the kernel otherwise, on the slowest
// tiles): of two far fields with at most kFarPoints points in the tile, thread 4 k + i of their
// half of the threads forms component i of point k -- sum_c A+[c][i] (q_c - qt_c) forward,
// sum_c A+[i][c] lambda_c adjoint -- into LDS, where the point's thread finds it.
using ConstTileInfo = const __attribute__((address_space(4))) TileInfo;
template <class S, bool ADJ>
__device__ __forceinline__ void far_ahead(const Geo& g, ConstTileInfo* I,
                                          global_ptr<const double> x, double* ff) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (I->far[s].ip < 0) continue;
    const int w = I->far[s].w, h = I->far[s].h, e = (int)threadIdx.x - (S::NT >= 8 * kFarPoints ? 4 * kFarPoints * s : 0);
    if (e < 0 || e >= 4 * w * h) continue;
    const int k = e >> 2, i = e & 3;
    const int dx = w == 1 ? 0 : h == 1 ? k : k % w, dy = w == 1 ? k : h == 1 ? 0 : k / w;
    const long p = (I->far[s].i0 + dx) + (long)g.n[0] * (I->far[s].j0 + dy);
    const long kp = dx + (long)I->far[s].ls * dy;
    const global_ptr<const double> A = glob(I->far[s].aplus) + kp * 16;
    double v = 0.0;
    if (ADJ) {
#pragma unroll
      for (int c = 0; c < NV2; ++c) v += A[i * 4 + c] * x[c * g.N + p];
    } else {
      const global_ptr<const double> qt = glob(I->far[s].target) + kp * 4;
#pragma unroll
      for (int c = 0; c < NV2; ++c) v += A[c * 4 + i] * (x[c * g.N + p] - qt[c]);
    }
    ff[s * 4 * kFarPoints + e] = v;
  }
}

// Far field ip of the tile at grid point (gi, gj): its term f and strength where the point is
// in the patch and the term was formed ahead (1), 0 where the point is not, -1 if not formed.
__device__ __forceinline__ int far_formed(ConstTileInfo* I, int ip, const double* ff, int gi, int gj,
                                          double* f, double* sigma_inv) {
  const int s = ip == I->far[0].ip ? 0 : ip == I->far[1].ip ? 1 : -1;
  if (s < 0) return -1;
  const int kx = gi - I->far[s].i0, ky = gj - I->far[s].j0, w = I->far[s].w;
  if ((unsigned)kx >= (unsigned)w || (unsigned)ky >= (unsigned)I->far[s].h) return 0;
  const double* x = ff + s * 4 * kFarPoints + 4 * (kx + w * ky);
#pragma unroll
  for (int l = 0; l < NV2; ++l) f[l] = x[l];
  *sigma_inv = I->far[s].sigma_inv;
  return 1;
}

// -------------------------------------------------------------------------- forward
// What bounds the stage: on small grids (a few blocks per CU) the chain load - LDS - stencils -
// store of one block, most of all of a corner tile's (101^2, cycles: 1800 to the first load, 3000
// to the barrier, 7300 of stencils against 4400 in an interior tile, 2900 to the end); so there
// is one barrier, every operand is asked for before it, and what a tile holds of patches comes
// with one record.  On batches the 160 bytes per point and stage (0.09 ms for 20 instances of 401 x 401 at the rate
// of a copy) beside 0.07 ms of FP64 issue and 0.06 ms of LDS reads, which overlap in part.
// Plain stores: the rows of a tile end inside cache lines that the neighbour completes, and
// non-temporal stores sent them to memory in pieces (8 x 273^2: 39.3 against 36.9 us).
// Against the stage with the dissipation's intermediates in LDS (three barriers, every patch
// read at the end): 401^2 15.2 -> 12.6 us, 201^2 10.8 -> 8.7, 20 x 401^2 191 -> 162.  One / two
// threads per point: 101^2 9.0 / 8.5 us, 257^2 10.0 / 9.9, 401^2 12.6 / 15.4.
// One forward stage on tile block `blk` of instance `inst` (uniform per work-group).
template <class S>
__device__ __forceinline__ void fwd_stage_body(const Geo& g, const Patches* patches,
                                               const Tiling& T, const FwdStage& a, int blk,
                                               long inst, double* lds) {
  constexpr int TX = S::TX, TY = S::TY, EX = S::EX, EY = S::EY, HS = S::kHaloIters;
  constexpr int NB = S::kBatchF;
  // D = 2: the group of threads, uniform per wave
  const int grp = S::D == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x / S::NP) : 0;
  const bool lead = grp == 0, halo = S::D == 1 || grp == 1;
  double* sq = lds;
  double* sfx = sq + S::SQ;
  double* sfy = sfx + S::SFX;
  double* tab = sfy + S::SFY;
  double* ff = tab + S::kTabF;
  double* sums = ff + S::kFar + threadIdx.x % S::NP;
  const int tile = block_tile(T, blk);
  ConstPatches* P = (ConstPatches*)patches;
  if (tile < 0) return;   // block beyond the tiles of its XCD (uniform per block)
  const TileGeo t = tile_geo(g, T, tile);
  const long NVN = (long)NV2 * g.N;
  const global_ptr<const double> qi = glob(a.qin) + inst * NVN;
  ConstTileInfo* I = (ConstTileInfo*)T.info + tile;
  const unsigned pmask = I->pmask;
  int tx, ty;
  const bool mine = thread_point<S>(t, &tx, &ty);
  const int gi = t.x0 + (mine ? tx : 0), gj = t.y0 + (mine ? ty : 0);
  const long p = gi + (long)g.n[0] * gj;
  // the operand: own point and halo points, then everything else the thread will need, in
  // the order of use (a wait for a load waits for those issued before it)
  double v[NV2], hv[HS][NV2], hm[HS];
#pragma unroll
  for (int l = 0; l < NV2; ++l) v[l] = qi[l * g.N + p];
  if (halo) {
#pragma unroll
    for (int it = 0; it < HS; ++it) {
      const HaloSlot h = halo_slot<S>(g, t, it);
      const long pp = h.gi + (long)g.n[0] * h.gj;
#pragma unroll
      for (int l = 0; l < NV2; ++l) hv[it][l] = qi[l * g.N + pp];
      // metric<2> of the halo's direction
      hm[it] = h.kind == 2 ? glob(g.h[0])[h.gi] : glob(g.h[1])[h.gj];
    }
  }
  const double h0 = glob(g.h[0])[gi], hw0 = glob(g.hw[0])[gi], h1 = glob(g.h[1])[gj], hw1 = glob(g.hw[1])[gj];
  double d1[5];                     // interior coefficients
#pragma unroll
  for (int k = 1; k <= 4; ++k) d1[k] = g.ops[SLOT_FIRST].c[kMaxHW + k];
  far_ahead<S, false>(g, I, qi, ff);
  if (t.bx || t.by) {
    stage_rows<S::NT, 8, 12>(g, SLOT_FIRST, tab);
    if (g.dissipation) {
      if (g.composite) stage_rows<S::NT, 8, 12>(g, SLOT_DISS, tab + 192);
      else stage_rows<S::NT, 5, 7>(g, SLOT_DISS_T, tab + 192);
    }
  }
  // stage the operand and the fluxes
  if (mine && lead) {
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
  if (halo) {
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
  }
  // RK operands, sponge, source and cost-target values, fetched while the stencils run
  const bool sponge = (pmask & T.tables.sponge_mask) != 0;            // uniform per block
  const bool cost = a.jpartial && a.ip_cost >= 0 && ((pmask >> a.ip_cost) & 1u);
  double q0[NV2], b2[NV2], qt[NV2], damp = 0.0, sx0 = 0.0, sy0 = 0.0, pb = 0.0, mo = 0.0;
  bool jin = false;
  int kj = 0;
#pragma unroll
  for (int l = 0; l < NV2; ++l) q0[l] = b2[l] = qt[l] = 0.0;
  if (lead) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      const long o = inst * NVN + l * g.N + p;
      if (a.stage == 2 || a.stage == 3) q0[l] = glob(a.q0)[o];
      if (a.stage >= 2) b2[l] = glob(a.b2)[o];
    }
    if (sponge) {
      damp = glob(T.tables.damp)[p];
#pragma unroll
      for (int l = 0; l < NV2; ++l) qt[l] = glob(T.tables.qtarget)[l * g.N + p];
    }
    if (a.nsrc > 0) {
      sx0 = glob(T.tables.srcx)[gi];
      sy0 = glob(T.tables.srcy)[gj];
    }
    if (cost) {
      ConstPatch& pt = P->p[a.ip_cost];
      jin = mine && in_patch(pt, gi, gj);
      kj = jin ? (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]) : 0;
      pb = glob(pt.aplus)[kj];
      mo = glob(pt.strength)[kj];
    }
  }
  __syncthreads();
  // r = 0 - (D_x F_x + D_y F_y), then the dissipation in x and in y
  double r[NV2];
  const EdgePlace ex = edge_place(g.dir[0], gi), ey = edge_place(g.dir[1], gj);
  const double ax = -fabs(h1), ay = -fabs(h0);          // -arc length along x, y
  const StagedLine fx = {sfx + ty * EX + tx + HX, tx, t.sx, t.bx, ex};
  const StagedLine fy = {sfy + (ty + HY) * TX + tx, ty, t.sy, t.by, ey};
  const StagedLine qx = {sq + (ty + HY) * EX + tx + HX, tx, t.sx, t.bx, ex};
  const StagedLine qy = {qx.c, ty, t.sy, t.by, ey};
  if (S::D == 1) {
    if (!mine) return;
    double d[NV2];
    line_derivative<1, TY * EX, NB>(fx, tab, d1, r);
    line_derivative<TX, EY * TX, NB>(fy, tab, d1, d);
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = 0.0 - (r[l] + d[l]);
    if (g.dissipation) {
      line_dissipation<1, EY * EX, NB>(g, qx, ax, hw0, tab + 192, d);
#pragma unroll
      for (int l = 0; l < NV2; ++l) r[l] = r[l] + g.diss_amount * d[l];
      line_dissipation<EX, EY * EX, NB>(g, qy, ay, hw1, tab + 192, d);
#pragma unroll
      for (int l = 0; l < NV2; ++l) r[l] = r[l] + g.diss_amount * d[l];
    }
  } else {
    double d[NV2], e[NV2];
    if (mine && !lead) {
      line_derivative<TX, EY * TX, NB>(fy, tab, d1, d);
      if (g.dissipation) line_dissipation<EX, EY * EX, NB>(g, qy, ay, hw1, tab + 192, e);
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        sums[l * S::NP] = d[l];
        if (g.dissipation) sums[(NV2 + l) * S::NP] = e[l];
      }
    }
    if (mine && lead) {
      line_derivative<1, TY * EX, NB>(fx, tab, d1, d);
      if (g.dissipation) line_dissipation<1, EY * EX, NB>(g, qx, ax, hw0, tab + 192, e);
    }
    __syncthreads();
    if (!mine || !lead) return;
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      r[l] = 0.0 - (d[l] + sums[l * S::NP]);
      if (g.dissipation) {
        r[l] = r[l] + g.diss_amount * e[l];
        r[l] = r[l] + g.diss_amount * sums[(NV2 + l) * S::NP];
      }
    }
  }
  // point terms, RK4 stage update (substepForwardRK4, src/RK4IntegratorImpl.f90:115-156) and
  // the functional term of the new stage state
  const double dt = a.dt;
  const double jac = 1.0 / (h0 * h1);   // jacobian<2>
#pragma unroll
  for (int l = 0; l < NV2; ++l) r[l] = r[l] * jac;
  // far fields, then sponges, then the other patches, each in the order of the patches
  for (unsigned m = pmask & T.tables.far_mask; m; m &= m - 1) {
    const int ip = __ffs(m) - 1;
    double f[NV2], sigma_inv;
    const int formed = far_formed(I, ip, ff, gi, gj, f, &sigma_inv);
    if (formed == 0) continue;
    if (formed < 0) {
      ConstPatch& pt = P->p[ip];
      if (!in_patch(pt, gi, gj)) continue;
      sigma_inv = pt.sigma_inv;
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
    const double sj = sigma_inv * jac;
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] - sj * f[l];
  }
  if (damp != 0.0) {      // 0 outside the sponges, whatever the target holds there
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] - damp * (v[l] - qt[l]);
  }
  unsigned rest = pmask & ~(T.tables.sponge_mask | T.tables.far_mask);
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
                      (glob(T.tables.srcx)[(long)s * g.n[0] + gi] * glob(T.tables.srcy)[(long)s * g.n[1] + gj]);
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
// last 20 bytes, 141).  Before: 401^2 15.1 -> 11.0 us, 201^2 10.8 -> 7.7, 20 x 401^2 170 -> 139.
// One adjoint stage on tile block `blk` of instance `inst` (uniform per work-group).
template <class S>
__device__ __forceinline__ void adj_stage_body(const Geo& g, const Patches* patches,
                                               const Tiling& T, const AdjStage& a, int blk,
                                               long inst, double* lds) {
  constexpr int EX = S::EX, EY = S::EY, HS = S::kHaloIters, NB = S::kBatchA;
  const int grp = S::D == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x / S::NP) : 0;
  const bool lead = grp == 0, halo = S::D == 1 || grp == 1;
  double* sq = lds;
  double* tab = sq + S::SQ;
  double* ff = tab + S::kTabA;
  double* sums = ff + S::kFar + threadIdx.x % S::NP;
  const int tile = block_tile(T, blk);
  ConstPatches* P = (ConstPatches*)patches;
  if (tile < 0) return;   // block beyond the tiles of its XCD (uniform per block)
  const TileGeo t = tile_geo(g, T, tile);
  const long NVN = (long)NV2 * g.N;
  const global_ptr<const double> li = glob(a.lam) + inst * NVN;
  const global_ptr<const double> qi = glob(a.q) + inst * NVN;
  ConstTileInfo* I = (ConstTileInfo*)T.info + tile;
  const unsigned pmask = I->pmask;
  int tx, ty;
  const bool mine = thread_point<S>(t, &tx, &ty);
  const int gi = t.x0 + (mine ? tx : 0), gj = t.y0 + (mine ? ty : 0);
  const long p = gi + (long)g.n[0] * gj;
  double v[NV2], hv[HS][NV2], q[NV2];
#pragma unroll
  for (int l = 0; l < NV2; ++l) v[l] = li[l * g.N + p];
  if (halo) {
#pragma unroll
    for (int it = 0; it < HS; ++it) {
      const HaloSlot h = halo_slot<S>(g, t, it);
      const long pp = h.gi + (long)g.n[0] * h.gj;
#pragma unroll
      for (int l = 0; l < NV2; ++l) hv[it][l] = li[l * g.N + pp];
    }
  }
  double d1[5], ds[5];              // interior coefficients
#pragma unroll
  for (int k = 0; k <= 4; ++k) {
    d1[k] = g.ops[SLOT_ADJ].c[kMaxHW + k];
    ds[k] = g.ops[SLOT_DISS2].c[kMaxHW + k];
  }
  far_ahead<S, true>(g, I, li, ff);
  if (t.bx || t.by) {
    stage_rows<S::NT, 12, 16>(g, SLOT_ADJ, tab);
    if (g.dissipation) stage_rows<S::NT, 8, 12>(g, SLOT_DISS2, tab + 384);
  }
  if (mine && lead) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) sq[(l * EY + ty + HY) * EX + tx + HX] = v[l];
  }
  if (halo) {
#pragma unroll
    for (int it = 0; it < HS; ++it) {
      const HaloSlot h = halo_slot<S>(g, t, it);
      if (h.kind == 0) continue;
#pragma unroll
      for (int l = 0; l < NV2; ++l) sq[(l * EY + h.ey) * EX + h.ex] = hv[it][l];
    }
  }
  // the forward stage state at the point and the grid values, fetched while the stencils run
  if (lead) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) q[l] = qi[l * g.N + p];
  }
  const double h0 = glob(g.h[0])[gi], hw0 = glob(g.hw[0])[gi], h1 = glob(g.h[1])[gj], hw1 = glob(g.hw[1])[gj];
  __syncthreads();
  // D+ lambda along x and y (T1) and the dissipation (w), from the same staged values
  double T1[2][NV2], w[NV2], l0[NV2], b2[NV2], d[NV2];
  const double sx = diss_scale(g, -g.diss_amount, fabs(h1), hw0);
  const double sy = diss_scale(g, -g.diss_amount, fabs(h0), hw1);
  const double* lc = sq + (ty + HY) * EX + tx + HX;
  const StagedLine lx = {lc, tx, t.sx, t.bx, edge_place(g.dir[0], gi)};
  const StagedLine ly = {lc, ty, t.sy, t.by, edge_place(g.dir[1], gj)};
  if (S::D == 1) {
    if (!mine) return;
    line_adjoint<1, EY * EX, NB>(g, lx, v, tab, d1, ds, T1[0], d);
#pragma unroll
    for (int l = 0; l < NV2; ++l) w[l] = sx * d[l];
    line_adjoint<EX, EY * EX, NB>(g, ly, v, tab, d1, ds, T1[1], d);
#pragma unroll
    for (int l = 0; l < NV2; ++l) w[l] = w[l] + sy * d[l];
  } else {
    if (mine && !lead) {
      line_adjoint<EX, EY * EX, NB>(g, ly, v, tab, d1, ds, T1[1], d);
#pragma unroll
      for (int l = 0; l < NV2; ++l) {
        sums[l * S::NP] = T1[1][l];
        if (g.dissipation) sums[(NV2 + l) * S::NP] = sy * d[l];
      }
    }
    if (mine && lead) line_adjoint<1, EY * EX, NB>(g, lx, v, tab, d1, ds, T1[0], d);
    __syncthreads();
    if (!mine || !lead) return;
#pragma unroll
    for (int l = 0; l < NV2; ++l) {
      T1[1][l] = sums[l * S::NP];
      if (g.dissipation) w[l] = sx * d[l] + sums[(NV2 + l) * S::NP];
    }
  }
  // here, not before: the closure rows need the registers
  const bool sponge = (pmask & T.tables.sponge_mask) != 0;            // uniform per block
  const double damp = sponge ? glob(T.tables.damp)[p] : 0.0;
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
  for (unsigned m = pmask & T.tables.far_mask; m; m &= m - 1) {
    const int ip = __ffs(m) - 1;
    double f[NV2], sigma_inv;
    const int formed = far_formed(I, ip, ff, gi, gj, f, &sigma_inv);
    if (formed == 0) continue;
    if (formed < 0) {
      ConstPatch& pt = P->p[ip];
      if (!in_patch(pt, gi, gj)) continue;
      sigma_inv = pt.sigma_inv;
      const int kp = (gi - pt.lo[0]) + pt.ls[0] * (gj - pt.lo[1]);
      const global_ptr<const double> A = glob(pt.aplus) + (long)kp * 16;
#pragma unroll
      for (int i = 0; i < NV2; ++i) {
        f[i] = 0.0;
#pragma unroll
        for (int c = 0; c < NV2; ++c) f[i] += A[i * 4 + c] * v[c];
      }
    }
    const double sj = sigma_inv * jac;
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] + sj * f[l];
  }
  if (sponge) {
#pragma unroll
    for (int l = 0; l < NV2; ++l) r[l] = r[l] + damp * v[l];
  }
  unsigned rest = pmask & ~(T.tables.sponge_mask | T.tables.far_mask);
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
// Each lane looks at one member (a walk through the members is a chain of loads).
static_assert(kMaxGroup <= 64, "a lane for each member");
__device__ __forceinline__ int group_member(const GroupMember* mem, int nmem, int* blk,
                                            long* inst) {
  const int lane = threadIdx.x & 63;
  const bool before = lane < nmem && mem[min(lane, nmem - 1)].block0 <= (int)blockIdx.x;
  const int m = __builtin_amdgcn_readfirstlane(__popcll(__ballot(before)) - 1);
  int lb = (int)blockIdx.x - mem[m].block0;
  const int nblk = mem[m].T.nblk;
  *inst = 0;
  if (lb >= nblk) {
    *inst = lb / nblk;
    lb %= nblk;
  }
  *blk = lb;
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
using S32x16 = Shape<32, 16, 1>;
using S16x32 = Shape<16, 32, 1>;
using S16x16 = Shape<16, 16, 1>;
using S24x16 = Shape<24, 16, 1>;
using S16x16d2 = Shape<16, 16, 2>;
using S16x12 = Shape<16, 12, 1>;

static const int kShapeDims[kNumTileShapes][2] = {{32, 16}, {16, 32}, {16, 16}, {24, 16},
                                                  {16, 16}, {16, 12}};

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
  TileInfo none{};
  none.far[0].ip = none.far[1].ip = -1;
  out->info.assign((size_t)out->nbx * out->nby, none);
  for (int by = 0; by < out->nby; ++by)
    for (int bx = 0; bx < out->nbx; ++bx) {
      const int xa = out->org[bx], xb = xa + out->size[bx] - 1;
      const int ya = out->org[out->nbx + by], yb = ya + out->size[out->nbx + by] - 1;
      TileInfo& info = out->info[(size_t)by * out->nbx + bx];
      int nfar = 0;
      for (int ip = 0; ip < hp.count; ++ip) {
        const DPatch& pt = hp.p[ip];
        if (xb < pt.lo[0] || xa > pt.hi[0] || yb < pt.lo[1] || ya > pt.hi[1]) continue;
        info.pmask |= 1u << ip;
        if (pt.type != MGD_PATCH_FAR_FIELD || nfar == 2) continue;
        const int i0 = std::max(pt.lo[0], xa), j0 = std::max(pt.lo[1], ya);
        const int w = std::min(pt.hi[0], xb) - i0 + 1, h = std::min(pt.hi[1], yb) - j0 + 1;
        if (w * h > kFarPoints) continue;
        const long k = (i0 - pt.lo[0]) + (long)pt.ls[0] * (j0 - pt.lo[1]);
        info.far[nfar++] = {ip, i0, j0, w, h, pt.ls[0], pt.sigma_inv, pt.aplus + 16 * k,
                            pt.aplus + 16L * pt.np + 4 * k};
      }
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
    case 4: dual_launch<S16x16d2>(g, P, T, a, f, st); break;
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
    case 4: fwd_launch<S16x16d2>(g, P, T, a, st); break;
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
    case 4: adj_launch<S16x16d2>(g, P, T, a, st); break;
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
