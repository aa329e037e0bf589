// enl_rhs_body.h -- device bodies of the rhs kernels (fortran/rhs_*.m4),
// shared by the single-patch kernels (enl_rhs.hip) and the batched
// hierarchy kernels (enl_batch.hip).  See enl_rhs.hip for the design.
#pragma once
#include <cmath>

#include "enl_device.h"
#include "enl_kernels.h"

#pragma clang fp contract(off)

namespace enl {

// A BX x BY tile of interior cells plus a 3-cell halo, staged in LDS.
template <int BX, int BY>
struct TileShape {
  static constexpr int halo = 3;
  static constexpr int TW = BX + 2 * halo;
  static constexpr int TH = BY + 2 * halo;
  static constexpr int TN = TW * TH;
  static constexpr int threads = BX * BY;
};

// Workgroups of a 1-D grid are dispatched round-robin over the 8 XCDs
// (workgroup b runs on XCD b % 8), each XCD with its own L2.  xcd_tile maps
// the dispatch index b of n workgroups to a tile index such that each XCD
// works through one contiguous range of tiles: neighbouring tiles, whose
// halos overlap, then share an L2.  A bijection on [0, n).
__device__ inline int xcd_tile(int b, int n) {
  const int q = n >> 3, r = n & 7, x = b & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

constexpr int kStrip = 32;
// Tile (tx, ty) of workgroup b on an nbx x nby tile grid.  The linear tile
// order runs through vertical strips kStrip tiles wide, row-major inside
// a strip, and xcd_tile gives each XCD a contiguous range of it.  A tile's
// upper neighbour then follows it kStrip tiles later on the same XCD,
// while the halo rows they share are still in that XCD's L2; in row-major
// order a whole row of tiles (128 at 4096^2) passes between them, more data
// than one XCD's 4 MB L2 keeps.
__device__ inline int2 strip_tile(int b, int nbx, int nby) {
  const int t = xcd_tile(b, nbx * nby);
  const int full = kStrip * nby;
  const int s = t / full, r = t - s * full;
  const int w = min(kStrip, nbx - s * kStrip);
  return make_int2(s * kStrip + r % w, r / w);
}

// LDS of one staged tile of the split kernels: rho, p, T and the quotients u =
// w1/w0, v, s, T_n, in pairs that a flux reads together, so that a point of the
// stencil takes three 16-byte reads at immediate offsets from one address
// (seven separate arrays took six 8-byte reads and, their distance exceeding
// an 8-byte pair's offset range, an address addition for most of them).
template <int BX, int BY>
struct SplitLds {
  static constexpr int TN = TileShape<BX, BY>::TN;
  double2 uv[TN], st[TN], wp[TN];
  double T[TN];
  unsigned nlist, base;  // the tile's WENO cells: count, place in the list
};
// Of the dense kernel: the stored components, p, T, u and v, read along lines.
template <int BX, int BY>
struct DenseLds {
  static constexpr int TN = TileShape<BX, BY>::TN;
  double w[5][TN], p[TN], T[TN], u[TN], v[TN];
};

// The constants of a launch, folded once on the host: every quotient by a
// grid constant becomes a product with a reciprocal (IEEE, so exact for
// power-of-two dx and dy and within half an ulp otherwise), and constants that
// always multiply each other are multiplied here.  One form serves every grid:
// with the quotients formed per cell the split kernel issued 240 more
// instructions on a grid whose dx is no power of two.
__host__ __device__ inline void fill_rhs_constants(RhsArgs& a, int order) {
  const double ix = 1.0 / a.dx, iy = 1.0 / a.dy;
  const double c[3] = {kA1, kA2, kA3};
  for (int m = 0; m < 3; m++) {
    a.drp_x[m] = -c[m] * ix;
    a.drp_y[m] = -c[m] * iy;
  }
  const double unit = order == 5 ? kWenoUnit<5> : kWenoUnit<3>;
  a.weno_x = unit * ix;
  a.weno_y = unit * iy;
  const double ix2 = 1.0 / (a.dx * a.dx), iy2 = 1.0 / (a.dy * a.dy);
  a.vis_x = (a.muB + kC4_3 * a.mu) * ix2;
  a.vis_y = (a.muB + kC4_3 * a.mu) * iy2;
  a.shear_x = a.mu * ix2;
  a.shear_y = a.mu * iy2;
  a.vis_xy = (a.muB + (1 - kC2_3) * a.mu) / (4 * a.dx * a.dy);
  a.grad_x = 1.0 / (2 * a.dx);
  a.grad_y = 1.0 / (2 * a.dy);
  a.cond_x = a.kappa * ix2;
  a.cond_y = a.kappa * iy2;
  a.half_mu = 0.5 * a.mu;
  a.relax = kC078 * a.R;
  a.inv_tau = 1.0 / a.tau_n;
  a.ep_pre = a.ep > 0 ? 5e-5 * a.ep : -1.0;
}

// A staged tile as cell_source reads it.
template <int BX, int BY>
struct SplitTile {
  const SplitLds<BX, BY>& L;
  __device__ double2 uv(int e) const { return L.uv[e]; }
  __device__ double T(int e) const { return L.T[e]; }
  __device__ double w0(int e) const { return L.wp[e].x; }
};
template <int BX, int BY>
struct DenseTile {
  const DenseLds<BX, BY>& L;
  __device__ double2 uv(int e) const { return make_double2(L.u[e], L.v[e]); }
  __device__ double T(int e) const { return L.T[e]; }
  __device__ double w0(int e) const { return L.w[0][e]; }
};
// The centre cell of this thread in the staged tile.
template <int BX, int BY>
__device__ inline int tile_centre() {
  using Sh = TileShape<BX, BY>;
  return threadIdx.y * Sh::TW + threadIdx.x + (Sh::halo * Sh::TW + Sh::halo);
}

// What a cell's rhs becomes (the FUSED parameter of the kernel bodies):
// kRhs stores it; kStage applies the runge_kutta update and update_state and
// stores the new state; kStageBc does that and, when the arguments' bc_fold
// asks for it, also writes the physical boundary ghosts (the single-patch
// stage: the batched kernels' patches fill ghosts by schedules).
constexpr int kRhs = 0, kStage = 1, kStageBc = 2;

// Result of one cell: store rhs (plain), or apply the runge_kutta update
// and update_state and store the new state (fused stage).
// The fused stage's operands of the runge_kutta update at cell (i, j):
// ww (wa) and the stage input w (wb).
__device__ inline void rk_operands(const RhsArgs& a, int i, int j, double wa[5], double wb[5]) {
  const Geom& G = a.geom;
  const long g = (long)(i + G.g0) + (long)(j + G.g1) * G.sy;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    wa[k] = a.ww[a.ww_off + i + j * a.ww_sy + k * a.ww_sk];
    wb[k] = a.w[g + k * G.sk];
  }
}

// The physical boundary fold of the fused stage (a.bc_fold nonzero): the
// ghost cells whose boundary copy comes from interior cell (i, j), as
// bc_kernel fills them (enlightning.C:836-1008):
// every layer of an edge strip is the nearest interior cell, with u negated
// on a reflecting left/right side and v on a reflecting bottom/top side;
// each corner block is the corner cell with both applicable negations.
// put(d, neg_u, neg_v) receives the ghost's offset in the ghosted arrays.
template <class Put>
__device__ inline void bc_fold_ghosts(const RhsArgs& a, int i, int j, Put put) {
  const Geom& G = a.geom;
  const int f = a.bc_fold;
  const bool lo0 = i == 0, hi0 = i == G.nx - 1, lo1 = j == 0, hi1 = j == G.ny - 1;
  if (!(lo0 || hi0 || lo1 || hi1)) return;
  const bool ru_lo = f & 2, ru_hi = f & 4, rv_lo = f & 8, rv_hi = f & 16;
  const long row = (long)(j + G.g1) * G.sy, col = i + G.g0;
  if (lo0)
    for (int l = 0; l < G.g0; l++) put(row + G.g0 - 1 - l, ru_lo, false);
  if (hi0)
    for (int l = 0; l < G.g0; l++) put(row + G.g0 + G.nx + l, ru_hi, false);
  if (lo1)
    for (int l = 0; l < G.g1; l++) put((long)(G.g1 - 1 - l) * G.sy + col, false, rv_lo);
  if (hi1)
    for (int l = 0; l < G.g1; l++) put((long)(G.g1 + G.ny + l) * G.sy + col, false, rv_hi);
  for (int cx = 0; cx < 2; cx++)
    for (int cy = 0; cy < 2; cy++) {
      if (!(cx ? hi0 : lo0) || !(cy ? hi1 : lo1)) continue;
      for (int lj = 0; lj < G.g1; lj++)
        for (int li = 0; li < G.g0; li++) {
          const int gi = cx ? G.g0 + G.nx + li : G.g0 - 1 - li;
          const int gj = cy ? G.g1 + G.ny + lj : G.g1 - 1 - lj;
          put((long)gi + (long)gj * G.sy, cx ? ru_hi : ru_lo, cy ? rv_hi : rv_lo);
        }
    }
}

template <int FUSED>
__device__ __forceinline__ void cell_output(const RhsArgs& a, int i, int j, const double K[5]) {
  const Geom& G = a.geom;
  const long c = (long)i + (long)j * G.nx;
  const long ik = (long)G.nx * G.ny;
  if constexpr (!FUSED) {
#pragma unroll
    for (int k = 0; k < 5; k++) a.KK[c + k * ik] = K[k];
  } else {
    const long g = (long)(i + G.g0) + (long)(j + G.g1) * G.sy;
    // the ten loads before the first store, so that they are in flight
    // together (w_out aliases neither, which the compiler cannot know)
    double wa[5], wb[5], wn[5];
    rk_operands(a, i, j, wa, wb);
#pragma unroll
    for (int k = 0; k < 5; k++) {
      wn[k] = a.alpha_1 * wa[k] + a.alpha_2 * wb[k] + a.bdt * K[k];
      a.w_out[g + k * G.sk] = wn[k];
    }
    double p = 0, T = 0;
    const bool pt = FUSED != kStageBc || a.p_out;  // uniform
    if (pt) {
      eos_p_T(a.eos, a.ylo + a.dy * ((double)(j) + 0.5), wn[0], wn[3], p, T);
      a.p_out[g] = p;
      a.T_out[g] = T;
    }
    if (FUSED == kStageBc && a.bc_fold)
      bc_fold_ghosts(a, i, j, [&](long d, bool neg_u, bool neg_v) {
        a.w_out[d] = wn[0];
        a.w_out[d + G.sk] = neg_u ? -wn[1] : wn[1];
        a.w_out[d + 2 * G.sk] = neg_v ? -wn[2] : wn[2];
        a.w_out[d + 3 * G.sk] = wn[3];
        a.w_out[d + 4 * G.sk] = wn[4];
        if (pt) {
          a.p_out[d] = p;
          a.T_out[d] = T;
        }
      });
  }
}

// Physical source H, rhs_hybrid_high_llf.m4:159-237.  The reference's entropy
// source sums thirteen quotients; two parts of it cancel identically,
//   kappa |grad T|^2 / T^2 (in sigma) against the same term of the heat flux,
//   (rho / T) A_n M_n - (rho / T_n) c_vn M_n = -(rho / T) c_vn M_n
// (A_n = (T / T_n - 1) c_vn), which leaves
//   H_3 = (muB (div u)^2 + mu/2 (...) + kappa lap T - rho c_vn M_n) / T.
// What cancelled is no longer rounded, and of the quotients 1/T and 1/T_n
// stay: both from one reciprocal of their product (rcp_cubic) where that is in
// range, else by IEEE division.
template <int S, class Tile>
__device__ __forceinline__ void cell_source(const Tile& t, int e, double T_n, double H0, const RhsArgs& a, double H[5]) {
  H[0] = H0;
  // every multiply-add is written out: the plain, fused and batched kernels
  // must round alike, whatever the compiler would contract in each
  const double2 cc = t.uv(e), ce = t.uv(e + 1), cw = t.uv(e - 1), cn = t.uv(e + S), cs = t.uv(e - S);
  const double2 ne = t.uv(e + 1 + S), se = t.uv(e + 1 - S), nw = t.uv(e - 1 + S), sw = t.uv(e - 1 - S);
  const double u0 = cc.x, v0 = cc.y, temp = t.T(e), w0 = t.w0(e);
  const double ue = ce.x, uw = cw.x, un = cn.x, us = cs.x;
  const double ve = ce.y, vw = cw.y, vn = cn.y, vs = cs.y;
  const double vxy = (ne.y - se.y) - (nw.y - sw.y);
  const double uxy = (ne.x - se.x) - (nw.x - sw.x);
  // (lo - 2 mid) + hi: exact for neighbouring values within a factor of two
  auto second = [](double lo, double mid, double hi) { return fma(-2.0, mid, lo) + hi; };
  H[1] = fma(a.vis_x, second(uw, u0, ue), fma(a.shear_y, second(us, u0, un), a.vis_xy * vxy));
  H[2] = fma(a.vis_y, second(vs, v0, vn), fma(a.shear_x, second(vw, v0, ve), a.vis_xy * uxy));
  const double ux = a.grad_x * (ue - uw), uy = a.grad_y * (un - us);
  const double vx = a.grad_x * (ve - vw), vy = a.grad_y * (vn - vs);
  const double phi_xx = fma(kC4_3, ux, -(kC2_3 * vy));
  const double phi_yy = fma(kC4_3, vy, -(kC2_3 * ux));
  const double rot = uy + vx, div = ux + vy;
  const double phi = fma(phi_xx, phi_xx, fma(phi_yy, phi_yy, 2 * rot * rot));
  const double heat = fma(a.cond_x, second(t.T(e - 1), temp, t.T(e + 1)), a.cond_y * second(t.T(e - S), temp, t.T(e + S)));
  double rT, rTn;
  const double TTn = temp * T_n;
  if (den_ok(TTn)) {
    const double r = rcp_cubic(TTn);
    rT = r * T_n;
    rTn = r * temp;
  } else {
    rT = 1.0 / temp;
    rTn = 1.0 / T_n;
  }
  const double Mn = (temp - T_n) * a.inv_tau;
  const double q = a.T_star_n * rTn;
  const double c_vn = a.relax * sq(q) * exp(-q);
  H[4] = w0 * Mn;
  H[3] = fma(a.muB * div, div, fma(a.half_mu, phi, fma(-c_vn, H[4], heat))) * rT;
}

// r = (2|t1 t2| + ep) / (t1^2 + t2^2 + ep) < float(0.9999)?  The numerator
// and denominator are formed exactly as in rhs_hybrid_high_llf.m4:246; the
// comparison of their IEEE quotient with the threshold is decided from a
// single-precision estimate (relative error < 3e-7) whenever that estimate
// is more than 1e-6 away from the threshold, else from the exact quotient.
__device__ inline bool ratio_below(double tmp1, double tmp2, double ep) {
  double num = 2 * fabs(tmp1 * tmp2) + ep;
  double den = sq(tmp1) + sq(tmp2) + ep;
  // den >= num up to rounding (t1^2 + t2^2 >= 2|t1 t2|), so these two bounds
  // keep both within a few ulps of [1e-30, 1e30], normal in single precision
  if (num > 1e-30 && den < 1e30) {
    float q = (float)num * __builtin_amdgcn_rcpf((float)den);
    if (q < (float)(kThresh * (1 - 1e-6))) return true;
    if (q > (float)(kThresh * (1 + 1e-6))) return false;
  }
  return num / den < kThresh;
}

// Hybrid density sensor, rhs_hybrid_high_llf.m4:239-256.  1 = WENO.  The
// triples of q = -1, 0, 1 share four density differences per direction:
// d[m] = rho(i-1+m) - rho(i-2+m), the triple of q being (d[q+1], d[q+2]),
// the reference's tmp1, tmp2 (same subtraction, same bits).  When the
// squares of all eight sum below ep_pre = 5e-5 * ep (ep > 0), every ratio
// (2|t1 t2| + ep) / (t1^2 + t2^2 + ep) is at least 1 / (1 + 5e-5), rounding
// included, far above float(0.9999): the cell is DRP and the six ratios
// need not be formed.  Otherwise they decide as in the reference.
template <int S, class Rho>
__device__ __forceinline__ int cell_sensor(Rho r, int e, double ep, double ep_pre, int level) {
  if (level != 0) return 1;
  double dx[4], dy[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    dx[m] = r(e - 1 + m) - r(e - 2 + m);
    dy[m] = r(e + (m - 1) * S) - r(e + (m - 2) * S);
  }
  {
#pragma clang fp contract(fast)
    double s = 0;
#pragma unroll
    for (int m = 0; m < 4; m++) s += dx[m] * dx[m] + dy[m] * dy[m];
    if (s < ep_pre) return 0;
  }
  int tag = 0;
#pragma unroll
  for (int q = -1; q <= 1; q++) {
    if (ratio_below(dx[q + 1], dx[q + 2], ep)) tag = 1;
    if (ratio_below(dy[q + 1], dy[q + 2], ep)) tag = 1;
  }
  return tag;
}

// DRP branch, rhs_hybrid_high_llf.m4:258-268, without the source: out[k] =
// the weighted sums of the fluxes F along x and G along y
// (rhs_hybrid_high_llf.m4:125-156), the weights over -dx and -dy.  Every flux
// is the mass flux rho u times 1, u, v, s or T_n, with the pressure for the
// normal momentum; opposite points have opposite weights, so their fluxes are
// subtracted before they are weighted: 17 operations a pair, and what the two
// points have in common is gone before anything is rounded at its size.
// Weighting the mass flux of each point first takes 16, but its errors were
// 1.6-2.0 times (mass) and 1.2-1.4 times (entropy, T_n) those of the
// reference's order with fused multiply-adds; this form's are 0.83-0.93 of
// them, the momenta's a fiftieth (waves through patches of 8 to 201 cells a
// side, at rest and in a stream).  Two steps at 4096^2: 3.25 and 3.26 ms.  The
// x stencil is finished before the y stencil's loads are issued
// (sched_barrier), which keeps the twelve points' values from being live at
// once.
//
// Points q1 and q0 opposite each other, weight c; N = 1 along x, 2 along y.
template <int N, int BX, int BY>
__device__ __forceinline__ void drp_pair(const SplitLds<BX, BY>& L, int q1, int q0, double c, double out[5]) {
  const double2 uv1 = L.uv[q1], st1 = L.st[q1], wp1 = L.wp[q1];
  const double2 uv0 = L.uv[q0], st0 = L.st[q0], wp0 = L.wp[q0];
  const double n1 = N == 1 ? uv1.x : uv1.y, n0 = N == 1 ? uv0.x : uv0.y;  // normal velocity
  const double t1 = N == 1 ? uv1.y : uv1.x, t0 = N == 1 ? uv0.y : uv0.x;  // transverse
  const double f1 = wp1.x * n1, f0 = wp0.x * n0;
  out[0] = fma(c, f1 - f0, out[0]);
  out[N] = fma(c, fma(-f0, n0, fma(f1, n1, wp1.y - wp0.y)), out[N]);
  out[3 - N] = fma(c, fma(f1, t1, -(f0 * t0)), out[3 - N]);
  out[3] = fma(c, fma(f1, st1.x, -(f0 * st0.x)), out[3]);
  out[4] = fma(c, fma(f1, st1.y, -(f0 * st0.y)), out[4]);
}
template <int S, int BX, int BY>
__device__ __forceinline__ void cell_drp(const SplitLds<BX, BY>& L, int e, const RhsArgs& a, double out[5]) {
#pragma unroll
  for (int m = 3; m >= 1; m--) drp_pair<1>(L, e + m, e - m, a.drp_x[m - 1], out);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int m = 3; m >= 1; m--) drp_pair<2>(L, e + m * S, e - m * S, a.drp_y[m - 1], out);
}

// One thread's share of the staging loads of a tile + halo (stage_load),
// held in registers until stage_store writes them to LDS.
template <int BX, int BY>
struct StageRegs {
  static constexpr int kIt = (TileShape<BX, BY>::TN + TileShape<BX, BY>::threads - 1) / TileShape<BX, BY>::threads;
  double v[kIt][7];  // w_n(5), p, T
  bool in[kIt];
};

// The global loads of the tile + halo at (i0, j0), all issued before any is
// used.  A cell outside the tile or the ghost box reads element 0 (always in
// the arrays) and is marked not to be stored; no interior cell of the patch
// reads it.
// Loads slots [IT0, IT1) of the thread's share (all of them by default).
template <int FUSED, int BX, int BY, int IT0 = 0, int IT1 = StageRegs<BX, BY>::kIt>
__device__ __forceinline__ void stage_load(const RhsArgs& a, int i0, int j0, StageRegs<BX, BY>& R) {
  using Sh = TileShape<BX, BY>;
  const Geom& G = a.geom;
  const int tid = threadIdx.x + threadIdx.y * BX;
  // the whole tile and halo inside the ghost box (every tile of a grid
  // whose sides are multiples of the tile's, with g >= halo): no per-cell
  // bounds test
  const bool inside = i0 - Sh::halo >= -G.g0 && i0 + Sh::TW - Sh::halo <= G.nx + G.g0 &&
                      j0 - Sh::halo >= -G.g1 && j0 + Sh::TH - Sh::halo <= G.ny + G.g1;
#pragma unroll
  for (int it = IT0; it < IT1; it++) {
    const int e = tid + it * Sh::threads;
    const int gi = i0 + (e % Sh::TW) - Sh::halo, gj = j0 + (e / Sh::TW) - Sh::halo;
    R.in[it] = e < Sh::TN && (inside || (gi >= -G.g0 && gi < G.nx + G.g0 && gj >= -G.g1 && gj < G.ny + G.g1));
    const long gidx = R.in[it] ? (long)(gi + G.g0) + (long)(gj + G.g1) * G.sy : 0;
#pragma unroll
    for (int k = 0; k < 5; k++) R.v[it][k] = a.w[gidx + k * G.sk];
    if (FUSED != kStageBc || a.p) {
      R.v[it][5] = a.p[gidx];
      R.v[it][6] = a.T[gidx];
    }
  }
}

// The height of ghosted row j's p and T where they are formed from w: a
// boundary ghost carries the p and T of the interior row it copies.
__device__ inline double eos_height(const RhsArgs& a, int j) {
  const int jc = j < 0 ? 0 : (j < a.geom.ny ? j : a.geom.ny - 1);
  return a.ylo + a.dy * ((double)jc + 0.5);
}

// rho, p, T and the quotients of the loaded cells
// into the LDS tile.
template <int FUSED, int BX, int BY>
__device__ __forceinline__ void stage_store(const RhsArgs& a, int j0, const StageRegs<BX, BY>& R, SplitLds<BX, BY>& L) {
  using Sh = TileShape<BX, BY>;
  const int tid = threadIdx.x + threadIdx.y * BX;
  const auto& v = R.v;
#pragma unroll
  for (int it = 0; it < R.kIt; it++) {
    if (!R.in[it]) continue;
    const int e = tid + it * Sh::threads;
    const double w0 = v[it][0], w1 = v[it][1], w2 = v[it][2], w3 = v[it][3], w4 = v[it][4];
    double p = v[it][5], T = v[it][6];
    if (FUSED == kStageBc && !a.p) {
      // T is read one cell around the tile only
      const int r = e / Sh::TW, c = e % Sh::TW;
      const bool ring = r >= Sh::halo - 1 && r <= BY + Sh::halo && c >= Sh::halo - 1 && c <= BX + Sh::halo;
      eos_p_T(a.eos, eos_height(a, j0 + r - Sh::halo), w0, w3, p, T, ring);
    }
    L.wp[e] = make_double2(w0, p);
    L.T[e] = T;
    // the four quotients through one reciprocal of w0
    const double iw0 = rcp_any(w0);
    L.uv[e] = make_double2(w1 * iw0, w2 * iw0);
    L.st[e] = make_double2(w3 * iw0, w4 * iw0);
  }
}

// Stage rho, p, T and the quotients of the tile +
// halo.  Cells outside the ghosted array are skipped.
template <int FUSED, int BX, int BY>
__device__ __forceinline__ void stage_tile(const RhsArgs& a, int i0, int j0, SplitLds<BX, BY>& L) {
  StageRegs<BX, BY> R;
  stage_load<FUSED>(a, i0, j0, R);
  stage_store<FUSED>(a, j0, R, L);
}

// The per-cell inputs of a split tile that come from global memory besides
// the staged tile: the source H0 and, where a switch was decided elsewhere,
// its decision (2: the sensor decides).  Loaded apart so that a kernel can
// issue them before prefetching its next tile.
struct SplitIn {
  double h0;
  int d;
};
template <int BX, int BY>
__device__ inline SplitIn split_inputs(const RhsArgs& a, int i0, int j0) {
  const Geom& G = a.geom;
  const int i = i0 + threadIdx.x, j = j0 + threadIdx.y;
  SplitIn s = {0.0, 2};
  if (i < G.nx && j < G.ny) {
    s.h0 = a.H0[(long)i + (long)j * a.h0_sy];
    if (a.decide) s.d = (int)a.decide[(long)i + (long)j * G.nx];
  }
  return s;
}

// Split tile: source H and sensor for every cell, DRP cells finished here,
// WENO cells (sensor on level 0; every cell on finer levels, where the
// reference switches the sensor off, and for rhs_weno_*) keep H in their rhs
// slots and are appended to the list as (patch << 32 | cell): one atomic per
// tile (adds to one address pass at ~8 ns each; one per wave held the small
// launches up: driven step at 512^2 500 -> 470 us, regrid pass 2.83 -> 2.65
// ms, the channel at 2048^2 unchanged).  split_compute runs on a staged tile.
template <int V, int FUSED, int BX, int BY>
__device__ __forceinline__ void split_compute(const RhsArgs& a, int i0, int j0, unsigned pid, SplitLds<BX, BY>& L,
                                     const SplitIn& in);
template <int V, int FUSED, int BX, int BY>
__device__ __forceinline__ void split_body(const RhsArgs& a, int i0, int j0, unsigned pid, SplitLds<BX, BY>& L) {
  stage_tile<FUSED>(a, i0, j0, L);
  const SplitIn in = split_inputs<BX, BY>(a, i0, j0);
  if (Scheme<V>::weno && threadIdx.x + threadIdx.y == 0) L.nlist = 0;
  __syncthreads();
  split_compute<V, FUSED, BX, BY>(a, i0, j0, pid, L, in);
}
template <int V, int FUSED, int BX, int BY>
__device__ __forceinline__ void split_compute(const RhsArgs& a, int i0, int j0, unsigned pid, SplitLds<BX, BY>& L,
                                     const SplitIn& in) {
  using Sc = Scheme<V>;
  using Sh = TileShape<BX, BY>;
  const Geom& G = a.geom;
  const int i = i0 + threadIdx.x, j = j0 + threadIdx.y;
  const bool valid = i < G.nx && j < G.ny;
  int tag = 0;
  if (valid) {
    const SplitTile<BX, BY> t{L};
    const int e = tile_centre<BX, BY>();
    const long icell = (long)i + (long)j * G.nx;
    const long ik = (long)G.nx * G.ny;
    if constexpr (Sc::hybrid) {
      tag = in.d == 2 ? cell_sensor<Sh::TW>([&](int q) { return L.wp[q].x; }, e, a.ep, a.ep_pre, a.level) : in.d;
    } else
      tag = Sc::drp ? 0 : 1;
    // Hybrid DRP cells: the stencil part first, so that H is not live
    // across it (the DRP-only variant keeps source then stencil)
    double out[5] = {0, 0, 0, 0, 0};
    double H[5];
    if constexpr (Sc::hybrid) {
      if (tag == 0) cell_drp<Sh::TW>(L, e, a, out);
      __builtin_amdgcn_sched_barrier(0);
      cell_source<Sh::TW>(t, e, L.st[e].y, in.h0, a, H);
    } else {
      cell_source<Sh::TW>(t, e, L.st[e].y, in.h0, a, H);
      if (tag == 0) cell_drp<Sh::TW>(L, e, a, out);
    }
    if (tag == 0) {
#pragma unroll
      for (int k = 0; k < 5; k++) out[k] = out[k] + H[k];
      cell_output<FUSED>(a, i, j, out);
    } else {
#pragma unroll
      for (int k = 0; k < 5; k++) a.KK[icell + k * ik] = H[k];
    }
    if (a.switch_map) a.switch_map[icell] = tag;
  }
  if constexpr (Sc::weno) {
    const unsigned long long mask = __ballot(tag);
    unsigned slot = 0;
    if (mask) {
      const int lane = __lane_id(), leader = __ffsll(mask) - 1;
      if (lane == leader) slot = atomicAdd(&L.nlist, (unsigned)__popcll(mask));
      slot = __shfl(slot, leader);
    }
    __syncthreads();
    if (L.nlist) {
      if (threadIdx.x + threadIdx.y == 0) L.base = atomicAdd(a.count, L.nlist);
      __syncthreads();
      if (tag)
        a.list[L.base + slot + __popcll(mask & __lanemask_lt())] =
            ((unsigned long long)pid << 32) | (unsigned)(i + j * G.nx);
    }
  }
}

// LLF speed of a cell in row j (rhs_hybrid_high_llf.m4:270-284): the largest
// |velocity| + c + c_lr height over the window, along x (dir 0) at the row's
// height, along y at each point's, and never below 0, where the reference's
// maximum starts.  un holds the normal velocity of the points m = -R..R
// (index m + 3).
template <int R>
__device__ inline double llf_speed(const RhsArgs& a, int j, int dir, const double* un) {
  const double c0 = fma(a.c_lr, fma(a.dy, (double)j + 0.5, a.ylo), a.c), c1 = dir == 0 ? 0.0 : a.c_lr * a.dy;
  double s = fabs(un[3]);
#pragma unroll
  for (int m = -R; m <= R; m++) s = fmax(s, fma((double)m, c1, fabs(un[m + 3])));
  return fmax(0.0, s + c0);
}

// One (direction, component) of a listed WENO cell: the x (dir 0) or y (dir
// 1) term of component k's rhs.  The five lanes of one (cell, direction)
// share the window: lane k forms the normal velocity of points k and k + 5
// and the others reach them by wavefront shuffles.
// gbase is the wave lane of the group's component 0; the group's lanes are
// active together.
template <int V, int FUSED>
__device__ __forceinline__ double list_item(const RhsArgs& a, int cell, int dir, int k, int gbase) {
  using Sc = Scheme<V>;
  constexpr int R = Sc::order == 5 ? 3 : 2;
  const Geom& G = a.geom;
  const int i = cell % G.nx, j = cell / G.nx;
  const long g = (long)(i + G.g0) + (long)(j + G.g1) * G.sy;
  const long step = dir == 0 ? 1 : G.sy;
  const long kn = dir == 0 ? G.sk : 2 * G.sk;
  // this lane's points of the window: pi = k and pi = k + 5 (point m = pi - R)
  const bool two = k + 5 <= 2 * R;
  double ua, ub, pa = 0, pb = 0;
  {
    const long ga = g + (long)(k - R) * step;
    const double na = a.w[ga + kn], da = a.w[ga];
    const long gb = g + (long)(two ? k + 5 - R : 0) * step;
    const double nb = a.w[gb + kn], db = a.w[gb];
    ua = na * rcp_any(da);
    ub = nb * rcp_any(db);
    if (FUSED == kStageBc && !a.p) {
      double T = 0;
      eos_p_T(a.eos, eos_height(a, dir == 0 ? j : j + k - R), da, a.w[ga + 3 * G.sk], pa, T, false);
      eos_p_T(a.eos, eos_height(a, dir == 0 || !two ? j : j + k + 5 - R), db, a.w[gb + 3 * G.sk], pb, T, false);
    }
  }
  double un[7];
#pragma unroll
  for (int pi = 0; pi <= 2 * R; pi++) un[pi - R + 3] = __shfl(pi < 5 ? ua : ub, gbase + pi % 5);
  double alpha = a.alpha;
  if constexpr (Sc::llf) alpha = llf_speed<R>(a, j, dir, un);
  // Every flux is the stored component times the normal velocity (rho u q_k =
  // u w_k, rhs_hybrid_high_llf.m4:125-156), plus the pressure for the normal
  // momentum.
  const bool normal = k == 1 + dir;
  double F[7], W[7], pr[7] = {0, 0, 0, 0, 0, 0, 0};
  const double* w = a.w + g + k * G.sk;
#pragma unroll
  for (int m = -R; m <= R; m++) W[m + 3] = w[m * step];
  if (FUSED == kStageBc && !a.p) {
#pragma unroll
    for (int pi = 0; pi <= 2 * R; pi++) {
      const double p = __shfl(pi < 5 ? pa : pb, gbase + pi % 5);
      pr[pi - R + 3] = normal ? p : 0.0;
    }
  } else if (normal) {
    const double* p = a.p + g;
#pragma unroll
    for (int m = -R; m <= R; m++) pr[m + 3] = p[m * step];
  }
#pragma unroll
  for (int m = -R; m <= R; m++) F[m + 3] = fma(W[m + 3], un[m + 3], pr[m + 3]);
  double d = weno_dir<Sc::order>(F, W, alpha);
  if (!__builtin_isfinite(d)) {
    // by the reference's expressions; the stencil is formed again, not kept for this
    long at = g;
    asm volatile("" : "+v"(at) : : "memory");
    auto point = [&](int m, double& f, double& x) {
      const long q = at + m * step;
      const double w0 = a.w[q];
      double p = 0, T;
      if (normal) {
        if (FUSED == kStageBc && !a.p)
          eos_p_T(a.eos, eos_height(a, dir == 0 ? j : j + m), w0, a.w[q + 3 * G.sk], p, T, false);
        else
          p = a.p[q];
      }
      x = a.w[q + k * G.sk];
      f = fma(x, a.w[q + kn] * rcp_any(w0), p);
    };
    d = weno_dir_ref<Sc::order>(point, alpha);
  }
  return d * (dir == 0 ? a.weno_x : a.weno_y);
}

// The WENO list, ten lanes per cell (two directions x five components) so a
// short list still spreads over the machine.  A wave holds six cells (lanes
// 0..59; a cell's ten lanes never straddle two waves, so they can shuffle):
// lane (dir, k) forms its term, lane (0, k) takes the y term of lane (1, k)
// by a shuffle, forms rhs_k = X[k] + Y[k] + H[k] (the reference's order) and
// writes component k the way cell_output does; in the fused form lane (0,
// 0) takes the new rho*s from lane (0, 3) for p and T.  The waves of a
// block work apart (no LDS, no barrier).  Entries are (patch << 32) | (i +
// j*nx); args_of(patch) gives the patch's arguments.  A wave serves its
// lanes patch by patch (consecutive entries come from one tile: usually a
// single pass) so the arguments stay uniform.
constexpr int kListCellsPerWave = 6;
constexpr int kListCellsPerBlock = 4 * kListCellsPerWave;

template <int V, int FUSED, class ArgsOf>
__device__ __forceinline__ void list_block(ArgsOf args_of, const unsigned long long* list, unsigned n, bool fold = false) {
  const int t = threadIdx.x;
  const int lane = t & 63, slot = lane / 10, item0 = lane % 10;
  const int lc = (t >> 6) * kListCellsPerWave + slot;
  for (unsigned c0 = blockIdx.x * kListCellsPerBlock; c0 < n; c0 += gridDim.x * kListCellsPerBlock) {
    // The grid covers most lists in one round: what depends on the lane's
    // component and direction is formed in it, not held in registers across
    // rounds (hidden from loop-invariant code motion: 30 VGPRs and their spills)
    int item = item0;
    asm volatile("" : "+v"(item));
    const int k = item % 5;
    const int gbase = lane - k;  // lane (dir, 0) of this lane's group
    const unsigned q = c0 + lc;
    bool todo = slot < kListCellsPerWave && q < n;
    const unsigned long long e = todo ? list[q] : 0ull;
    const int pid = (int)(e >> 32);
    for (;;) {
      const unsigned long long m = __ballot(todo);
      if (!m) break;
      const int cur = __builtin_amdgcn_readfirstlane(__shfl(pid, __ffsll((long long)m) - 1));
      if (todo && pid == cur) {
        const RhsArgs& a = args_of(cur);
        const int cell = (int)(e & 0xffffffffu);
        const double term = list_item<V, FUSED>(a, cell, item / 5, k, gbase);
        const double y = __shfl(term, item < 5 ? lane + 5 : lane);
        if (item < 5) {
          const Geom& G = a.geom;
          const long ik = (long)G.nx * G.ny;
          const double K = term + y + a.KK[(long)cell + k * ik];
          const int i = cell % G.nx, j = cell / G.nx;
          if constexpr (!FUSED) {
            a.KK[(long)cell + k * ik] = K;
          } else {
            const long g = (long)(i + G.g0) + (long)(j + G.g1) * G.sy;
            const double wa = a.ww[a.ww_off + i + j * a.ww_sy + k * a.ww_sk];
            const double wb = a.w[g + k * G.sk];
            const double wn = a.alpha_1 * wa + a.alpha_2 * wb + a.bdt * K;
            a.w_out[g + k * G.sk] = wn;
            const double wn3 = __shfl(wn, gbase + 3);
            if (k == 0 && (FUSED != kStageBc || a.p_out)) {
              const double xc1 = a.ylo + a.dy * ((double)(j) + 0.5);
              double p, T;
              eos_p_T(a.eos, xc1, wn, wn3, p, T);
              a.p_out[g] = p;
              a.T_out[g] = T;
            }
          }
        }
        todo = false;
      }
    }
  }
  if constexpr (FUSED == kStageBc) {
    // The boundary fold (fold: the arguments' bc_fold is set), as a second
    // pass so that it adds no live registers to the one above: each lane
    // (0, k) revisits its cells and copies the value it stored there
    // (component k; p and T on lane k = 0) into the ghosts.
    const int k = item0 % 5;
    if (fold && item0 < 5 && slot < kListCellsPerWave)
      for (unsigned q = blockIdx.x * kListCellsPerBlock + lc; q < n; q += gridDim.x * kListCellsPerBlock) {
        const unsigned long long e = list[q];
        const RhsArgs& a = args_of((int)(e >> 32));
        const Geom& G = a.geom;
        const int cell = (int)(e & 0xffffffffu);
        const int i = cell % G.nx, j = cell / G.nx;
        if (i != 0 && i != G.nx - 1 && j != 0 && j != G.ny - 1) continue;
        const long g = (long)(i + G.g0) + (long)(j + G.g1) * G.sy;
        double* w = a.w_out + (long)k * G.sk;
        const double v = w[g];
        bc_fold_ghosts(a, i, j, [&](long d, bool neg_u, bool neg_v) {
          w[d] = (k == 1 && neg_u) || (k == 2 && neg_v) ? -v : v;
        });
        if (k == 0 && a.p_out) {
          const double p = a.p_out[g], T = a.T_out[g];
          bc_fold_ghosts(a, i, j, [&](long d, bool, bool) {
            a.p_out[d] = p;
            a.T_out[d] = T;
          });
        }
      }
  }
}

// Dense tile (every cell WENO) on two thread planes: threadIdx.z = 0 forms the source H and
// the x direction of its cell's five components, threadIdx.z = 1 the y
// direction.  Every flux is the stored component times the normal velocity,
// plus the pressure for the normal momentum (rho u q_k = u w_k), so the tile
// holds w_n, p, T, u and v and no other quotient.  A scheduling barrier after
// each component keeps the next one's loads out of its live range (104 VGPRs
// against 127 at 1024^2 all-WENO: 291 against 300 us per step).  Components
// whose WENO products left the finite range are evaluated again by the
// reference's expressions (weno_dir_ref) in a rolled loop behind them.  The x plane's results
// meet the y plane's in LDS (xs: X then H, 10 x BX*BY doubles) and the y
// plane forms each component as (X + Y) + H,
// the reference's order, and writes the cell.  One direction per thread
// needs about half the registers of both, so more waves fit a SIMD.
template <int V, int FUSED, int BX, int BY>
__device__ __forceinline__ void dense2_body(const RhsArgs& a, int i0, int j0, DenseLds<BX, BY>& L, double* xs) {
  using Sh = TileShape<BX, BY>;
  using Sc = Scheme<V>;
  const Geom& G = a.geom;
  constexpr int NT = 2 * Sh::threads;
  constexpr int S = Sh::TW;
  constexpr int R = Sc::order == 5 ? 3 : 2;
  const int tid = threadIdx.x + BX * (threadIdx.y + BY * threadIdx.z);
  {
    // staging by both planes; every load of a thread before its first store
    constexpr int kIt = (Sh::TN + NT - 1) / NT;
    const bool inside = i0 - Sh::halo >= -G.g0 && i0 + Sh::TW - Sh::halo <= G.nx + G.g0 &&
                        j0 - Sh::halo >= -G.g1 && j0 + Sh::TH - Sh::halo <= G.ny + G.g1;
    double v[kIt][7];
    bool in[kIt];
#pragma unroll
    for (int it = 0; it < kIt; it++) {
      const int e = tid + it * NT;
      const int gi = i0 + (e % Sh::TW) - Sh::halo, gj = j0 + (e / Sh::TW) - Sh::halo;
      in[it] = e < Sh::TN && (inside || (gi >= -G.g0 && gi < G.nx + G.g0 && gj >= -G.g1 && gj < G.ny + G.g1));
      const long gidx = in[it] ? (long)(gi + G.g0) + (long)(gj + G.g1) * G.sy : 0;
#pragma unroll
      for (int k = 0; k < 5; k++) v[it][k] = a.w[gidx + k * G.sk];
      v[it][5] = a.p[gidx];
      v[it][6] = a.T[gidx];
    }
#pragma unroll
    for (int it = 0; it < kIt; it++) {
      if (!in[it]) continue;
      const int e = tid + it * NT;
      const double w0 = v[it][0];
      L.w[0][e] = w0;
      L.p[e] = v[it][5];
      L.T[e] = v[it][6];
      const double iw0 = rcp_any(w0);
      L.u[e] = v[it][1] * iw0;
      L.v[e] = v[it][2] * iw0;
#pragma unroll
      for (int k = 1; k < 5; k++) L.w[k][e] = v[it][k];
    }
  }
  __syncthreads();
  const int i = i0 + threadIdx.x, j = j0 + threadIdx.y;
  const bool live = i < G.nx && j < G.ny;
  const int c = threadIdx.x + BX * threadIdx.y;
  const int e = tile_centre<BX, BY>();
  const DenseTile<BX, BY> t{L};
  const bool yplane = threadIdx.z != 0;
  double Y[5];
  if (live && !yplane) {
    {
      double H[5];
      const double Tn = L.w[4][e] * rcp_any(L.w[0][e]);
      cell_source<S>(t, e, Tn, a.H0[(long)i + (long)j * a.h0_sy], a, H);
#pragma unroll
      for (int k = 0; k < 5; k++) xs[(5 + k) * Sh::threads + c] = H[k];
    }
    double un[7];
#pragma unroll
    for (int m = -R; m <= R; m++) un[m + 3] = L.u[e + m];
    const double af = Sc::llf ? llf_speed<R>(a, j, 0, un) : a.alpha;
    auto term = [&](int k) {
      double F[7], W[7];
#pragma unroll
      for (int m = -R; m <= R; m++) {
        W[m + 3] = L.w[k][e + m];
        F[m + 3] = fma(W[m + 3], un[m + 3], k == 1 ? L.p[e + m] : 0.0);
      }
      return weno_dir<Sc::order>(F, W, af) * a.weno_x;
    };
    auto again = [&](int k) {
      auto point = [&](int m, double& f, double& w) {
        w = L.w[k][e + m];
        f = fma(w, L.u[e + m], k == 1 ? L.p[e + m] : 0.0);
      };
      return weno_dir_ref<Sc::order>(point, af) * a.weno_x;
    };
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const double x = term(k);
      xs[k * Sh::threads + c] = x;
      bad = bad || !__builtin_isfinite(x);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (bad) {
#pragma unroll 1
      for (int k = 0; k < 5; k++)
        if (!__builtin_isfinite(xs[k * Sh::threads + c])) xs[k * Sh::threads + c] = again(k);
    }
  } else if (live) {
    double un[7];
#pragma unroll
    for (int m = -R; m <= R; m++) un[m + 3] = L.v[e + m * S];
    const double ag = Sc::llf ? llf_speed<R>(a, j, 1, un) : a.alpha;
    auto term = [&](int k) {
      double F[7], W[7];
#pragma unroll
      for (int m = -R; m <= R; m++) {
        W[m + 3] = L.w[k][e + m * S];
        F[m + 3] = fma(W[m + 3], un[m + 3], k == 2 ? L.p[e + m * S] : 0.0);
      }
      return weno_dir<Sc::order>(F, W, ag) * a.weno_y;
    };
    auto again = [&](int k) {
      auto point = [&](int m, double& f, double& w) {
        w = L.w[k][e + m * S];
        f = fma(w, L.v[e + m * S], k == 2 ? L.p[e + m * S] : 0.0);
      };
      return weno_dir_ref<Sc::order>(point, ag) * a.weno_y;
    };
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 5; k++) {
      Y[k] = term(k);
      bad = bad || !__builtin_isfinite(Y[k]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (bad) {
#pragma unroll 1
      for (int k = 0; k < 5; k++) {
        const double y = again(k);
#pragma unroll
        for (int q = 0; q < 5; q++)
          if (q == k && !__builtin_isfinite(Y[q])) Y[q] = y;
      }
    }
  }
  __syncthreads();
  if (!live || !yplane) return;
  double K[5];
#pragma unroll
  for (int k = 0; k < 5; k++) K[k] = (xs[k * Sh::threads + c] + Y[k]) + xs[(5 + k) * Sh::threads + c];
  cell_output<FUSED>(a, i, j, K);
  if (a.switch_map) a.switch_map[(long)i + (long)j * G.nx] = 1;
}

}  // namespace enl
