// bgk_level.h -- one level of the wave-streaming kernels whose node update needs
// its pulled populations only through their moments: moment storage
// (bgk_stream_mom.hip), FP32 populations (bgk_stream32.hip) and the adjoint
// (bgk_adjoint.hip).  A: double, or float for the adjoint of the FP32 step.
//
// A row's populations are formed once, in the lane of their node, and enter the
// pulled sums of the rows below, beside and above it as three numbers per
// moment family (struct Triple), the columns beside it through lane shifts.
#ifndef BGK_LEVEL_H
#define BGK_LEVEL_H

#include "bgk_mom.h"
#include "bgk_wave.h"

// Every multiply-add below is written out: contraction chosen by the compiler
// could differ between instantiations, and a step has to give the same bits
// whichever launch it is part of.
#pragma clang fp contract(off)

namespace bgk {
namespace level {

using namespace mom;
using namespace wave;

// The nine populations of a node from (m0, m, j = m (u, v) and P): m0 = m =
// rho for f; m0 = T - T_crit, m = T for g, whose populations are the
// deviations g_k - w_k T_crit.  With Q = 9/2 (m u u + P), E = m0 - tr Q / 3:
// p_k = w_k (E + c c : Q + 3 c . j).
template <bool HAVE_P, typename A>
__device__ __forceinline__ void populations(A m0, A m, A u, A v, A pxx, A pyy, A pxy, A p[9]) {
  const A jx = m * u, jy = m * v;
  A qxx, qyy, qxy;
  if constexpr (HAVE_P) {
    qxx = A(4.5) * fma(jx, u, pxx);
    qyy = A(4.5) * fma(jy, v, pyy);
    qxy = A(9.0) * fma(jx, v, pxy);
  } else {
    qxx = A(4.5) * (jx * u);
    qyy = A(4.5) * (jy * v);
    qxy = A(9.0) * (jx * v);
  }
  const A s = qxx + qyy;
  const A e = fma(s, A(-1.0 / 3.0), m0);
  const A ax = (e + qxx) * A(1.0 / 9.0), ay = (e + qyy) * A(1.0 / 9.0), d = e + s;
  const A dp = (d + qxy) * A(1.0 / 36.0), dm = (d - qxy) * A(1.0 / 36.0);
  const A jp = jx + jy, jm = jx - jy;
  p[0] = e * A(4.0 / 9.0);
  p[1] = fma(jx, A(1.0 / 3.0), ax);
  p[3] = fma(jx, A(-1.0 / 3.0), ax);
  p[2] = fma(jy, A(1.0 / 3.0), ay);
  p[4] = fma(jy, A(-1.0 / 3.0), ay);
  p[5] = fma(jp, A(1.0 / 12.0), dp);
  p[7] = fma(jp, A(-1.0 / 12.0), dp);
  p[8] = fma(jm, A(1.0 / 12.0), dm);
  p[6] = fma(jm, A(-1.0 / 12.0), dm);
}

// What three neighbouring source nodes of one row give to a node's pulled
// sums: their total, the total of the two diagonals, and the difference
// (eastward - westward) of the diagonals.
template <typename A>
struct TripleT {
  A n, p, d;
};
template <typename A>
__device__ __forceinline__ TripleT<A> triple(A c, A w, A e) {
  const A p = w + e;
  return TripleT<A>{c + p, p, w - e};
}

// The pulled sums of a node from the row below (sf, sg) and its own (cf, cg).
template <typename A>
__device__ __forceinline__ PullSumsT<A> row_sums(const TripleT<A>& sf, const TripleT<A>& cf,
                                                 const TripleT<A>& sg, const TripleT<A>& cg) {
  PullSumsT<A> s;
  s.rho = sf.n + cf.n;
  s.jx = sf.d + cf.d;
  s.jy = sf.n;
  s.fxx = sf.p + cf.p;
  s.fyy = sf.n;
  s.fxy = sf.d;
  s.dT = sg.n + cg.n;
  s.gxx = sg.p + cg.p;
  s.gyy = sg.n;
  s.gxy = sg.d;
  return s;
}

// Registers of one level between two rows.
template <typename A>
struct LevelT {
  // row awaiting its northern neighbours: pulled sums so far, phi sums of
  // its own and the southern row, its centre tap
  PullSumsT<A> s;
  A t1, t2, pc;
  // the southern share of the row after it
  TripleT<A> sf, sg;
  A n1, n2;
};
using Level = LevelT<double>;

struct Updated {
  double rho, dT, u, v, pfxx, pfyy, pfxy, pgxx, pgyy, pgxy, phi;  // stored
  double dT2, u2, v2;                                              // before the forces
};

// momentsPre .. collision of one node (see core_from_sums in bgk_mom.h for
// the citations), on explicit fused multiply-adds; st, st2: sums of the nine
// phi_prec taps and of their squares, pc the centre tap.
struct StepC {
  double crit_shift, two_over_tw, half_dt_st, gb, t_ref, inv_omega_f, omf1, omega_g, alpha3,
      k_ratio;
};

template <typename R, bool EQF>
__device__ __forceinline__ Updated update(const StepC& c, const PullSums& S, double st, double st2,
                                          double pc) {
  Updated o;
  o.rho = S.rho;
  o.dT2 = S.dT;
  const double irho = rcp_nr(S.rho);
  o.u2 = S.jx * irho;
  o.v2 = S.jy * irho;
  // sum_m ((1 +/- t_m)/2)^2 = (9 +/- 2 sum t + sum t^2) / 4
  const double h = 9.0 + st2;
  const double kp = 0.25 * fma(2.0, st, h), km = 0.25 * fma(-2.0, st, h);
  const bool react = !((kp == 0.0 || pc == 1.0) && (km == 0.0 || pc == -1.0));
  double rm = 0.5;
  if (react) rm = 1.0 / (1.0 + exp((o.dT2 + c.crit_shift) * c.two_over_tw));
  const double rp = 1.0 - rm;
  const double kpr = kp * 0.0625 * rp, kmr = km * 0.0625 * rm;
  o.phi = pc + fma(kpr, 1.0 - pc, -(kmr * (1.0 + pc)));
  o.dT = fma(-c.half_dt_st, o.phi - pc, o.dT2);
  const double T = kTcrit + o.dT;
  const double a = 0.5 - 0.5 * o.phi;
  const double fy = fma(S.rho * c.gb, (T - c.t_ref) * fma(0.5, o.phi, 1.0), -(o.v2 * a));
  const double sc = irho * c.inv_omega_f;
  o.u = fma(-(o.u2 * a), sc, o.u2);
  o.v = fma(fy, sc, o.v2);
  double omg1;
  if (c.k_ratio == 1.0) {
    omg1 = 1.0 - c.omega_g;
  } else {
    const double fl = fma(0.5, o.phi, 0.5);
    omg1 = 1.0 - rcp_nr(fma(c.alpha3, fma(c.k_ratio, 1.0 - fl, fl), 0.5));
  }
  const double Tu = T * o.u, Tv = T * o.v;
  const double g0 = fma(o.dT2, -kCs2, S.gxx), g1 = fma(o.dT2, -kCs2, S.gyy);
  o.pgxx = (double)(R)(omg1 * fma(-Tu, o.u, g0));
  o.pgyy = (double)(R)(omg1 * fma(-Tv, o.v, g1));
  o.pgxy = (double)(R)(omg1 * fma(-Tu, o.v, S.gxy));
  if constexpr (EQF) {
    o.pfxx = o.pfyy = o.pfxy = 0.0;
  } else {
    const double ru = S.rho * o.u, rv = S.rho * o.v;
    const double f0 = fma(S.rho, -kCs2, S.fxx), f1 = fma(S.rho, -kCs2, S.fyy);
    o.pfxx = (double)(R)(c.omf1 * fma(-ru, o.u, f0));
    o.pfyy = (double)(R)(c.omf1 * fma(-rv, o.v, f1));
    o.pfxy = (double)(R)(c.omf1 * fma(-ru, o.v, S.fxy));
  }
  o.u = (double)(R)o.u;
  o.v = (double)(R)o.v;
  return o;
}

// Feed row j (1..Ny, or Ny+1: nothing more comes) of one level: nd holds the
// row's nodes, one per lane.  Gives the completed pulled sums and tap sums of
// row j - 1.  i: this lane's column; has_w / has_e: the wave holds column 1
// / Nx (uniform).
//
// BC_f type 4 and BC_g (STEP_7/BC_f.f90:62-68,101-107,125-136,181-192;
// BC_g.f90:9-64): the lanes of the ghost columns 0 and Nx+1 carry rho = 0
// (their f vanish) and the wall's temperature and velocity (their g are the
// thermal ghosts); bounce-back adds a node's own opposite populations; rows 0
// and Ny+1 of g and phi are rows 1 and Ny.
template <bool EDGE, typename A>
__device__ __forceinline__ void feed(LevelT<A>& L, const A f[9], const A g[9], A phi, int j, int ny,
                                     int i, int nx, bool has_w, bool has_e, A frozen6, A frozen7,
                                     PullSumsT<A>* S, A* st, A* st2, A* pc) {
  *S = L.s;
  *st = L.t1;
  *st2 = L.t2;
  *pc = L.pc;
  if (EDGE && j > ny) return;
  // row sums of the phi taps
  const A pw = from_west(phi), pe = from_east(phi);
  const A r1 = (pw + pe) + phi;
  const A r2 = fma(phi, phi, fma(pw, pw, pe * pe));
  // northern sources of row j - 1
  const TripleT<A> nf = triple(f[4], from_west(f[8]), from_east(f[7]));
  const TripleT<A> ng = triple(g[4], from_west(g[8]), from_east(g[7]));
  S->rho += nf.n;
  S->jx += nf.d;
  S->jy -= nf.n;
  S->fxx += nf.p;
  S->fyy += nf.n;
  S->fxy -= nf.d;
  S->dT += ng.n;
  S->gxx += ng.p;
  S->gyy += ng.n;
  S->gxy -= ng.d;
  *st += r1;
  *st2 += r2;
  // southern sources of row j + 1
  const TripleT<A> sf = triple(f[2], from_west(f[5]), from_east(f[6]));
  const TripleT<A> sg = triple(g[2], from_west(g[5]), from_east(g[6]));
  if (EDGE && j == 1) {  // row 0: bounce-back, copied g and phi
    const A f6 = i == nx ? frozen6 : f[8];
    L.sf = triple(f[4], f[7], f6);
    L.sg = sg;
    L.n1 = r1;
    L.n2 = r2;
  }
  // row j: southern share, then its own row's sources
  {
    const TripleT<A> cf = triple(f[0], from_west(f[1]), from_east(f[3]));
    const TripleT<A> cg = triple(g[0], from_west(g[1]), from_east(g[3]));
    L.s = row_sums(L.sf, cf, L.sg, cg);
    L.t1 = L.n1 + r1;
    L.t2 = L.n2 + r2;
    L.pc = phi;
  }
  if (EDGE) {
    if (j == ny) {  // row Ny+1: bounce-back, copied g and phi
      const TripleT<A> v = triple(f[2], f[6], i == nx ? frozen7 : f[5]);
      L.s.rho += v.n;
      L.s.jx += v.d;
      L.s.jy -= v.n;
      L.s.fxx += v.p;
      L.s.fyy += v.n;
      L.s.fxy -= v.d;
      L.s.dT += ng.n;
      L.s.gxx += ng.p;
      L.s.gyy += ng.n;
      L.s.gxy -= ng.d;
      L.t1 += r1;
      L.t2 += r2;
    }
    if (has_w) {  // column 1: directions 1, 5, 8 bounce back
      const bool on = i == 1;
      const A a = on ? f[3] : A(0);
      const A b = on && j != 1 ? f[7] : A(0);
      const A d = on && j != ny ? f[6] : A(0);
      L.s.rho += a + b + d;
      L.s.jx += a + b + d;
      L.s.jy += b - d;
      L.s.fxx += a + b + d;
      L.s.fyy += b + d;
      L.s.fxy += b - d;
    }
    if (has_e) {  // column Nx: directions 3, 6, 7 bounce back
      const bool on = i == nx;
      const A a = on ? f[1] : A(0);
      const A b = on && j != 1 ? f[8] : A(0);
      const A d = on && j != ny ? f[5] : A(0);
      L.s.rho += a + b + d;
      L.s.jx -= a + b + d;
      L.s.jy += b - d;
      L.s.fxx += a + b + d;
      L.s.fyy += b + d;
      L.s.fxy += d - b;
    }
  }
  L.sf = sf;
  L.sg = sg;
  L.n1 = r1;
  L.n2 = r2;
}

// Moments of a node as the rebuild of its populations takes them.
struct NodeD {
  double rho, th, u, v, pfxx, pfyy, pfxy, pgxx, pgyy, pgxy, phi;
};

// `feed` away from the walls, where the neighbours' populations and phi come from
// elsewhere than the lanes beside: w, c, e of the columns i - 1, i, i + 1.  The same
// operations, so the same bits.
struct Pops {
  double f[9], g[9];
};
__device__ __forceinline__ void feed_three(Level& L, const Pops& w, const Pops& c, const Pops& e,
                                           double pw, double p, double pe, PullSums* S, double* st,
                                           double* st2, double* pc) {
  const TripleT<double> nf = triple(c.f[4], w.f[8], e.f[7]), ng = triple(c.g[4], w.g[8], e.g[7]);
  const TripleT<double> cf = triple(c.f[0], w.f[1], e.f[3]), cg = triple(c.g[0], w.g[1], e.g[3]);
  const double r1 = (pw + pe) + p, r2 = fma(p, p, fma(pw, pw, pe * pe));
  *S = L.s;
  S->rho += nf.n;
  S->jx += nf.d;
  S->jy -= nf.n;
  S->fxx += nf.p;
  S->fyy += nf.n;
  S->fxy -= nf.d;
  S->dT += ng.n;
  S->gxx += ng.p;
  S->gyy += ng.n;
  S->gxy -= ng.d;
  *st = L.t1 + r1;
  *st2 = L.t2 + r2;
  *pc = L.pc;
  L.s = row_sums(L.sf, cf, L.sg, cg);
  L.t1 = L.n1 + r1;
  L.t2 = L.n2 + r2;
  L.pc = p;
  L.sf = triple(c.f[2], w.f[5], e.f[6]);
  L.sg = triple(c.g[2], w.g[5], e.g[6]);
  L.n1 = r1;
  L.n2 = r2;
}

// The sums that `feed` completes for a node (i, j), from its nine sources at once
// and in the same order.  f, g: population k of node (i - cx_k, j - cy_k); rows 0
// and Ny+1 are rows 1 and Ny, the ghost columns carry f = 0 and the wall's g.
// own: the node's own f.  EDGE: the node may be beside a wall.
template <bool EDGE>
__device__ __forceinline__ PullSums pulled_sums(const double f[9], const double g[9],
                                                const double own[9], int i, int j, int nx, int ny,
                                                double frozen6, double frozen7) {
  using Triple = TripleT<double>;
  const bool south = EDGE && j == 1, north = EDGE && j == ny;
  const Triple sf = south ? triple(own[4], own[7], i == nx ? frozen6 : own[8])
                          : triple(f[2], f[5], f[6]);
  const Triple nf = north ? triple(own[2], own[6], i == nx ? frozen7 : own[5])
                          : triple(f[4], f[8], f[7]);
  const Triple ng = triple(g[4], g[8], g[7]);
  PullSums s = row_sums(sf, triple(f[0], f[1], f[3]), triple(g[2], g[5], g[6]),
                        triple(g[0], g[1], g[3]));
  const auto add_north = [&]() __attribute__((always_inline)) {
    s.rho += nf.n;
    s.jx += nf.d;
    s.jy -= nf.n;
    s.fxx += nf.p;
    s.fyy += nf.n;
    s.fxy -= nf.d;
    s.dT += ng.n;
    s.gxx += ng.p;
    s.gyy += ng.n;
    s.gxy -= ng.d;
  };
  if (north) add_north();
  if (EDGE && i == 1) {
    const double a = own[3], b = south ? 0.0 : own[7], d = north ? 0.0 : own[6];
    s.rho += a + b + d;
    s.jx += a + b + d;
    s.jy += b - d;
    s.fxx += a + b + d;
    s.fyy += b + d;
    s.fxy += b - d;
  }
  if (EDGE && i == nx) {
    const double a = own[1], b = south ? 0.0 : own[8], d = north ? 0.0 : own[5];
    s.rho += a + b + d;
    s.jx -= a + b + d;
    s.jy += b - d;
    s.fxx += a + b + d;
    s.fyy += b + d;
    s.fxy += d - b;
  }
  if (!north) add_north();
  return s;
}

// The phi sums that `feed` completes: taps C, E, N, W, S, NE, NW, SW, SE.
__device__ __forceinline__ void tap_sums(const double t[9], double* st, double* st2) {
  const auto sum = [](double w, double c, double e) { return (w + e) + c; };
  const auto square = [](double w, double c, double e) { return fma(c, c, fma(w, w, e * e)); };
  *st = (sum(t[7], t[4], t[8]) + sum(t[3], t[0], t[1])) + sum(t[6], t[2], t[5]);
  *st2 = (square(t[7], t[4], t[8]) + square(t[3], t[0], t[1])) + square(t[6], t[2], t[5]);
}

inline StepC step_constants(const Consts& c) {
  StepC s;
  s.crit_shift = c.crit_shift;
  s.two_over_tw = c.two_over_tw;
  s.half_dt_st = 0.5 * c.dt_st;
  s.gb = c.grav * c.beta;
  s.t_ref = c.t_ref;
  s.inv_omega_f = c.inv_omega_f;
  s.omf1 = 1.0 - c.omega_f;
  s.omega_g = c.omega_g;
  s.alpha3 = 3.0 * c.alpha_l;
  s.k_ratio = c.k_ratio;
  return s;
}

}  // namespace level
}  // namespace bgk

#endif  // BGK_LEVEL_H
