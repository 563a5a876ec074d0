// bgk_adjoint.hip -- discrete adjoint of the moment-storage time step.
//
// Forward model: the moment-storage step (bgk_fused_mom.hip, clean rounding,
// no-slip cavity, extensions t_hot and k_ratio) with FP64 moments, or FP32
// moments (R = float: the adjoint of the step evaluated at the stored
// states, the storage rounding taken as the identity).  Loss: any
// function of the averaged temperature T (STEP_7/moments.f90:11-25) at a
// set of probe nodes after every step; the caller supplies dL/dT(step,
// probe) and receives dL/d(stefan_number, k_ratio, t_hot).
//
// Adjoint state per node (step n): the adjoints of the ten pulled moments
// the node update depends on (PullSums of bgk_mom.h: rho, j, the second
// moments of f; T and the second moments of g) and of the two tap sums and
// the centre tap of the phase field: 13 values, 10 with omega_f = 1, stored
// and computed in the state's precision.  The pull fp_k(x) =
// f_k(x - c_k) is reversed as a gather, so no atomics: node y collects,
// for every direction k, the adjoint of the population k that node y + c_k
// pulled from it, and turns it into the adjoint of its own stored moments
// through the derivative of the population rebuild.  The node update is
// reversed by hand (core_backward below), on values recomputed with the
// same node update the forward kernels run (core_from_sums, bgk_mom.h): the
// adjoint of step n reads only the state before step n.
//
// Checkpointing, binomial (bgk_adj_setup_binomial): the optimal schedule for
// a number of state slots (see rev_cost below).  Levels (bgk_adj_setup,
// bgk_adj_setup_levels): bgk_adj_forward keeps the state every seg_len steps;
// bgk_adj_backward recomputes one segment at a time from its checkpoint,
// keeping every state of the segment, then runs the adjoint kernels over
// the segment backwards.  Memory: (nsteps/seg_len + seg_len + 1) states.
// With two levels the forward run keeps every seg_outer-th state, and each
// outer segment is first recomputed to checkpoints every seg_inner steps:
// nsteps/seg_outer + seg_outer/seg_inner + seg_inner + 1 states.
#include <algorithm>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "bgk_level.h"

// (the adjoint's arithmetic need not be the same in two instantiations)
#pragma clang fp contract(fast)

namespace bgk {
namespace {

using namespace level;

// one stored state: moment planes, phi, east-wall column
struct StatePtrs {
  double2* a;
  void* b;
  void* c;
  double* phi;
  double* te;
};

// Adjoint of one step as stored and computed, in the state's precision: node q
// at [q] of
//   v[0] (rho, jx, jy, dT)  v[1] (gxx, gyy, gxy, kp)  v[2] (km, pc)
// and, unless omega_f = 1, v[2] (km, pc, fxx, fyy)  v[3] fxy.
struct AdjPlanes {
  void* v[4];
};

struct AdjArgs {
  // the state before step n (the inputs of step n); the state after it, whose
  // moments the gather of step n+1's pulls differentiates at, is recomputed
  // from it in the kernel, or is this state itself (the launch for the
  // initial state)
  StatePtrs sprev;
  AdjPlanes next;  // adjoint of step n+1 (read)
  AdjPlanes cur;   // adjoint of step n (written)
  int has_next;    // 0 at the last step: no step n+1
  const int* probe_idx;
  const double* seeds;  // dL/dT at the probes after step n (null: none)
  double* partial;      // 3 per workgroup: dL/dSt, dL/dk_ratio, dL/dt_hot (accumulated)
  Consts c;
  ConstsF cf;    // FP32 copies for the FP32 kernel
  double gd[9];  // d (thermal ghost of direction k) / dT
  int nx, ny;
  int64_t pitch;
  int interf;
  WaveGrid g;
};

// Stored moments of a node (EQF: Pf = 0), or their adjoints, in the
// arithmetic type A.
template <typename A>
struct Mom {
  A rho, th, u, v, pf[3], pg[3];
};

// The moments a forward step stores for a node, widened back to A: rho and T -
// T_crit as computed, u, v and the scaled non-equilibrium moments rounded to
// the storage type R.
template <typename R, bool EQF, typename A, typename C>
__device__ __forceinline__ Mom<A> stored_mom(const C& c, const CoreT<A>& o) {
  Mom<A> m;
  m.rho = o.rho;
  m.th = o.dT;
  m.u = (A)(R)o.u;
  m.v = (A)(R)o.v;
  const A omg1 = A(1) - o.omega_g;
  m.pg[0] = (A)(R)(omg1 * o.qgxx);
  m.pg[1] = (A)(R)(omg1 * o.qgyy);
  m.pg[2] = (A)(R)(omg1 * o.qgxy);
  if constexpr (EQF) {
    m.pf[0] = m.pf[1] = m.pf[2] = A(0);
  } else {
    const A omf1 = A(1) - (A)c.omega_f;
    m.pf[0] = (A)(R)(omf1 * o.qfxx);
    m.pf[1] = (A)(R)(omf1 * o.qfyy);
    m.pf[2] = (A)(R)(omf1 * o.qfxy);
  }
  return m;
}

// Weighted moments sum_k w_k c_k^n a_k (n = 0, 1, 2) of a vector over the
// nine directions.
template <typename A>
struct WMom {
  A m0, mx, my, mxx, myy, mxy;
};

// The share of the three directions with c_y = 1 (or -1) in them: c the value
// of the axis direction, e and w those of the diagonals with c_x = 1 and -1.
template <typename A>
__device__ __forceinline__ TripleT<A> weighted(A c, A e, A w) {
  const A p = A(kW[5]) * (e + w);
  return TripleT<A>{A(kW[1]) * c + p, p, A(kW[5]) * (e - w)};
}
template <typename A>
__device__ __forceinline__ void add_north(WMom<A>& m, const TripleT<A>& t) {
  m.m0 += t.n;
  m.mx += t.d;
  m.my += t.n;
  m.mxx += t.p;
  m.myy += t.n;
  m.mxy += t.d;
}
template <typename A>
__device__ __forceinline__ void add_south(WMom<A>& m, const TripleT<A>& t) {
  m.m0 += t.n;
  m.mx += t.d;
  m.my -= t.n;
  m.mxx += t.p;
  m.myy += t.n;
  m.mxy -= t.d;
}
// c_y = 0: s the southern share, a0, e, w the values of directions 0, 1, 3
template <typename A>
__device__ __forceinline__ WMom<A> centre(const TripleT<A>& s, A a0, A e, A w) {
  const A p = A(kW[1]) * (e + w);
  return WMom<A>{A(kW[0]) * a0 + p + s.n, A(kW[1]) * (e - w) + s.d, -s.n, p + s.p, s.n, -s.d};
}

// The adjoints of a step's pulled sums and taps at a node.
template <typename A>
struct Lam {
  A rho, jx, jy, fxx, fyy, fxy, dT, gxx, gyy, gxy, kp, km, pc;
};

// Registers of the gather between two rows: what the row awaiting its northern
// neighbours has so far, and the southern share of the row after it.  te: the
// adjoint of the east wall's temperature (column Nx).
template <typename A>
struct AdjLevel {
  WMom<A> F, G;
  A kp, km, te, pc;
  TripleT<A> sf, sg;
  A skp, skm, ste;
};

// Reverse of step n+1's pulls.  Population k as pulled by node x has the adjoint
// (rho + c j + c c : f)(x), which belongs to node x - c_k: feed row j (1..Ny, or
// Ny+1: nothing more comes) of these, one node per lane; gives row j - 1's
// weighted moments F, G over its nine populations, the sums over the nine
// nodes that read its phi, and tin, row j's adjoint of the west wall's
// temperature.
//
// Boundaries (feed in bgk_level.h): a direction pulled from a ghost was the
// node's own opposite population (not the two frozen corners); rows 0 and
// Ny+1 of g and phi were rows 1 and Ny; the ghosts of columns 0 and Nx+1 are
// thermal equilibria (gd their derivative).  Lanes outside 1..Nx carry zeros.
template <bool EQF, bool EDGE, typename A>
__device__ __forceinline__ void feed_adjoint(AdjLevel<A>& L, const Lam<A>& x, int j, int ny, int i,
                                             int nx, bool has_w, bool has_e, const A gd[9],
                                             AdjLevel<A>* out, A* tin) {
  *out = L;
  *tin = A(0);
  if (EDGE && j > ny) return;
  A fx = x.rho, fy = x.rho, fp = x.rho, fm = x.rho;
  if constexpr (!EQF) {
    fx += x.fxx;
    fy += x.fyy;
    const A d = fx + x.fyy;
    fp = d + x.fxy;
    fm = d - x.fxy;
  }
  const A jp = x.jx + x.jy, jm = x.jx - x.jy;
  const A f1 = fx + x.jx, f3 = fx - x.jx, f2 = fy + x.jy, f4 = fy - x.jy;
  const A f5 = fp + jp, f7 = fp - jp, f8 = fm + jm, f6 = fm - jm;
  const A g1 = x.dT + x.gxx, g2 = x.dT + x.gyy, gs = g1 + x.gyy;
  const A g5 = gs + x.gxy, g6 = gs - x.gxy;  // directions 5 and 7, 6 and 8
  const A rkp = (from_west(x.kp) + from_east(x.kp)) + x.kp;
  const A rkm = (from_west(x.km) + from_east(x.km)) + x.km;
  const A g5w = from_west(g5), g5e = from_east(g5), g6w = from_west(g6), g6e = from_east(g6);
  // row j - 1 pulled from here with directions 4, 7, 8: its 2, 5, 6
  const TripleT<A> nf = weighted(f2, from_east(f5), from_west(f6));
  const TripleT<A> ng = weighted(g2, g5e, g6w);
  add_north(out->F, nf);
  add_north(out->G, ng);
  out->kp += rkp;
  out->km += rkm;
  // and row j + 1
  const TripleT<A> uf = weighted(f4, from_east(f8), from_west(f7));
  const TripleT<A> ug = weighted(g2, g6e, g5w);
  if (EDGE && has_e) out->te += gd[6] * g6;
  if (EDGE && j == 1) {
    L.sf = weighted(f2, i == nx ? A(0) : f6, f5);
    L.sg = TripleT<A>{A(0), A(0), A(0)};
    L.skp = rkp;
    L.skm = rkm;
    L.ste = A(0);
  }
  L.F = centre(L.sf, x.rho, from_east(f1), from_west(f3));
  L.G = centre(L.sg, x.dT, from_east(g1), from_west(g1));
  L.kp = L.skp + rkp;
  L.km = L.skm + rkm;
  L.pc = x.pc;
  if (EDGE) {
    L.te = L.ste + gd[3] * g1;
    if (j == 1) {
      add_north(L.G, ng);
      L.te += gd[6] * g6;
    }
    if (j == ny) {
      add_north(L.F, weighted(f4, i == nx ? A(0) : f7, f8));
      add_south(L.G, ug);
      L.kp += rkp;
      L.km += rkm;
      L.te += gd[7] * g5;
    }
    if (has_w) {  // column 1: directions 1, 5, 8 were its own 3, 7, 6
      const bool on = i == 1;
      const A a = on ? A(kW[1]) * f1 : A(0);
      const A b = on && j != 1 ? A(kW[5]) * f5 : A(0);
      const A d = on && j != ny ? A(kW[5]) * f8 : A(0);
      L.F.m0 += a + b + d;
      L.F.mx -= a + b + d;
      L.F.my += d - b;
      L.F.mxx += a + b + d;
      L.F.myy += b + d;
      L.F.mxy += b - d;
      if (on) *tin = gd[1] * g1 + gd[5] * g5 + gd[8] * g6;
    }
    if (has_e) {  // column Nx: directions 3, 6, 7 were its own 1, 8, 5
      const bool on = i == nx;
      const A a = on ? A(kW[1]) * f3 : A(0);
      const A b = on && j != 1 ? A(kW[5]) * f6 : A(0);
      const A d = on && j != ny ? A(kW[5]) * f7 : A(0);
      L.F.m0 += a + b + d;
      L.F.mx += a + b + d;
      L.F.my += d - b;
      L.F.mxx += a + b + d;
      L.F.myy += b + d;
      L.F.mxy += d - b;
    }
    L.ste = gd[7] * g5;
  }
  L.sf = uf;
  L.sg = ug;
  L.skp = rkp;
  L.skm = rkm;
}

// Accumulate into lm the adjoint of the node's moments from the weighted
// moments F, G of the adjoints of its nine populations f_k and gd_k (the
// transposed rebuild Jacobian).  Population k is w_k rho (1 + p_k) + c_k H_k :
// Pf for f and w_k (dT + T p_k) + c_k H_k : Pg for gd, with p_k = 3 cu + 9/2
// cu^2 - 3/2 |u|^2, cu = c_k . u, c_k = w_k / (2 cs^4) and H_k = c_k c_k - cs^2
// I; its derivatives are polynomials in c_k, so the sums over k reduce to the
// weighted moments.
template <typename A>
__device__ __forceinline__ void rebuild_adjoint(const Mom<A>& m, const WMom<A>& F,
                                                const WMom<A>& G, Mom<A>* lm) {
  const A u = m.u, v = m.v, uu = u * u, vv = v * v, uv2 = A(2) * u * v;
  const A c0 = A(1) - A(1.5) * (uu + vv);
  // sum_k w_k a_k (1 + p_k)
  lm->rho += F.m0 * c0 + A(3) * (u * F.mx + v * F.my) +
             A(4.5) * (uu * F.mxx + uv2 * F.mxy + vv * F.myy);
  lm->th += G.m0 * c0 + A(3) * (u * G.mx + v * G.my) +
            A(4.5) * (uu * G.mxx + uv2 * G.mxy + vv * G.myy);
  // sum_k w_k L_k dp_k/du, L_k = rho lf_k + T lg_k (and dv)
  const A rho = m.rho, tt = A(kTcrit) + m.th;
  const A L0 = rho * F.m0 + tt * G.m0;
  const A Lx = rho * F.mx + tt * G.mx, Ly = rho * F.my + tt * G.my;
  const A Lxx = rho * F.mxx + tt * G.mxx, Lyy = rho * F.myy + tt * G.myy;
  const A Lxy = rho * F.mxy + tt * G.mxy;
  lm->u += A(3) * (Lx - u * L0) + A(9) * (u * Lxx + v * Lxy);
  lm->v += A(3) * (Ly - v * L0) + A(9) * (u * Lxy + v * Lyy);
  // sum_k c_k H_k a_k = (9/2) (Mxx - cs2 M0, Myy - cs2 M0, 2 Mxy)
  lm->pf[0] += A(4.5) * (F.mxx - A(kCs2) * F.m0);
  lm->pf[1] += A(4.5) * (F.myy - A(kCs2) * F.m0);
  lm->pf[2] += A(9) * F.mxy;
  lm->pg[0] += A(4.5) * (G.mxx - A(kCs2) * G.m0);
  lm->pg[1] += A(4.5) * (G.myy - A(kCs2) * G.m0);
  lm->pg[2] += A(9) * G.mxy;
}

// Reverse of core_from_sums (bgk_mom.h) and of the state it stores.  lo: the
// adjoint of the node's stored moments after the step (rho, T - T_crit, u,
// v, Pf, Pg) and of its phi; ldT2 an extra adjoint on the pulled T (the
// averaged T of moments.f90 seeds half of its adjoint here).  Returns the
// adjoints of the pulled sums, of the tap sums and of the centre tap (direct
// terms) in lS; gives the parameter adjoints of the Stefan number and k_ratio
// in g.  EQF: (1 - omega_f) = 0, the second moments of f carry none.
template <bool EQF, typename A, typename C>
__device__ __forceinline__ void core_backward(const C& c, const PullSumsT<A>& S,
                                              const CoreT<A>& o, const Mom<A>& lo, A lphi_o,
                                              A ldT2_in, Lam<A>* lS, A g[2]) {
  A lrho = lo.rho, lu = lo.u, lv = lo.v, lphi = lphi_o;
  A ldT2 = ldT2_in;
  // Pg = (1 - omega_g) Qg, Pf = (1 - omega_f) Qf
  const A omg1 = A(1) - o.omega_g;
  const A lqgxx = omg1 * lo.pg[0], lqgyy = omg1 * lo.pg[1], lqgxy = omg1 * lo.pg[2];
  const A lomg = -(o.qgxx * lo.pg[0] + o.qgyy * lo.pg[1] + o.qgxy * lo.pg[2]);
  // Qg = S_g - cs2 dT2 - T u u
  ldT2 += -A(kCs2) * (lqgxx + lqgyy);
  A lT = -(o.u * o.u * lqgxx + o.v * o.v * lqgyy + o.u * o.v * lqgxy);
  lu += -A(2) * o.T * o.u * lqgxx - o.T * o.v * lqgxy;
  lv += -A(2) * o.T * o.v * lqgyy - o.T * o.u * lqgxy;
  if constexpr (!EQF) {
    // Qf = S_f - cs2 rho - rho u u
    const A omf1 = A(1) - (A)c.omega_f;
    const A lqfxx = omf1 * lo.pf[0], lqfyy = omf1 * lo.pf[1], lqfxy = omf1 * lo.pf[2];
    lrho += -(A(kCs2) + o.u * o.u) * lqfxx - (A(kCs2) + o.v * o.v) * lqfyy - o.u * o.v * lqfxy;
    lu += -A(2) * o.rho * o.u * lqfxx - o.rho * o.v * lqfxy;
    lv += -A(2) * o.rho * o.v * lqfyy - o.rho * o.u * lqfxy;
    lS->fxx = lqfxx;
    lS->fyy = lqfyy;
    lS->fxy = lqfxy;
  }
  // omega_g(phi, k_ratio) = 1 / (1/2 + alpha/cs2), alpha = alpha_l (fl +
  // k_ratio (1 - fl)): the k_ratio derivative is taken at k_ratio = 1 too,
  // where the forward uses the constant omega_g (the same value)
  {
    const A fl = A(0.5) * (A(1) + o.phi);
    const A domg_dalpha = -o.omega_g * o.omega_g * A(3);  // 1/cs2
    lphi += lomg * domg_dalpha * (A)c.alpha_l * (A(1) - (A)c.k_ratio) * A(0.5);
    g[1] = lomg * domg_dalpha * (A)c.alpha_l * (A(1) - fl);
  }
  // u = u2 + fx s, v = v2 + fy s, s = irho / omega_f
  const A s = o.irho * (A)c.inv_omega_f;
  const A fx = -(o.u2 * (A(1) - o.phi) * A(0.5));
  const A gb = (A)c.grav * (A)c.beta;
  const A fy0 = o.rho * gb * (o.T - (A)c.t_ref) * (A(1) + o.phi * A(0.5));
  const A fy = fy0 - o.v2 * (A(1) - o.phi) * A(0.5);
  A lu2 = lu, lv2 = lv;
  const A lfx = s * lu, lfy = s * lv;
  A lirho = (fx * lu + fy * lv) * (A)c.inv_omega_f;
  // fy = fy0 - v2 (1 - phi)/2, fx = -u2 (1 - phi)/2
  lv2 += -(A(1) - o.phi) * A(0.5) * lfy;
  lphi += o.v2 * A(0.5) * lfy;
  lu2 += -(A(1) - o.phi) * A(0.5) * lfx;
  lphi += o.u2 * A(0.5) * lfx;
  // fy0 = rho g beta (T - t_ref) (1 + phi/2)
  lrho += gb * (o.T - (A)c.t_ref) * (A(1) + o.phi * A(0.5)) * lfy;
  lT += o.rho * gb * (A(1) + o.phi * A(0.5)) * lfy;
  lphi += o.rho * gb * (o.T - (A)c.t_ref) * A(0.5) * lfy;
  // stored T - T_crit = dT; T = T_crit + dT; dT = dT2 - dt_st (phi - pc)/2
  const A ldT = lT + lo.th;
  ldT2 += ldT;
  lphi += -(A)c.dt_st * A(0.5) * ldT;
  A lpcv = (A)c.dt_st * A(0.5) * ldT;
  // dt_st = delta_T / St
  g[0] = (-(o.phi - o.pc) * A(0.5) * ldT) * (-(A)c.dt_st * (A)c.inv_stefan);
  // phi = pc + 0.5 kpr (1 - pc) - 0.5 kmr (1 + pc), kpr = kp/8 rp, kmr = km/8 rm
  const A rp = A(1) - o.rm;
  const A kpr = o.kp_sum * A(0.125) * rp, kmr = o.km_sum * A(0.125) * o.rm;
  const A lkpr = A(0.5) * (A(1) - o.pc) * lphi, lkmr = -A(0.5) * (A(1) + o.pc) * lphi;
  lpcv += lphi * (A(1) - A(0.5) * kpr - A(0.5) * kmr);
  lS->kp = rp * A(0.125) * lkpr;
  lS->km = o.rm * A(0.125) * lkmr;
  const A lrm = o.km_sum * A(0.125) * lkmr - o.kp_sum * A(0.125) * lkpr;
  // rm = 1/(1 + exp((dT2 + crit_shift) * 2/T_width))
  ldT2 += -o.rm * rp * (A)c.two_over_tw * lrm;
  lS->pc = lpcv;
  // u2 = jx irho, v2 = jy irho, irho = 1/rho
  lS->jx = o.irho * lu2;
  lS->jy = o.irho * lv2;
  lirho += S.jx * lu2 + S.jy * lv2;
  lrho += -o.irho * o.irho * lirho;
  lS->rho = lrho;
  lS->dT = ldT2;
  lS->gxx = lqgxx;
  lS->gyy = lqgyy;
  lS->gxy = lqgxy;
}

// The constants in the arithmetic type: Consts for FP64, ConstsF for FP32.
template <typename A>
struct ConstsOf;
template <>
struct ConstsOf<double> {
  static __device__ __forceinline__ const Consts& of(const AdjArgs& a) { return a.c; }
};
template <>
struct ConstsOf<float> {
  static __device__ __forceinline__ const ConstsF& of(const AdjArgs& a) { return a.cf; }
};

// The kernel walks as the forward kernels do (bgk_wave.h): a wave owns 62
// columns and goes up a strip of rows, the columns beside a node come by lane
// shifts, the rows below and above it as sums kept in registers: step n's
// pulled sums and taps (feed, bgk_level.h) and the gather of step n+1's
// adjoints (feed_adjoint).  Every node is read from HBM once but for a strip's
// two rows and a wave's two columns of its neighbours.  The adjoints lie in
// planes of four values, so that a row is seven loads and three stores, and the
// next row's loads are issued as soon as this one's values are taken.
//
// Registers decide: FP32 162 (omega_f = 1) and 174, held to two waves per SIMD
// (three: the same with omega_f = 1, 4% slower with 20 bytes spilled without;
// four: twice the time, spilled); FP64 more than 256, so one wave per SIMD (two:
// 46 spilled, twice the time).  Bound by HBM from 2048^2 up; below, by the
// latency of one row after another in a few waves.
// Measured against tiles of 64 x 8 and 64 x 4 nodes with a window of everything
// in LDS (765 VALU instructions per wave, the populations rebuilt for every
// pull), us per launch, before -> now: FP32 moments with omega_f = 1 2048^2 139 ->
// 120, 8192^2 2085 -> 1804 (4.6 TB/s of the 124 bytes per node that a launch
// cannot do without), general 2048^2 193 -> 153; FP64 moments with omega_f = 1
// 512^2 27.6 -> 18.9, 4096^2 1210 -> 775 (4.8 TB/s of 224 bytes), general 512^2
// 30.5 -> 21.9, 4096^2 1380 -> 1031.
constexpr int kAdjCols = kLanes - 2;
template <typename R>
constexpr int adj_waves() {
  return sizeof(R) == 4 ? 2 : 1;
}
// FP64 adjoints are stored through the caches: small lattices find them there
// (gradient at 512^2, 300 steps: 9.4 ms for 9.8; 4096^2, 24 steps: 27.4 for
// 29.3); FP32 ones past them (2048^2, 48 steps: 9.2 ms for 9.3).
template <typename R>
constexpr int adj_store() {
  return sizeof(R) == 4 ? kNonTemporal : kCached;
}
// The initial phi of the ghost columns 0 and Nx+1, which no step changes
// (STEP_7/initialization.f90:15-26: liquid for i <= Nx/40).
constexpr double kPhiWest = 1.0, kPhiEast = -1.0;

template <typename R>
struct V2Of;
template <>
struct V2Of<double> {
  using T = double2;
};
template <>
struct V2Of<float> {
  using T = float2;
};

// A row as loaded: the state before the step and the adjoint of the step after.
template <typename R, bool EQF>
struct AdjRow {
  using V4 = typename Vec<R>::V4;
  using C = typename CType<R, EQF>::T;
  using L2 = typename std::conditional<EQF, typename V2Of<R>::T, V4>::type;
  double2 a;
  V4 b;
  C c;
  double phi;
  V4 l0, l1;
  L2 l2;
  R l3;

  // columns counted from ib
  __device__ __forceinline__ void load_state(const AdjArgs& A, int j, int ib, unsigned ic) {
    const int64_t q = (int64_t)j * A.pitch + ib;
    a = at(A.sprev.a + q, ic * (unsigned)sizeof(double2));
    b = at(static_cast<const V4*>(A.sprev.b) + q, ic * (unsigned)sizeof(V4));
    c = at(static_cast<const C*>(A.sprev.c) + q, ic * (unsigned)sizeof(C));
    phi = at(A.sprev.phi + q, ic * (unsigned)sizeof(double));
  }
  __device__ __forceinline__ void load_lam(const AdjArgs& A, int j, int ib, unsigned ic) {
    const int64_t q = (int64_t)j * A.pitch + ib;
    l0 = at(static_cast<const V4*>(A.next.v[0]) + q, ic * (unsigned)sizeof(V4));
    l1 = at(static_cast<const V4*>(A.next.v[1]) + q, ic * (unsigned)sizeof(V4));
    l2 = at(static_cast<const L2*>(A.next.v[2]) + q, ic * (unsigned)sizeof(L2));
    if constexpr (!EQF) l3 = at(static_cast<const R*>(A.next.v[3]) + q, ic * (unsigned)sizeof(R));
  }
  __device__ __forceinline__ Mom<R> state(R* ph) const {
    Mom<R> m;
    if constexpr (sizeof(R) == 4) {
      m.rho = (R)a.x;
      m.th = (R)a.y;
      *ph = (R)phi;
    } else {
      m.rho = taken(a.x);
      m.th = taken(a.y);
      *ph = taken(phi);
    }
    m.u = taken(b.x);
    m.v = taken(b.y);
    if constexpr (EQF) {
      m.pf[0] = m.pf[1] = m.pf[2] = R(0);
      m.pg[0] = taken(b.z);
      m.pg[1] = taken(b.w);
      m.pg[2] = taken(c);
    } else {
      m.pf[0] = taken(b.z);
      m.pf[1] = taken(b.w);
      m.pf[2] = taken(c.x);
      m.pg[0] = taken(c.y);
      m.pg[1] = taken(c.z);
      m.pg[2] = taken(c.w);
    }
    return m;
  }
  // (zeros where there is no step after, and outside the lattice)
  __device__ __forceinline__ Lam<R> lam(bool live) const {
    Lam<R> x;
    const auto get = [&](R y) __attribute__((always_inline)) { return live ? taken(y) : R(0); };
    x.rho = get(l0.x);
    x.jx = get(l0.y);
    x.jy = get(l0.z);
    x.dT = get(l0.w);
    x.gxx = get(l1.x);
    x.gyy = get(l1.y);
    x.gxy = get(l1.z);
    x.kp = get(l1.w);
    x.km = get(l2.x);
    x.pc = get(l2.y);
    if constexpr (EQF) {
      x.fxx = x.fyy = x.fxy = R(0);
    } else {
      x.fxx = get(l2.z);
      x.fyy = get(l2.w);
      x.fxy = get(l3);
    }
    return x;
  }
};

// Stores of row j at column i of n from ib on (lanes that must not store: kPastStrip).
template <typename R, bool EQF>
__device__ __forceinline__ void store_adjoint(const AdjArgs& A, int j, int ib, int n, int i,
                                              const Lam<R>& x) {
  using Row = AdjRow<R, EQF>;
  const int64_t q = (int64_t)j * A.pitch + ib;
  buffer_put<adj_store<R>()>(strip_buffer(static_cast<typename Row::V4*>(A.cur.v[0]) + q, n), i,
             make4<R>(x.rho, x.jx, x.jy, x.dT));
  buffer_put<adj_store<R>()>(strip_buffer(static_cast<typename Row::V4*>(A.cur.v[1]) + q, n), i,
             make4<R>(x.gxx, x.gyy, x.gxy, x.kp));
  const auto b2 = strip_buffer(static_cast<typename Row::L2*>(A.cur.v[2]) + q, n);
  if constexpr (EQF) {
    typename Row::L2 y;
    y.x = x.km;
    y.y = x.pc;
    buffer_put<adj_store<R>()>(b2, i, y);
  } else {
    buffer_put<adj_store<R>()>(b2, i, make4<R>(x.km, x.pc, x.fxx, x.fyy));
    buffer_put<adj_store<R>()>(strip_buffer(static_cast<R*>(A.cur.v[3]) + q, n), i, x.fxy);
  }
}

// One wave's strip, rows j0..j1.  EDGE: the wave or the strip touches a wall.
// INIT: the share of the initial state, sprev itself (nothing is stored).  g: this
// lane's parameter adjoints, summed in FP64.  WIDE: a row is more than a 32-bit byte
// offset reaches, so columns are counted from the wave's first one (at every width
// 2% slower with FP64 moments).
template <typename R, bool EQF, bool EDGE, bool INIT, bool WIDE>
__device__ __forceinline__ void adjoint_strip(const AdjArgs& A, int j0, int j1, int i0, int i,
                                              bool has_w, bool has_e, double g[3]) {
  const auto& c = ConstsOf<R>::of(A);
  const int nx = A.nx, ny = A.ny, lane = (int)threadIdx.x;
  const int ib = WIDE ? i0 - 1 : 0;
  const unsigned ic = (unsigned)((i < 0 ? 0 : (i > nx + 1 ? nx + 1 : i)) - ib);  // column loaded
  const bool ghost = EDGE && (i == 0 || i == nx + 1);
  const bool own = lane >= 1 && lane < kLanes - 1 && i <= nx;  // columns this wave stores
  const bool live = A.has_next && (!EDGE || (i >= 1 && i <= nx));
  R gd[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) gd[k] = (R)A.gd[k];

  // rows of the strip that hold a probe (column 0 of the probe index plane is
  // >= 0 there; at most kMaxRows rows)
  uint64_t probes = 0;
  if (!INIT && A.seeds)
    probes = __ballot(j0 + lane <= j1 &&
                      A.probe_idx[(int64_t)min(j0 + lane, j1) * A.pitch] >= 0);

  LevelT<R> S = LevelT<R>{};
  AdjLevel<R> L = AdjLevel<R>{};
  R u_was = R(0), v_was = R(0);  // INIT: the completed row's velocity
  const int ra = EDGE ? max(1, j0 - 1) : j0 - 1, rb = j1 + 1;
  AdjRow<R, EQF> row;
  row.load_lam(A, ra, ib, ic);
  row.load_state(A, ra, ib, ic);
  const scalar_ptr te_in = as_scalar(A.sprev.te);
  double te_row = EDGE ? te_in[ra] : 0.0;
  __builtin_amdgcn_s_waitcnt(kWaitLoads);
  auto feed_row = [&](int r, auto feed_only) __attribute__((always_inline)) {
    const Lam<R> x = row.lam(live);
    __builtin_amdgcn_sched_barrier(0);
    row.load_lam(A, min(r + 1, ny), ib, ic);
    const int jc = r - 1;  // row completed
    const bool on = own && jc >= j0 && jc <= j1;
    // ---- step n+1's pulls reversed
    AdjLevel<R> G;
    R tin;
    feed_adjoint<EQF, EDGE>(L, x, r, ny, i, nx, has_w, has_e, gd, &G, &tin);
    if (EDGE && r >= j0 && r <= j1 && own) g[2] += (double)tin;
    __builtin_amdgcn_sched_barrier(0);
    R phi;
    Mom<R> m = row.state(&phi);
    __builtin_amdgcn_sched_barrier(0);
    row.load_state(A, min(r + 1, ny), ib, ic);
    Mom<R> lm = {};
    if constexpr (INIT) {
      Mom<R> was = {};
      was.u = u_was;
      was.v = v_was;
      rebuild_adjoint<R>(was, G.F, G.G, &lm);
      // T = t_hot in the liquid strip (initialization.f90:15-26)
      if (on && i <= A.interf) g[2] += (double)lm.th;
      u_was = m.u;
      v_was = m.v;
      return;
    }
    // ---- step n's pulled sums and taps
    if (EDGE) {
      const double te = A.c.east_cold ? A.c.t_cold : te_row;
      te_row = te_in[min(r + 1, ny)];
      if (ghost) {  // no flow populations, the wall's T and velocity
        m.rho = m.pf[0] = m.pf[1] = m.pf[2] = m.pg[0] = m.pg[1] = m.pg[2] = R(0);
        m.th = (R)((i == 0 ? A.c.tin : te) - kTcrit);
        m.u = (R)A.c.u0;
        m.v = (R)A.c.v0;
        phi = i == 0 ? R(kPhiWest) : R(kPhiEast);
      }
    }
    R f[9], gp[9];
    populations<!EQF>(m.rho, m.rho, m.u, m.v, m.pf[0], m.pf[1], m.pf[2], f);
    populations<true>(m.th, R(kTcrit) + m.th, m.u, m.v, m.pg[0], m.pg[1], m.pg[2], gp);
    PullSumsT<R> P;
    R st, st2, pc;
    feed<EDGE>(S, f, gp, phi, r, ny, i, nx, has_w, has_e, (R)A.c.frozen6, (R)A.c.frozen7, &P, &st,
               &st2, &pc);
    if constexpr (decltype(feed_only)::value) return;
    __builtin_amdgcn_sched_barrier(0);
    const CoreT<R> o = core_from_sums<R>(c, P, st, st2, pc);
    // ---- the adjoint of the state after step n
    rebuild_adjoint<R>(stored_mom<R, EQF, R>(c, o), G.F, G.G, &lm);
    const R lphi = R(0.5) * (R(1) + o.phi) * G.kp - R(0.5) * (R(1) - o.phi) * G.km + G.pc;
    // averaged T = T_crit + (dT + dT2)/2: its adjoint half on the stored dT,
    // half on dT2.  The east ghosts of step n+1 are equilibria at this node's
    // (not with the cold-wall extension: then a constant)
    R lt = EDGE && i == nx && !A.c.east_cold ? G.te : R(0);
    if (jc >= j0 && ((probes >> (jc - j0)) & 1) && on) {
      const int p = A.probe_idx[(int64_t)jc * A.pitch + i];
      if (p >= 0) lt += (R)A.seeds[p];
    }
    lm.th += R(0.5) * lt;
    // ---- reverse of step n at this node
    Lam<R> out;
    R gp2[2];
    core_backward<EQF, R>(c, P, o, lm, lphi, R(0.5) * lt, &out, gp2);
    store_adjoint<R, EQF>(A, min(max(jc, j0), j1), ib, WIDE ? kLanes : (int)A.pitch,
                          on ? i - ib : kPastStrip, out);
    g[0] += on ? (double)gp2[0] : 0.0;
    g[1] += on ? (double)gp2[1] : 0.0;
  };
  // Up to row j0 no row of the strip is complete.  Leaving the node update out
  // there pays with FP64 moments, whose strips are a few rows of latency (ms per
  // gradient of 300 steps, backward pass: 301 x 207 6.24 -> 5.83, 512^2 9.33 -> 9.08);
  // with FP32 moments it gave nothing (2048^2, 48 steps: 8.5 and 8.5).
  int r = ra;
  if (!INIT && sizeof(R) == sizeof(double))
    for (; r <= j0; ++r) feed_row(r, std::true_type{});
  for (; r <= rb; ++r) feed_row(r, std::false_type{});
}

template <typename R, bool EQF, bool INIT, bool WIDE>
__global__ __launch_bounds__(kLanes, (adj_waves<R>())) void k_adjoint(AdjArgs A) {
  int seg, j0, j1;
  bool edge;
  if (!wave_tile(A.g, A.ny, &seg, &j0, &j1, &edge)) return;
  const int i0 = seg * kAdjCols + 1;
  const int i = i0 - 1 + (int)threadIdx.x;
  double g[3] = {0.0, 0.0, 0.0};
  if (edge)
    adjoint_strip<R, EQF, true, INIT, WIDE>(A, j0, j1, i0, i, i0 == 1, i0 + kAdjCols >= A.nx, g);
  else
    adjoint_strip<R, EQF, false, INIT, WIDE>(A, j0, j1, i0, i, false, false, g);
  // parameter adjoints: butterfly over the wave, then this workgroup's own
  // slot (deterministic)
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    for (int m = 32; m > 0; m >>= 1) g[k] += __shfl_xor(g[k], m, 64);
    if (threadIdx.x == 0) A.partial[3 * (int64_t)blockIdx.x + k] += g[k];
  }
}

// Deterministic sum of the per-workgroup slots.
__global__ void k_adj_sum(const double* partial, int n, double* out) {
  __shared__ double red[3][256];
  const int t = threadIdx.x;
  double s[3] = {0.0, 0.0, 0.0};
  for (int b = t; b < n; b += 256)
    for (int c = 0; c < 3; ++c) s[c] += partial[3 * b + c];
  for (int c = 0; c < 3; ++c) red[c][t] = s[c];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w)
      for (int c = 0; c < 3; ++c) red[c][t] += red[c][t + w];
    __syncthreads();
  }
  if (t == 0)
    for (int c = 0; c < 3; ++c) out[c] = red[c][0];
}

// probe index plane: -1 everywhere (k_probe_clear), then p at probe p's
// node and 0 in column 0 of its row (k_probe_set, a second launch on the
// same stream): the forward kernels read the row flag once per row
__global__ void k_probe_clear(int* idx, int64_t n) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) idx[q] = -1;
}

__global__ void k_probe_set(int* idx, const int* pij, int np, int64_t pitch) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < np) {
    idx[(int64_t)pij[2 * p + 1] * pitch + pij[2 * p]] = p;
    idx[(int64_t)pij[2 * p + 1] * pitch] = 0;
  }
}

}  // namespace

// ------------------------------------------------------------------ host

struct AdjCtx {
  int nsteps = 0, np = 0;
  int seg = 0;    // inner segment: every state of one is stored
  int seg1 = 0;   // outer segment (two levels), 0: one level
  int nckpt = 0;  // checkpoints of the forward run (every seg1, or seg, steps)
  int nckpt2 = 0; // checkpoints of one outer segment (two levels)
  int nsnap = 0;  // binomial schedule: snapshot slots (state 0's included); 0: levels
  void* pool = nullptr;
  size_t bytes = 0;
  std::vector<StatePtrs> slot;   // states 1..seg of an inner segment (slot[0] spare)
  std::vector<StatePtrs> ckpt;   // checkpoints of the forward run
  std::vector<StatePtrs> ckpt2;  // checkpoints of the outer segment being reversed
  std::vector<StatePtrs> snap;   // binomial: snapshot slots
  StatePtrs work[2] = {};        // binomial: states being advanced
  std::vector<int> chain;        // binomial: steps stored by the forward run (state
                                 // chain[k] in snap[k + 1], state 0 in snap[0])
  AdjPlanes lam[2];
  int* probe_idx = nullptr;
  int* probe_ij = nullptr;
  double* probe_T = nullptr;  // nsteps x np
  double* seeds = nullptr;    // nsteps x np
  double* partial = nullptr;
  double* out3 = nullptr;
  int nblk = 0;
  int64_t recomputed = 0;     // forward steps the last backward pass ran
  bool forward_done = false;
};

namespace {

// ---- binomial checkpointing (Griewank's "revolve" schedule, written from
// the published method: A. Griewank, A. Walther, ACM TOMS 26 (2000) 19-45).
// Reversing l steps from a held state with s free snapshot slots costs, at
// best, T(l, s) = r l - C(S + r, S + 1) forward steps, S = s + 1 and r the
// least integer with C(S + r, S) >= l (T(l, 0) = l (l - 1)/2: every state
// advanced to from the held one).  An optimal schedule advances to a split
// m, stores that state, reverses [m, l) with s - 1 slots, frees the slot and
// reverses [0, m) with s slots; m minimises m + T(l - m, s - 1) + T(m, s).

int64_t rev_cost(int64_t l, int64_t s) {
  if (l <= 1) return 0;
  const int64_t S = s + 1;
  int64_t r = 0, beta = 1;  // beta = C(S + r, S)
  while (beta < l) {
    ++r;
    beta = beta * (S + r) / r;
  }
  return r * l - beta * r / (S + 1);  // C(S + r, S + 1) = C(S + r, S) r / (S + 1)
}

int64_t rev_split(int64_t l, int64_t s) {
  int64_t best = 1, cost = -1;
  for (int64_t m = 1; m < l; ++m) {
    const int64_t c = m + rev_cost(l - m, s - 1) + rev_cost(m, s);
    if (cost < 0 || c < cost) {
      cost = c;
      best = m;
    }
  }
  return best;
}

// Steps the forward run stores (the splits of the schedule's rightmost
// branch, which the recorded forward reaches anyway).
std::vector<int> binomial_chain(int nsteps, int nsnap) {
  std::vector<int> chain;
  int a = 0, freeslots = nsnap - 1;
  while (nsteps - a >= 2 && freeslots >= 1) {
    a += (int)rev_split(nsteps - a, freeslots);
    chain.push_back(a);
    --freeslots;
  }
  return chain;
}

// The operations of reversing steps a+1..b (step k maps state k-1 to k)
// from state a held in snapshot slot sa, with the snapshot slots `freev`
// free: `advance(src_state_slot_or_-1, from, to, dst)` and `adjoint(step,
// state_slot)` callbacks; work slots are -1 - w.  Returns false when a
// callback fails.
template <typename Advance, typename Adjoint>
bool reverse_steps(int a, int b, int sa, std::vector<int>& freev, Advance& advance,
                   Adjoint& adjoint) {
  const int l = b - a;
  if (l == 1) return adjoint(b, sa);
  if (freev.empty()) {
    for (int k = b; k > a; --k) {
      int st = sa;
      if (k - 1 > a) {
        st = -1 - ((k - 1 - a - 1) & 1);  // a work state
        if (!advance(sa, a, k - 1, st)) return false;
      }
      if (!adjoint(k, st)) return false;
    }
    return true;
  }
  const int m = a + (int)rev_split(l, (int64_t)freev.size());
  const int sm = freev.back();
  freev.pop_back();
  if (!advance(sa, a, m, sm)) return false;
  if (!reverse_steps(m, b, sm, freev, advance, adjoint)) return false;
  freev.push_back(sm);
  return reverse_steps(a, m, sa, freev, advance, adjoint);
}

}  // namespace

// Forward steps the backward pass of a binomial schedule runs (the whole
// schedule's advances minus those of the stored chain, which the recorded
// forward run did).
int64_t binomial_recompute(int nsteps, int nsnap) {
  const std::vector<int> chain = binomial_chain(nsteps, nsnap);
  int64_t n = 0;
  auto advance = [&](int, int from, int to, int) {
    n += to - from;
    return true;
  };
  auto adjoint = [&](int, int) { return true; };
  int right = nsteps;
  for (int k = (int)chain.size(); k >= 0; --k) {
    const int a = k == 0 ? 0 : chain[(size_t)k - 1];
    std::vector<int> freev;
    for (int f = nsnap - 1; f > k; --f) freev.push_back(f);
    reverse_steps(a, right, k, freev, advance, adjoint);
    right = a;
  }
  return n;
}

namespace {

// bytes per node of the B and C moment planes of the handle's storage
size_t b_bytes(const bgk_handle* h) {
  return h->prm.precision == BGK_FP64_MOM ? sizeof(double4) : sizeof(float4);
}
size_t lam_bytes(const bgk_handle* h) {
  return h->prm.precision == BGK_FP64_MOM ? sizeof(double) : sizeof(float);
}
size_t c_bytes(const bgk_handle* h) {
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  if (h->mom_eqf) return f64 ? sizeof(double) : sizeof(float);
  return f64 ? sizeof(double4) : sizeof(float4);
}
// the adjoint kernel's work split: strips of at most 32 rows with FP32 moments
// (2048^2 and 4096^2 with 16 / 32 / 64: 9.3 / 9.2 / 9.5 and 17.3 / 17.3 / 17.4
// ms), 16 with FP64 (4096^2 with 8 / 16 / 32 / 64: 29.3 / 29.3 / 29.2 / 29.6)
WaveGrid adj_grid(const bgk_handle* h) {
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  return make_wave_grid(h->nx, h->ny, kAdjCols, 1, 2, 1.4, f64 ? 16 : 32, h->n_cu, h->strip_rows,
                        f64 ? adj_waves<double>() : adj_waves<float>());
}

struct Bump {
  char* base;
  size_t off;
  template <typename T>
  T* take(size_t n) {
    off = (off + 255) / 256 * 256;
    T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
    off += n * sizeof(T);
    return p;
  }
  // a lattice plane of elements of esize bytes placed as the handle places
  // its own: element 1 (column 1 of row 0) on a 256-byte boundary, so that
  // with the 64-element pitch every row's column 1 is (the kernels' row
  // accesses then cover whole cache lines)
  template <typename T>
  T* plane(size_t n, size_t esize = sizeof(T)) {
    off = (off + 255) / 256 * 256 + 256 - esize;
    T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
    off += n * esize;
    return p;
  }
};

void carve_state(Bump& b, const bgk_handle* h, StatePtrs* s) {
  const size_t n = (size_t)h->plane_elems;
  s->a = b.plane<double2>(n);
  s->b = b.plane<char>(n, b_bytes(h));
  s->c = b.plane<char>(n, c_bytes(h));
  s->phi = b.plane<double>(n);
  s->te = b.take<double>((size_t)h->ny + 2);
}

// device bytes of everything but the stored states
size_t carve_fixed(bgk_handle* h, AdjCtx* a, Bump& b) {
  const size_t n = (size_t)h->plane_elems;
  const size_t before = b.off;
  for (int l = 0; l < 2; ++l) {
    const size_t e = lam_bytes(h);
    a->lam[l].v[0] = b.plane<char>(n, 4 * e);
    a->lam[l].v[1] = b.plane<char>(n, 4 * e);
    a->lam[l].v[2] = b.plane<char>(n, (h->mom_eqf ? 2 : 4) * e);
    a->lam[l].v[3] = h->mom_eqf ? nullptr : b.plane<char>(n, e);
  }
  a->probe_idx = b.plane<int>(n);
  a->probe_ij = b.take<int>(2 * (size_t)std::max(a->np, 1));
  a->probe_T = b.take<double>((size_t)a->nsteps * std::max(a->np, 1));
  a->seeds = b.take<double>((size_t)a->nsteps * std::max(a->np, 1));
  a->partial = b.take<double>(3 * (size_t)a->nblk);
  a->out3 = b.take<double>(3);
  return b.off - before;
}

size_t carve_ctx(bgk_handle* h, AdjCtx* a, char* base) {
  Bump b{base, 0};
  if (a->nsnap > 0) {
    a->slot.clear();
    a->ckpt.clear();
    a->ckpt2.clear();
    a->snap.assign((size_t)a->nsnap, StatePtrs{});
    for (auto& s : a->snap) carve_state(b, h, &s);
    for (auto& s : a->work) carve_state(b, h, &s);
  } else {
    a->slot.assign((size_t)a->seg + 1, StatePtrs{});
    a->ckpt.assign((size_t)a->nckpt, StatePtrs{});
    a->ckpt2.assign((size_t)a->nckpt2, StatePtrs{});
    for (auto& s : a->slot) carve_state(b, h, &s);
    for (auto& s : a->ckpt) carve_state(b, h, &s);
    for (auto& s : a->ckpt2) carve_state(b, h, &s);
  }
  carve_fixed(h, a, b);
  return b.off + 256;
}

// device bytes of one stored state and of the rest of a context
size_t state_bytes(bgk_handle* h) {
  Bump b{nullptr, 0};
  StatePtrs s;
  carve_state(b, h, &s);
  carve_state(b, h, &s);
  Bump b1{nullptr, 0};
  carve_state(b1, h, &s);
  return b.off - b1.off;
}

hipError_t copy_state(bgk_handle* h, const StatePtrs& dst, const double2* a, const void* bb,
                      const void* c, const double* phi, const double* te) {
  const size_t n = (size_t)h->plane_elems;
  hipError_t e = hipMemcpyAsync(dst.a, a, n * sizeof(double2), hipMemcpyDeviceToDevice, h->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(dst.b, bb, n * b_bytes(h), hipMemcpyDeviceToDevice, h->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(dst.c, c, n * c_bytes(h), hipMemcpyDeviceToDevice, h->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(dst.phi, phi, n * sizeof(double), hipMemcpyDeviceToDevice, h->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(dst.te, te, ((size_t)h->ny + 2) * sizeof(double), hipMemcpyDeviceToDevice,
                       h->stream);
  return e;
}

template <typename R, bool EQF>
void run_adjoint(bgk_handle* h, const AdjArgs& a, int core) {
  const bool wide = wide_rows(h);
  const auto k = core ? (wide ? k_adjoint<R, EQF, false, true> : k_adjoint<R, EQF, false, false>)
                      : (wide ? k_adjoint<R, EQF, true, true> : k_adjoint<R, EQF, true, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)a.g.nwg), dim3(kLanes), 0, h->stream, a);
}

// adjoint of the step from state `sprev` (core = 1), or the initial state's
// share (core = 0, sprev = the initial state)
hipError_t launch_adjoint(bgk_handle* h, AdjCtx* x, const StatePtrs& sprev, int lam_next,
                          int has_next, int core, const double* seeds) {
  AdjArgs a;
  a.sprev = sprev;
  a.next = x->lam[lam_next];
  a.cur = x->lam[1 - lam_next];
  a.has_next = has_next;
  a.probe_idx = x->probe_idx;
  a.seeds = seeds;
  a.partial = x->partial;
  a.c = h->c;
  a.cf = consts_f(h->c);
  const double u = h->c.u0, v = h->c.v0;
  for (int k = 0; k < 9; ++k) {
    const double cu = CX[k] * u + CY[k] * v;
    a.gd[k] = kW[k] * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * (u * u + v * v));
  }
  a.nx = h->nx;
  a.ny = h->ny;
  a.pitch = h->pitch;
  a.interf = h->nx / 40;
  a.g = adj_grid(h);
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  if (h->mom_eqf)
    f64 ? run_adjoint<double, true>(h, a, core) : run_adjoint<float, true>(h, a, core);
  else
    f64 ? run_adjoint<double, false>(h, a, core) : run_adjoint<float, false>(h, a, core);
  return hipGetLastError();
}

// Whether two steps with the state between them kept go in one launch.  Measured,
// ms per gradient of 60 steps (segments of 20), backward pass, two launches / one:
// FP32 moments 512^2 1.70 / 1.71, 1024^2 4.20 / 3.96, 2048^2 15.5 / 14.1, FP64
// 512^2 2.26 / 2.35, 724^2 3.53 / 3.61, 1024^2 7.49 / 7.19, 2048^2 26.7 / 24.7; with
// omega_f = 1 FP32 512^2 1.55 / 1.56, 724^2 2.15 / 2.07, 2048^2 12.5 / 11.4, FP64 724^2
// 2.98 / 2.71, 2048^2 20.1 / 18.4.  (BGK_MOM_VARIANT of 2 or 3: at any size.)
bool keeps_between(const bgk_handle* h) {
  if (mom_most_steps(h, true) < 2) return false;
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  const int64_t least = (int64_t)1 << (f64 && !h->mom_eqf ? 20 : 19);
  return h->mom_variant > 0 || (int64_t)h->nx * h->ny >= least;
}

// T forward steps from state `in` to state `out` (explicit buffers) in one launch;
// T = 2 with `mid`: the state between them too
hipError_t fwd_steps(bgk_handle* h, int T, const StatePtrs& in, const StatePtrs* mid,
                     const StatePtrs& out, double* probe_out, const int* probe_idx, int np,
                     bool write_all) {
  mom::MomStep st;
  st.in = mom::MomIn{in.a, in.b, in.c};
  st.out = mom::MomOut{out.a, out.b, out.c};
  st.pa = in.phi;
  st.pb = out.phi;
  st.te_in = in.te;
  st.te_out = out.te;
  st.write_all = write_all;
  st.probe_idx = probe_idx;
  st.probe_out = probe_out;
  st.probe_np = np;
  if (mid) {
    st.mid = mom::MomOut{mid->a, mid->b, mid->c};
    st.phi_mid = mid->phi;
    st.te_mid = mid->te;
  }
  return launch_mom_steps(h, st, T);
}

}  // namespace

void adj_free(bgk_handle* h) {
  if (!h->adj) return;
  if (h->adj->pool) (void)hipFree(h->adj->pool);
  delete h->adj;
  h->adj = nullptr;
}

int64_t adj_state_bytes(bgk_handle* h) { return (int64_t)state_bytes(h); }

int64_t adj_bytes(bgk_handle* h, int nsteps, int np, int nsnap) {
  AdjCtx x;
  x.nsteps = nsteps;
  x.np = np;
  x.nsnap = nsnap;
  x.nblk = adj_grid(h).nwg;
  return (int64_t)carve_ctx(h, &x, nullptr);
}

// nsnap > 0: binomial schedule with nsnap snapshot slots; else the level
// schedule (seg_outer > 0: two levels)
hipError_t adj_setup(bgk_handle* h, int nsteps, int seg_outer, int seg, int nsnap, int np,
                     const int32_t* pi, const int32_t* pj) {
  adj_free(h);
  AdjCtx* x = new (std::nothrow) AdjCtx();
  if (!x) return hipErrorOutOfMemory;
  x->nsteps = nsteps;
  x->np = np;
  x->nsnap = nsnap;
  if (nsnap > 0) {
    x->chain = binomial_chain(nsteps, nsnap);
  } else {
    x->seg = seg;
    x->seg1 = seg_outer;
    const int lvl1 = seg_outer > 0 ? seg_outer : seg;
    x->nckpt = (nsteps + lvl1 - 1) / lvl1;
    // (the first checkpoint of an outer segment is the outer checkpoint)
    x->nckpt2 = seg_outer > 0 ? (std::min(seg_outer, nsteps) + seg - 1) / seg - 1 : 0;
  }
  x->nblk = adj_grid(h).nwg;
  x->bytes = carve_ctx(h, x, nullptr);
  hipError_t e = hipMalloc(&x->pool, x->bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // (the failed allocation's error is reported here)
    delete x;
    return e;
  }
  carve_ctx(h, x, static_cast<char*>(x->pool));
  h->adj = x;
  std::vector<int> ij(2 * (size_t)std::max(np, 1), 0);
  for (int p = 0; p < np; ++p) {
    ij[2 * p] = pi[p];
    ij[2 * p + 1] = pj[p];
  }
  e = hipMemsetAsync(x->pool, 0, x->bytes, h->stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(x->probe_ij, ij.data(), ij.size() * sizeof(int), hipMemcpyHostToDevice,
                       h->stream);
  if (e == hipSuccess) {
    const int64_t n = h->plane_elems;
    hipLaunchKernelGGL(k_probe_clear, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream,
                       x->probe_idx, n);
    if (np > 0)
      hipLaunchKernelGGL(k_probe_set, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, h->stream,
                         x->probe_idx, x->probe_ij, np, h->pitch);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  return e;
}

bool adj_forward_done(const bgk_handle* h) { return h->adj && h->adj->forward_done; }

void adj_invalidate(bgk_handle* h) {
  if (h->adj) h->adj->forward_done = false;
}

hipError_t adj_forward(bgk_handle* h, double* probe_T_host) {
  AdjCtx* x = h->adj;
  x->forward_done = false;
  // east column of the initial state (T(Nx, :) as the first BC_g reads it)
  hipError_t e = launch_teast_prologue(h);
  if (e != hipSuccess) return e;
  size_t next_chain = 0;
  const int lvl1 = x->seg1 > 0 ? x->seg1 : x->seg;
  // the state before step 0: the handle's own, kept as a copy
  StatePtrs in{h->ma[h->cur], h->mb[h->cur], h->mc[h->cur], h->phi[h->pc], h->teast[h->te_cur]};
  const StatePtrs& first = x->nsnap > 0 ? x->snap[0] : x->ckpt[0];
  e = copy_state(h, first, in.a, in.b, in.c, in.phi, in.te);
  // the first state after n that is kept (its step in *stop), null: none is
  auto next_kept = [&](int n, size_t chain, int* stop) -> const StatePtrs* {
    *stop = x->nsteps;
    if (x->nsnap > 0) {
      if (chain >= x->chain.size()) return nullptr;
      *stop = x->chain[chain];
      return &x->snap[chain + 1];
    }
    if ((n / lvl1 + 1) * lvl1 >= x->nsteps) return nullptr;
    *stop = (n / lvl1 + 1) * lvl1;
    return &x->ckpt[(size_t)(*stop / lvl1)];
  };
  const int cur0 = h->cur;
  for (int n = 0; e == hipSuccess && n < x->nsteps;) {
    // the launch that reaches a state that is kept writes it in its place, and
    // the one after reads it there, so no state but the first is copied (2048^2,
    // FP32, 12 states kept of 48 steps: 11 copies of 84 us less in 4 ms)
    int stop;
    const StatePtrs *keep = next_kept(n, next_chain, &stop), *mid = nullptr;
    int T = mom_next_steps(h, stop - n, true);
    if (keep && stop == n + 1 && n + 4 <= x->nsteps && keeps_between(h)) {
      mid = keep;
      keep = next_kept(n + 1, ++next_chain, &stop);
      T = 2;
    }
    const int b = 1 - h->cur;
    const StatePtrs own{h->ma[b], h->mb[b], h->mc[b], h->phi[1 - h->pc], h->teast[1 - h->te_cur]};
    const bool kept = keep && n + T == stop;
    const StatePtrs out = kept ? *keep : own;
    e = fwd_steps(h, T, in, mid, out, x->np > 0 ? x->probe_T + (size_t)n * x->np : nullptr,
                  x->probe_idx, x->np, mom_write_all(x->nsteps - n - T, false));
    if (e != hipSuccess) return e;
    if (kept) {
      ++next_chain;
    } else {
      h->cur = b;
      h->pc = 1 - h->pc;
      h->te_cur = 1 - h->te_cur;
    }
    in = out;
    n += T;
  }
  if (e == hipSuccess && h->recorded && (h->cur ^ cur0) != (x->nsteps & 1)) {
    const int b = 1 - h->cur;
    const StatePtrs own{h->ma[b], h->mb[b], h->mc[b], h->phi[1 - h->pc], h->teast[1 - h->te_cur]};
    e = copy_state(h, own, in.a, in.b, in.c, in.phi, in.te);
    h->cur = b;
    h->pc = 1 - h->pc;
    h->te_cur = 1 - h->te_cur;
  }
  if (e == hipSuccess && x->np > 0)
    e = hipMemcpyAsync(probe_T_host, x->probe_T, (size_t)x->nsteps * x->np * sizeof(double),
                       hipMemcpyDeviceToHost, h->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  if (e == hipSuccess) x->forward_done = true;
  return e;
}

void adj_info(const bgk_handle* h, int64_t* bytes, int32_t* n_states) {
  const AdjCtx* x = h->adj;
  *bytes = (int64_t)x->bytes;
  *n_states = x->nsnap > 0 ? (int32_t)(x->snap.size() + 2)
                           : (int32_t)(x->slot.size() + x->ckpt.size() + x->ckpt2.size());
}

int64_t adj_recomputed(const bgk_handle* h) { return h->adj ? h->adj->recomputed : 0; }

hipError_t adj_backward(bgk_handle* h, const double* seeds_host, double grad[3]) {
  AdjCtx* x = h->adj;
  hipError_t e = hipSuccess;
  x->recomputed = 0;
  if (x->np > 0)
    e = hipMemcpyAsync(x->seeds, seeds_host, (size_t)x->nsteps * x->np * sizeof(double),
                       hipMemcpyHostToDevice, h->stream);
  if (e == hipSuccess)
    e = hipMemsetAsync(x->partial, 0, 3 * (size_t)x->nblk * sizeof(double), h->stream);
  int ln = 0;  // lam[ln] holds the adjoint of the step after the current one
  bool has_next = false;
  // adjoint of step n (1-based) from the state before it
  auto adjoint_step = [&](int n, const StatePtrs& before) {
    const double* sd = x->np > 0 ? x->seeds + (size_t)(n - 1) * x->np : nullptr;
    e = launch_adjoint(h, x, before, ln, has_next ? 1 : 0, 1, sd);
    ln = 1 - ln;
    has_next = true;
    return e == hipSuccess;
  };
  auto steps = [&](int T, const StatePtrs& in, const StatePtrs* mid, const StatePtrs& out) {
    x->recomputed += T;
    e = fwd_steps(h, T, in, mid, out, nullptr, nullptr, 0, false);
    return e == hipSuccess;
  };
  const bool pairs = keeps_between(h);
  auto step = [&](const StatePtrs& in, const StatePtrs& out) {
    return steps(1, in, nullptr, out);
  };
  // from state `src` on by n steps to state `dst`, through two scratch states,
  // of which `dst` may be one, and `src` the one that the first launch does not
  // write: launch m writes scratch (first_scratch + m) & 1, the one before last
  // not `dst`
  auto first_scratch = [&](int n, const StatePtrs& dst, const StatePtrs* scratch) {
    int launches = 0;
    for (int left = n; left > 0; ++launches) left -= mom_next_steps(h, left, true);
    return (&dst == &scratch[0] ? 1 : 0) ^ (launches & 1);
  };
  auto run = [&](const StatePtrs& src, int n, const StatePtrs& dst, const StatePtrs* scratch) {
    int k = first_scratch(n, dst, scratch);
    const StatePtrs* in = &src;
    for (int left = n; left > 0; k ^= 1) {
      const int T = mom_next_steps(h, left, true);
      left -= T;
      const StatePtrs* out = left == 0 ? &dst : &scratch[k];
      if (!steps(T, *in, nullptr, *out)) return false;
      in = out;
    }
    return true;
  };
  if (x->nsnap > 0) {
    // binomial schedule: slots >= 0 are snapshots, -1 and -2 the work states
    auto at = [&](int sl) -> const StatePtrs& { return sl >= 0 ? x->snap[(size_t)sl] : x->work[-1 - sl]; };
    // an advance by one step waits for the next one from the state it gives,
    // to share its first launch
    const StatePtrs *one_src = nullptr, *one_dst = nullptr;
    auto flush = [&]() {
      if (!one_src) return true;
      const StatePtrs* src = one_src;
      one_src = nullptr;
      return step(*src, *one_dst);
    };
    auto advance = [&](int src, int from, int to, int dst) {
      const StatePtrs *s = &at(src), *d = &at(dst);
      const int n = to - from;
      if (one_src && one_dst == s) {
        const StatePtrs* o = n == 1 ? d : &x->work[1 - first_scratch(n - 1, *d, x->work)];
        const StatePtrs* from0 = one_src;
        one_src = nullptr;
        if (!steps(2, *from0, s, *o)) return false;
        return n == 1 || run(*o, n - 1, *d, x->work);
      }
      if (!flush()) return false;
      if (n == 1 && pairs && src >= 0 && dst >= 0) {
        one_src = s;
        one_dst = d;
        return true;
      }
      return run(*s, n, *d, x->work);
    };
    auto adjoint = [&](int n, int sl) { return flush() && adjoint_step(n, at(sl)); };
    int right = x->nsteps;
    for (int k = (int)x->chain.size(); k >= 0 && e == hipSuccess; --k) {
      const int a = k == 0 ? 0 : x->chain[(size_t)k - 1];
      std::vector<int> freev;
      for (int f = x->nsnap - 1; f > k; --f) freev.push_back(f);
      reverse_steps(a, right, k, freev, advance, adjoint);
      right = a;
    }
  } else {
    // steps n0..n1-1 from `start` (the state before step n0): recompute every
    // state of the segment (state n0 is `start` itself), then reverse them
    auto inner = [&](const StatePtrs& start, int n0, int n1) {
      auto st = [&](int n) -> const StatePtrs& { return n == n0 ? start : x->slot[n - n0]; };
      for (int n = n0 + 1; n < n1 && e == hipSuccess;) {
        const bool two = pairs && n + 1 < n1;
        two ? steps(2, st(n - 1), &st(n), st(n + 1)) : step(st(n - 1), st(n));
        n += two ? 2 : 1;
      }
      for (int n = n1; n > n0 && e == hipSuccess; --n) adjoint_step(n, st(n - 1));
    };
    if (x->seg1 == 0) {
      for (int s = x->nckpt - 1; s >= 0 && e == hipSuccess; --s)
        inner(x->ckpt[s], s * x->seg, std::min((s + 1) * x->seg, x->nsteps));
    } else {
      for (int s1 = x->nckpt - 1; s1 >= 0 && e == hipSuccess; --s1) {
        const int m0 = s1 * x->seg1, m1 = std::min(m0 + x->seg1, x->nsteps);
        const int ns2 = (m1 - m0 + x->seg - 1) / x->seg;
        // checkpoints of this outer segment: c2(k) = state m0 + k seg, c2(0)
        // the outer checkpoint itself; the steps in between go through
        // slot[0] and slot[1]
        auto c2 = [&](int k) -> const StatePtrs& { return k == 0 ? x->ckpt[s1] : x->ckpt2[k - 1]; };
        for (int k = 1; k < ns2 && e == hipSuccess; ++k) {
          run(c2(k - 1), x->seg, x->ckpt2[k - 1], x->slot.data());
        }
        for (int s2 = ns2 - 1; s2 >= 0 && e == hipSuccess; --s2)
          inner(c2(s2), m0 + s2 * x->seg, std::min(m0 + (s2 + 1) * x->seg, m1));
      }
    }
  }
  // the initial state's share (hot-wall temperature of the liquid strip)
  const StatePtrs& s0 = x->nsnap > 0 ? x->snap[0] : x->ckpt[0];
  if (e == hipSuccess) e = launch_adjoint(h, x, s0, ln, has_next ? 1 : 0, 0, nullptr);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_adj_sum, dim3(1), dim3(256), 0, h->stream, x->partial, x->nblk, x->out3);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(grad, x->out3, 3 * sizeof(double), hipMemcpyDeviceToHost, h->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  return e;
}

}  // namespace bgk
