// bgk_stream_mom.hip -- T moment-storage time steps in one launch.
//
// The node update is that of bgk_mom.h on the walk of bgk_wave.h: one wave,
// 64 columns, row after row, level t of T one step ahead of level t - 1.  A
// level keeps of a row only what its neighbours' pulls need: the populations
// of a row are formed once, in the lane of their node, and enter the pulled
// sums of the rows below, beside and above it as three numbers per moment
// family (struct Triple), the columns beside it through lane shifts.  That is
// 290 VALU instructions per node and step; rebuilding the nine upstream
// populations at every pull (bgk_fused_mom.hip) takes 470.
//
// What bounds it: one step per launch is bound by HBM (112 B per node with
// FP32 moments); two steps per launch halve the bytes and leave it bound by
// VALU issue at two waves per SIMD (FP32 moments: 212 VGPRs).  Measured at
// 4096^2, us per step, against one step per launch of the ring kernel:
// FP32 moments 203 (362), with omega_f = 1 168 (290), FP64 moments 323 (648),
// with omega_f = 1 180 (462, three steps per launch).  FP32 moments with three
// steps per launch: 230 (spills), with omega_f = 1 172.
#include <algorithm>

#include "bgk_mom.h"
#include "bgk_wave.h"

// Every multiply-add below is written out: contraction chosen by the compiler
// could differ between instantiations, and a step has to give the same bits
// whichever launch it is part of.
#pragma clang fp contract(off)

namespace bgk {
namespace {

using namespace mom;
using namespace wave;

struct Macro {
  double *rho, *u, *v, *T;
};

// Moments of a node as the rebuild of its populations takes them.
struct NodeD {
  double rho, th, u, v, pfxx, pfyy, pfxy, pgxx, pgyy, pgxy, phi;
};

// A row as loaded: converted only when it is fed.
template <typename R, bool EQF>
struct Raw {
  double2 a;
  typename Vec<R>::V4 b;
  typename CType<R, EQF>::T c;
  double phi;
};

template <typename R, bool EQF>
__device__ __forceinline__ Raw<R, EQF> load_raw(const MomIn& in, const double* __restrict__ pa,
                                                int64_t q) {
  Raw<R, EQF> n;
  n.a = in.a[q];
  n.b = b_at<R, EQF>(in.b, q);
  n.c = c_at<R, EQF>(in.c, q);
  n.phi = pa[q];
  return n;
}

template <typename R, bool EQF>
__device__ __forceinline__ NodeD widen(const Raw<R, EQF>& r) {
  NodeD n;
  n.rho = taken(r.a.x);
  n.th = taken(r.a.y);
  n.u = (double)r.b.x;
  n.v = (double)r.b.y;
  if constexpr (EQF) {
    n.pfxx = n.pfyy = n.pfxy = 0.0;
    n.pgxx = (double)r.b.z;
    n.pgyy = (double)r.b.w;
    n.pgxy = (double)r.c;
  } else {
    n.pfxx = (double)r.b.z;
    n.pfyy = (double)r.b.w;
    n.pfxy = (double)r.c.x;
    n.pgxx = (double)r.c.y;
    n.pgyy = (double)r.c.z;
    n.pgxy = (double)r.c.w;
  }
  n.phi = taken(r.phi);
  return n;
}

// The nine populations of a node from (m0, m, j = m (u, v) and P): m0 = m =
// rho for f; m0 = T - T_crit, m = T for g, whose populations are the
// deviations g_k - w_k T_crit.  With Q = 9/2 (m u u + P), E = m0 - tr Q / 3:
// p_k = w_k (E + c c : Q + 3 c . j).
template <bool HAVE_P>
__device__ __forceinline__ void populations(double m0, double m, double u, double v, double pxx,
                                            double pyy, double pxy, double p[9]) {
  const double jx = m * u, jy = m * v;
  double qxx, qyy, qxy;
  if constexpr (HAVE_P) {
    qxx = 4.5 * fma(jx, u, pxx);
    qyy = 4.5 * fma(jy, v, pyy);
    qxy = 9.0 * fma(jx, v, pxy);
  } else {
    qxx = 4.5 * (jx * u);
    qyy = 4.5 * (jy * v);
    qxy = 9.0 * (jx * v);
  }
  const double s = qxx + qyy;
  const double e = fma(s, -1.0 / 3.0, m0);
  const double ax = (e + qxx) * (1.0 / 9.0), ay = (e + qyy) * (1.0 / 9.0), d = e + s;
  const double dp = (d + qxy) * (1.0 / 36.0), dm = (d - qxy) * (1.0 / 36.0);
  const double jp = jx + jy, jm = jx - jy;
  p[0] = e * (4.0 / 9.0);
  p[1] = fma(jx, 1.0 / 3.0, ax);
  p[3] = fma(jx, -1.0 / 3.0, ax);
  p[2] = fma(jy, 1.0 / 3.0, ay);
  p[4] = fma(jy, -1.0 / 3.0, ay);
  p[5] = fma(jp, 1.0 / 12.0, dp);
  p[7] = fma(jp, -1.0 / 12.0, dp);
  p[8] = fma(jm, 1.0 / 12.0, dm);
  p[6] = fma(jm, -1.0 / 12.0, dm);
}

// What three neighbouring source nodes of one row give to a node's pulled
// sums: their total, the total of the two diagonals, and the difference
// (eastward - westward) of the diagonals.
struct Triple {
  double n, p, d;
};
__device__ __forceinline__ Triple triple(double c, double w, double e) {
  const double p = w + e;
  return Triple{c + p, p, w - e};
}

// Registers of one level between two rows.
struct Level {
  // row awaiting its northern neighbours: pulled sums so far, phi sums of
  // its own and the southern row, its centre tap
  PullSums s;
  double t1, t2, pc;
  // the southern share of the row after it
  Triple sf, sg;
  double n1, n2;
};

struct Updated {
  double rho, dT, u, v, pfxx, pfyy, pfxy, pgxx, pgyy, pgxy, phi;  // stored
  double dT2, u2, v2;                                              // before the forces
};

// momentsPre .. collision of one node (see core_forward_t in bgk_mom.h for
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

// The initial phi of the ghost columns 0 and Nx+1, which no step changes
// (STEP_7/initialization.f90:15-26: liquid for i <= Nx/40).
constexpr double kPhiWest = 1.0, kPhiEast = -1.0;

// Stores of a strip's nodes through buffer descriptors: a lane that must not
// store gives an offset past the strip.
template <typename R, bool EQF>
struct StoreMom {
  using V4 = typename Vec<R>::V4;
  using C = typename CType<R, EQF>::T;
  __amdgpu_buffer_rsrc_t a, b, c, phi;
  __device__ __forceinline__ StoreMom(const MomOut& out, double* pb, int64_t qs, int n) {
    a = strip_buffer(out.a + qs, n);
    b = strip_buffer(static_cast<V4*>(out.b) + qs, n);
    c = strip_buffer(static_cast<C*>(out.c) + qs, n);
    phi = strip_buffer(pb + qs, n);
  }
  __device__ __forceinline__ void store(int q, bool on, bool on_phi, const Updated& o) const {
    const int qa = on ? q : kPastStrip;
    buffer_put(a, qa, make_double2(o.rho, o.dT));
    if constexpr (EQF) {
      buffer_put(b, qa, make4<R>((R)o.u, (R)o.v, (R)o.pgxx, (R)o.pgyy));
      buffer_put(c, qa, (R)o.pgxy);
    } else {
      buffer_put(b, qa, make4<R>((R)o.u, (R)o.v, (R)o.pfxx, (R)o.pfyy));
      buffer_put(c, qa, make4<R>((R)o.pfxy, (R)o.pgxx, (R)o.pgyy, (R)o.pgxy));
    }
    buffer_put(phi, on_phi ? q : kPastStrip, o.phi);
  }
};

struct StreamArgs {
  MomIn in;
  MomOut out;
  const double* pa;
  double* pb;
  const double* te_in;
  double* te_out;
  Macro m;
  StepC c;
  double tin, t_cold, u0, v0, frozen6, frozen7;
  int east_cold;
  int nx, ny;
  int64_t pitch;
  WaveGrid g;
  const int* probe_idx;
  double* probe_out;
  int probe_np;
};

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
template <bool EQF, bool EDGE>
__device__ __forceinline__ void feed(Level& L, const NodeD& nd, int j, int ny, int i, int nx,
                                     bool has_w, bool has_e, double frozen6, double frozen7,
                                     PullSums* S, double* st, double* st2, double* pc) {
  *S = L.s;
  *st = L.t1;
  *st2 = L.t2;
  *pc = L.pc;
  if (EDGE && j > ny) return;
  double f[9], g[9];
  populations<!EQF>(nd.rho, nd.rho, nd.u, nd.v, nd.pfxx, nd.pfyy, nd.pfxy, f);
  populations<true>(nd.th, kTcrit + nd.th, nd.u, nd.v, nd.pgxx, nd.pgyy, nd.pgxy, g);
  // row sums of the phi taps
  const double pw = from_west(nd.phi), pe = from_east(nd.phi);
  const double r1 = (pw + pe) + nd.phi;
  const double r2 = fma(nd.phi, nd.phi, fma(pw, pw, pe * pe));
  // northern sources of row j - 1
  const Triple nf = triple(f[4], from_west(f[8]), from_east(f[7]));
  const Triple ng = triple(g[4], from_west(g[8]), from_east(g[7]));
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
  const Triple sf = triple(f[2], from_west(f[5]), from_east(f[6]));
  const Triple sg = triple(g[2], from_west(g[5]), from_east(g[6]));
  if (EDGE && j == 1) {  // row 0: bounce-back, copied g and phi
    const double f6 = i == nx ? frozen6 : f[8];
    L.sf = triple(f[4], f[7], f6);
    L.sg = sg;
    L.n1 = r1;
    L.n2 = r2;
  }
  // row j: southern share, then its own row's sources
  {
    const Triple cf = triple(f[0], from_west(f[1]), from_east(f[3]));
    const Triple cg = triple(g[0], from_west(g[1]), from_east(g[3]));
    L.s.rho = L.sf.n + cf.n;
    L.s.jx = L.sf.d + cf.d;
    L.s.jy = L.sf.n;
    L.s.fxx = L.sf.p + cf.p;
    L.s.fyy = L.sf.n;
    L.s.fxy = L.sf.d;
    L.s.dT = L.sg.n + cg.n;
    L.s.gxx = L.sg.p + cg.p;
    L.s.gyy = L.sg.n;
    L.s.gxy = L.sg.d;
    L.t1 = L.n1 + r1;
    L.t2 = L.n2 + r2;
    L.pc = nd.phi;
  }
  if (EDGE) {
    if (j == ny) {  // row Ny+1: bounce-back, copied g and phi
      const Triple v = triple(f[2], f[6], i == nx ? frozen7 : f[5]);
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
      const double a = on ? f[3] : 0.0;
      const double b = on && j != 1 ? f[7] : 0.0;
      const double d = on && j != ny ? f[6] : 0.0;
      L.s.rho += a + b + d;
      L.s.jx += a + b + d;
      L.s.jy += b - d;
      L.s.fxx += a + b + d;
      L.s.fyy += b + d;
      L.s.fxy += b - d;
    }
    if (has_e) {  // column Nx: directions 3, 6, 7 bounce back
      const bool on = i == nx;
      const double a = on ? f[1] : 0.0;
      const double b = on && j != 1 ? f[8] : 0.0;
      const double d = on && j != ny ? f[5] : 0.0;
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

// What the last launch of a call adds for row jc (1..Ny) completed by level t
// of T: the halo as BC_f / BC_g leave it at the start of the last step, and
// the macroscopic fields after it.
template <int T>
__device__ __forceinline__ void finish(const StreamArgs& A, int t, int jc, int i,
                                       const Updated& o, double tav) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch, q = (int64_t)jc * P + i;
  if (t == (T >= 2 ? T - 2 : 0)) {
    const bool s_row = jc == 1, n_row = jc == ny;
    const int64_t rj = (int64_t)jc * P, rn = (int64_t)(ny + 1) * P;
    // the state the last step starts from: of this level, or (T = 1) still in
    // the planes, which this lane overwrites below
    double rho = o.rho, Tp = tav, ph = o.phi, te = tav;
    if (T == 1 && (s_row || n_row)) {
      rho = A.m.rho[q];
      Tp = A.m.T[q];
      ph = A.pa[q];
    }
    if (s_row) {
      A.m.rho[i] = rho;
      A.m.T[i] = Tp;
      A.m.u[i] = A.m.v[i] = 0.0;
      A.pb[i] = ph;
    }
    if (n_row) {
      A.m.rho[rn + i] = rho;
      A.m.T[rn + i] = Tp;
      A.m.u[rn + i] = A.m.v[rn + i] = 0.0;
      A.pb[rn + i] = ph;
    }
    if (i == 1) {
      A.m.T[rj] = A.tin;
      if (s_row) A.m.T[0] = A.tin;
      if (n_row) A.m.T[rn] = A.tin;
      if (s_row) A.pb[0] = kPhiWest;
      if (n_row) A.pb[rn] = kPhiWest;
    }
    if (i == nx) {
      if (T == 1) te = A.te_in[jc];
      if (A.east_cold) te = A.t_cold;
      A.m.T[rj + nx + 1] = te;
      if (s_row) A.m.T[nx + 1] = te;
      if (n_row) A.m.T[rn + nx + 1] = te;
      if (s_row) A.pb[nx + 1] = kPhiEast;
      if (n_row) A.pb[rn + nx + 1] = kPhiEast;
    }
  }
  if (t == T - 1) {
    A.m.rho[q] = o.rho;
    A.m.T[q] = tav;
    A.m.u[q] = (o.u + o.u2) * 0.5;
    A.m.v[q] = (o.v + o.v2) * 0.5;
  }
}

// The probe record of row jc after level t (T averaged as moments.f90).
__device__ __forceinline__ void record(const StreamArgs& A, int t, int jc, int i, double tav) {
  const int p = A.probe_idx[(int64_t)jc * A.pitch + i];
  if (p >= 0) A.probe_out[(int64_t)t * A.probe_np + p] = tav;
}

// What a launch observes besides the state: nothing, probes, or probes and the
// end of a call (separate instantiations: the probe test alone costs the
// plain loop 40 VGPRs).
enum { kPlain, kProbes, kFinal };

// One wave's strip.  EDGE: the wave or the strip touches a wall.  But for the
// last launch of a call the loop holds one path for its loads
// and stores: masked lanes and rows store out of the buffer's range, which
// the hardware drops, so that the wait for a row's loads (issued two rows
// ahead) never has to cover stores issued since.  With conditional stores the
// compiler's waits did, and a row cost 2.2 us of store latency on top.
template <int T, typename R, bool EQF, bool EDGE, int MODE>
__device__ __forceinline__ void stream_strip(const StreamArgs& A, int i0, int j0, int j1, int i,
                                             bool has_w, bool has_e) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch;
  const int lane = (int)threadIdx.x;
  const int ic = i < 0 ? 0 : (i > nx + 1 ? nx + 1 : i);  // column loaded
  const bool ghost = EDGE && (i == 0 || i == nx + 1);
  const bool own = lane >= T && lane < kLanes - T && i <= nx;  // columns this wave stores
  // phi also in the ghost columns next to an owned column
  const bool own_phi = own || (ghost && (i == 0 ? has_w : lane <= kLanes - T));
  const int64_t qs = (int64_t)j0 * P;  // first node of the strip
  const StoreMom<R, EQF> out(A.out, A.pb, qs, (j1 - j0 + 1) * (int)P);

  // rows of the strip that hold a probe (the flags in column 0 of the probe
  // index plane; at most kMaxRows rows)
  uint64_t probes = 0;
  if (MODE != kPlain && A.probe_out)
    probes = __ballot(j0 + lane <= j1 && A.probe_idx[(int64_t)min(j0 + lane, j1) * P] >= 0);

  Level L[T];
#pragma unroll
  for (int t = 0; t < T; ++t) L[t] = Level{};
  const int ra = EDGE ? max(1, j0 - T) : j0 - T, rb = j1 + T;
  Raw<R, EQF> raw0 = load_raw<R, EQF>(A.in, A.pa, (int64_t)ra * P + ic);
  Raw<R, EQF> raw1 = load_raw<R, EQF>(A.in, A.pa, (int64_t)min(ra + 1, ny) * P + ic);
  const scalar_ptr te_in = as_scalar(A.te_in);
  const __amdgpu_buffer_rsrc_t te_out = strip_buffer(A.te_out, ny + 2);
  double te_row = EDGE ? te_in[ra] : 0.0;
  __builtin_amdgcn_s_waitcnt(kWaitLoads);
  auto feed_row = [&](int r, Raw<R, EQF>& raw) __attribute__((always_inline)) {
    NodeD nd = widen<R, EQF>(raw);
    __builtin_amdgcn_sched_barrier(0);
    raw = load_raw<R, EQF>(A.in, A.pa, (int64_t)min(r + 2, ny) * P + ic);
    const double te0 = te_row;
    if (EDGE) te_row = te_in[min(r + 1, ny)];
    Updated o;
    double tav = 0.0;  // averaged T of the row fed to the level
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int j = r - t;  // row fed to level t
      if (j < j0 - (T - t) || (EDGE && (j < 1 || j > ny + 1))) continue;
      if (EDGE && j <= ny) {
        // ghost columns: no flow populations, the wall's T and velocity
        double te = t == 0 ? te0 : from_west(tav);
        if (A.east_cold) te = A.t_cold;
        if (ghost) {
          nd.rho = nd.pfxx = nd.pfyy = nd.pfxy = nd.pgxx = nd.pgyy = nd.pgxy = 0.0;
          nd.th = (i == 0 ? A.tin : te) - kTcrit;
          nd.u = A.u0;
          nd.v = A.v0;
          nd.phi = i == 0 ? kPhiWest : kPhiEast;
        }
      }
      PullSums S;
      double st, st2, pc;
      feed<EQF, EDGE>(L[t], nd, j, ny, i, nx, has_w, has_e, A.frozen6, A.frozen7, &S, &st, &st2,
                      &pc);
      o = update<R, EQF>(A.c, S, st, st2, pc);
      tav = kTcrit + (o.dT + o.dT2) * 0.5;
      const int jd = j - 1 - j0;  // (rows outside the strip are its neighbours')
      if (MODE != kPlain && jd >= 0 && jd < kMaxRows && ((probes >> jd) & 1) && own)
        record(A, t, j - 1, i, tav);
      if (MODE == kFinal && jd >= 0 && j - 1 <= j1 && own) finish<T>(A, t, j - 1, i, o, tav);
      if (t < T - 1) {
        nd.rho = o.rho;
        nd.th = o.dT;
        nd.u = o.u;
        nd.v = o.v;
        nd.pfxx = o.pfxx;
        nd.pfyy = o.pfyy;
        nd.pfxy = o.pfxy;
        nd.pgxx = o.pgxx;
        nd.pgyy = o.pgyy;
        nd.pgxy = o.pgxy;
        nd.phi = o.phi;
      }
    }
    const int jc = r - T;  // row completed by the last level
    const bool on = jc >= j0;
    const int qo = (jc - j0) * (int)P + i;
    if (EDGE && ghost) o.phi = i == 0 ? kPhiWest : kPhiEast;
    out.store(qo, on && own, on && own_phi, o);
    if (EDGE) buffer_put(te_out, on && jc <= j1 && own && i == nx ? jc : kPastStrip, tav);
  };
  for (int r = ra; r <= rb; r += 2) {
    feed_row(r, raw0);
    feed_row(r + 1, raw1);
  }
}

template <int T, typename R, bool EQF, int MODE>
__global__ __launch_bounds__(kLanes, 2) void k_stream_mom(StreamArgs A) {
  int seg, j0, j1;
  bool edge;
  if (!wave_tile(A.g, A.ny, &seg, &j0, &j1, &edge)) return;
  const int i0 = seg * (kLanes - 2 * T) + 1;
  const int i = i0 - T + (int)threadIdx.x;
  if (edge)
    stream_strip<T, R, EQF, true, MODE>(A, i0, j0, j1, i, i0 - T <= 1, i0 - T + kLanes - 1 >= A.nx);
  else
    stream_strip<T, R, EQF, false, MODE>(A, i0, j0, j1, i, false, false);
}

StepC step_constants(const Consts& c) {
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

template <int T, typename R, bool EQF>
hipError_t launch_t(bgk_handle* h, const MomStep& st) {
  StreamArgs a;
  a.in = st.in;
  a.out = st.out;
  a.pa = st.pa;
  a.pb = st.pb;
  a.te_in = st.te_in;
  a.te_out = st.te_out;
  a.m = Macro{h->rho, h->u, h->v, h->T};
  a.c = step_constants(h->c);
  a.tin = h->c.tin;
  a.t_cold = h->c.t_cold;
  a.u0 = h->c.u0;
  a.v0 = h->c.v0;
  a.frozen6 = h->c.frozen6;
  a.frozen7 = h->c.frozen7;
  a.east_cold = h->c.east_cold;
  a.nx = h->nx;
  a.ny = h->ny;
  a.pitch = h->pitch;
  a.probe_idx = st.probe_idx;
  a.probe_out = st.probe_out;
  a.probe_np = st.probe_np;
  // Strips of at most 64 rows with FP32 moments, 16 with FP64; a row beside a
  // wall counts 1.4 (measured at 1.2 / 1.6 / 2.2, us per step: 512^2 8.9 / 9.5
  // / 10.9, 1003 x 777 15.2 / 15.3 / 17.4, 4096^2 210 / 202 / 209; all strips
  // alike, walls in turn: 11.0, 18.5, 210).  FP64 moments at 4096^2 with at most
  // 16 / 32 rows: 323 / 334.
  constexpr int most = sizeof(R) == sizeof(float) ? 64 : 16;
  a.g = make_wave_grid(h->nx, h->ny, kLanes - 2 * T, T, 2 * T, 1.4, most, h->n_cu, h->strip_rows);
  const dim3 grd((unsigned)a.g.nwg);
  if (st.write_all)
    hipLaunchKernelGGL((k_stream_mom<T, R, EQF, kFinal>), grd, dim3(kLanes), 0, h->stream, a);
  else if (st.probe_out)
    hipLaunchKernelGGL((k_stream_mom<T, R, EQF, kProbes>), grd, dim3(kLanes), 0, h->stream, a);
  else
    hipLaunchKernelGGL((k_stream_mom<T, R, EQF, kPlain>), grd, dim3(kLanes), 0, h->stream, a);
  return hipGetLastError();
}

template <int T>
hipError_t launch_types(bgk_handle* h, const MomStep& st) {
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  if (h->mom_eqf) return f64 ? launch_t<T, double, true>(h, st) : launch_t<T, float, true>(h, st);
  return f64 ? launch_t<T, double, false>(h, st) : launch_t<T, float, false>(h, st);
}

}  // namespace

hipError_t launch_mom_stream(bgk_handle* h, const MomStep& st, int T) {
  if (T == 3) return launch_t<3, double, true>(h, st);
  return T == 2 ? launch_types<2>(h, st) : launch_types<1>(h, st);
}

}  // namespace bgk
