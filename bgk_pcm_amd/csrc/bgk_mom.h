// bgk_mom.h -- moment form of the BGK_PCM step, shared by the moment-storage
// forward kernels (bgk_fused_mom.hip) and the adjoint (bgk_adjoint.hip).
//
// After the regularised collision (STEP_7/collision.f90:44-150, clean
// rounding) every population of a node is a function of ten numbers:
//   f_k = w_k rho (1 + P_k(u,v)) + coef_k H_k : Pf,   Pf = (1 - omega_f) Pi_f^neq
//   g_k = w_k T   (1 + P_k(u,v)) + coef_k H_k : Pg,   Pg = (1 - omega_g) Pi_g^neq
// with P_k the equilibrium polynomial minus its leading 1, H_k = c_k c_k -
// cs2 I and coef_k = w_k / (2 cs2^2).  A node stores
//   A = (rho, T - T_crit)                 double2
//   B = (u, v, Pf_xx, Pf_yy)              R4 (float4 or double4)
//   C = (Pf_xy, Pg_xx, Pg_yy, Pg_xy)      R4
// and, when omega_f = 1 (Pf = 0, "EQF"): B = (u, v, Pg_xx, Pg_yy), C = Pg_xy.
// The node update depends on its pulled populations only through ten
// moments (PullSums), which is what makes the adjoint compact.
#ifndef BGK_MOM_H
#define BGK_MOM_H

#include "bgk_internal.h"

namespace bgk {
namespace mom {

constexpr double kTcrit = 273.0;  // T_crit, STEP_7/phase_field.f90:16

// ---- storage traits: R = float (FP32 moments) or double (FP64 moments)
template <typename R>
struct Vec;
template <>
struct Vec<float> {
  using V4 = float4;
  typedef float nt4 __attribute__((ext_vector_type(4)));
};
template <>
struct Vec<double> {
  using V4 = double4;
  typedef double nt4 __attribute__((ext_vector_type(4)));
};
template <typename R, bool EQF>
struct CType {
  using T = typename Vec<R>::V4;
};
template <typename R>
struct CType<R, true> {
  using T = R;
};

template <typename R>
__device__ __forceinline__ typename Vec<R>::V4 make4(R x, R y, R z, R w) {
  typename Vec<R>::V4 v;
  v.x = x;
  v.y = y;
  v.z = z;
  v.w = w;
  return v;
}
template <typename R>
__device__ __forceinline__ typename Vec<R>::V4 nt_load4(const typename Vec<R>::V4* p) {
  const typename Vec<R>::nt4 v =
      __builtin_nontemporal_load(reinterpret_cast<const typename Vec<R>::nt4*>(p));
  return make4<R>(v.x, v.y, v.z, v.w);
}
template <typename R>
__device__ __forceinline__ void nt_store4(typename Vec<R>::V4* p, R x, R y, R z, R w) {
  typename Vec<R>::nt4 v;
  v.x = x;
  v.y = y;
  v.z = z;
  v.w = w;
  __builtin_nontemporal_store(v, reinterpret_cast<typename Vec<R>::nt4*>(p));
}

// Planes of one moment state (typed by the kernels through R, EQF).
struct MomIn {
  const double2* a;
  const void* b;
  const void* c;
};
struct MomOut {
  double2* a;
  void* b;
  void* c;
};

template <typename R, bool EQF>
struct Node {
  double2 a;                       // rho, T - T_crit
  typename Vec<R>::V4 b;           // u, v, Pf_xx, Pf_yy  (EQF: u, v, Pg_xx, Pg_yy)
  typename CType<R, EQF>::T c;     // Pf_xy, Pg_xx, Pg_yy, Pg_xy  (EQF: Pg_xy)
  double phi;
};

template <typename R, bool EQF>
__device__ __forceinline__ typename Vec<R>::V4 b_at(const void* b, int64_t q) {
  return static_cast<const typename Vec<R>::V4*>(b)[q];
}
template <typename R, bool EQF>
__device__ __forceinline__ typename CType<R, EQF>::T c_at(const void* c, int64_t q) {
  return static_cast<const typename CType<R, EQF>::T*>(c)[q];
}
template <typename R, bool EQF>
__device__ __forceinline__ typename CType<R, EQF>::T c_stream(const void* c, int64_t q) {
  if constexpr (EQF)
    return __builtin_nontemporal_load(static_cast<const R*>(c) + q);
  else
    return nt_load4<R>(static_cast<const typename Vec<R>::V4*>(c) + q);
}

// Moments of the pulled populations of a node: zeroth, first and second
// moments of f, and of gd = g - w*T_crit (its first moment is not needed).
// A: the arithmetic type, double but for the adjoint of the FP32 moment step,
// which evaluates its Jacobians in FP32.
template <typename A>
struct PullSumsT {
  A rho, jx, jy, fxx, fyy, fxy;
  A dT, gxx, gyy, gxy;
};
using PullSums = PullSumsT<double>;

// The node update in moment form: momentsPre (STEP_7/momentsPre.f90:8-21),
// phase field (phase_field.f90:24-52, reaction rates in closed form),
// latent heat and forces (forces.f90:18-26), and the collision's
// non-equilibrium moments (collision.f90:44-92: for the second-order D2Q9
// equilibrium sum_k H_k feq_k = rho u u).  Everything the adjoint needs is
// kept in the struct.
//
// Phase field: 0.5 (1 -/+ tanh x) = 1 / (1 + exp(+/-2x)), x = (T - 273) /
// T_width: one exp and one division instead of the branchy glibc-exact
// tanh of the FP64 population kernels, which this clean-rounding path need
// not reproduce bit for bit (the rates' absolute error stays a few ulp of
// 1).  No branch inside one phase: there the reaction terms are multiplied
// by exact zeros anyway, and a branch splits the node's code (~70 more
// registers).
//
// Extensions: the phase field's T_crit (273 + crit_shift off) and a
// buoyancy reference t_ref (0: STEP_7's absolute T; both exact when off).
// Off when k_ratio == 1: solid/liquid conductivity ratio through
// a phase-dependent thermal relaxation, alpha(phi) = alpha_l (fl + k_ratio
// (1 - fl)), fl = (1 + phi)/2 the liquid fraction, tau_g = 1/2 + alpha/cs2.
template <typename A>
struct CoreT {
  A rho, irho, u2, v2, dT2;     // momentsPre
  A kp_sum, km_sum, rm, phi, pc;  // phase field
  A dT, T;                        // after latent heat
  A u, v;                         // after forces
  A omega_g;                      // thermal relaxation rate used
  A qfxx, qfyy, qfxy;             // Pi_f^neq
  A qgxx, qgyy, qgxy;             // Pi_g^neq
};

// 1/d as the hardware estimate refined by two Newton steps (r <- r + r (1 -
// d r), each doubling the correct bits): within an ulp or two of the IEEE
// quotient and about ten instructions cheaper.  The moment path uses it for
// its per-node reciprocals (the two divisions of the conductivity ratio's
// rate cost 1.2% of the moment step at 4096^2); the FP64 population kernels
// keep IEEE division to stay bit-exact.
__device__ __forceinline__ double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  r = fma(r, fma(-d, r, 1.0), r);
  return r;
}
// FP32: the hardware estimate and one Newton step
__device__ __forceinline__ float rcp_nr(float d) {
  float r = __builtin_amdgcn_rcpf(d);
  return fmaf(r, fmaf(-d, r, 1.0f), r);
}

// FP32 copies of the constants the node update and its adjoint read, for
// the FP32-arithmetic adjoint (filled from Consts on the host, so that no
// kernel converts them).
struct ConstsF {
  float crit_shift, two_over_tw, dt_st, grav, beta, t_ref, inv_omega_f, omega_f, omega_g,
      alpha_l, k_ratio, inv_stefan;
};
inline ConstsF consts_f(const Consts& c) {
  return ConstsF{(float)c.crit_shift, (float)c.two_over_tw, (float)c.dt_st,   (float)c.grav,
                 (float)c.beta,       (float)c.t_ref,       (float)c.inv_omega_f,
                 (float)c.omega_f,    (float)c.omega_g,     (float)c.alpha_l,
                 (float)c.k_ratio,    (float)c.inv_stefan};
}

// C: Consts, or ConstsF (the same fields in FP32) for FP32 arithmetic.
template <typename A, typename C>
__device__ __forceinline__ A omega_g_of(const C& c, A phi) {
  if (c.k_ratio == 1.0) return (A)c.omega_g;
  const A fl = A(0.5) * (A(1) + phi);
  const A alpha = (A)c.alpha_l * (fl + (A)c.k_ratio * (A(1) - fl));
  return rcp_nr(A(0.5) + alpha * A(3));  // 1/(1/2 + alpha/cs2)
}

// st, st2: sums of the nine phi_prec taps and of their squares, pc the centre tap.
template <typename A, typename C>
__device__ __forceinline__ CoreT<A> core_from_sums(const C& c, const PullSumsT<A>& S, A st, A st2,
                                                   A pc) {
  CoreT<A> o;
  o.rho = S.rho;
  o.dT2 = S.dT;
  o.irho = rcp_nr(o.rho);
  o.u2 = S.jx * o.irho;
  o.v2 = S.jy * o.irho;

  // sum_m ((1 +/- t_m)/2)^2 = (9 +/- 2 sum t + sum t^2) / 4
  const A kp = A(0.25) * ((A(9) + st2) + A(2) * st);
  const A km = A(0.25) * ((A(9) + st2) - A(2) * st);
  o.kp_sum = kp;
  o.km_sum = km;
  o.pc = pc;
  // Both reaction terms vanish exactly when kp = 0 (all taps -1) or pc = 1,
  // and km = 0 (all taps +1) or pc = -1: phi = pc whatever the rates, which
  // are then not evaluated (rm = 1/2 keeps every product below finite; the
  // adjoint multiplies its rate terms by the same exact zeros).
  const bool react = !((kp == A(0) || o.pc == A(1)) && (km == A(0) || o.pc == A(-1)));
  o.rm = A(0.5);
  if (react) o.rm = A(1) / (A(1) + exp((o.dT2 + (A)c.crit_shift) * (A)c.two_over_tw));
  const A rp = A(1) - o.rm;
  const A kpr = (kp * A(0.125)) * rp;
  const A kmr = (km * A(0.125)) * o.rm;
  o.phi = o.pc + (A(0.5) * kpr * (A(1) - o.pc) - A(0.5) * kmr * (A(1) + o.pc));

  o.dT = o.dT2 - ((A)c.dt_st * (o.phi - o.pc) * A(0.5));
  o.T = A(kTcrit) + o.dT;
  A fy = o.rho * (A)c.grav * (A)c.beta * (o.T - (A)c.t_ref) * (A(1) + o.phi * A(0.5));
  const A fx = -(o.u2 * (A(1) - o.phi) * A(0.5));
  fy = fy - o.v2 * (A(1) - o.phi) * A(0.5);
  const A s = o.irho * (A)c.inv_omega_f;
  o.u = o.u2 + fx * s;
  o.v = o.v2 + fy * s;

  o.omega_g = omega_g_of<A, C>(c, o.phi);
  o.qfxx = S.fxx - A(kCs2) * o.rho - o.rho * o.u * o.u;
  o.qfyy = S.fyy - A(kCs2) * o.rho - o.rho * o.v * o.v;
  o.qfxy = S.fxy - o.rho * o.u * o.v;
  o.qgxx = S.gxx - A(kCs2) * o.dT2 - o.T * o.u * o.u;
  o.qgyy = S.gyy - A(kCs2) * o.dT2 - o.T * o.v * o.v;
  o.qgxy = S.gxy - o.T * o.u * o.v;
  return o;
}

// One launch of T moment-storage steps: state and phi in and out, the
// east-wall temperature column before and after, an optional probe record (T
// averaged as moments.f90 at the nodes whose probe_idx is >= 0, after step t
// of the launch to probe_out[t*probe_np + probe_idx]; probe_idx in column 0 of
// a row is >= 0 when the row holds a probe).  write_all: the macroscopic
// fields of every node and the halo.  One-step launches of the ring kernel
// write those of the boundary nodes in any case, and record no probes: the
// adjoint's runs keep to the streaming kernel, whose steps have the same bits
// however a run is split.
struct MomStep {
  bool ring = false;  // (one step) through the ring kernel
  MomIn in;
  MomOut out;
  const double* pa;
  double* pb;
  const double* te_in;
  double* te_out;
  bool write_all;
  const int* probe_idx;
  double* probe_out;
  int probe_np;
  // two steps, not the last of a call: the state between them, where it is
  // kept (mid.a null: it is not)
  MomOut mid{};
  double* phi_mid = nullptr;
  double* te_mid = nullptr;
};

}  // namespace mom

// T steps in one launch (bgk_fused_mom.hip; T at most mom_next_steps), and the
// streaming kernel's share of them (bgk_stream_mom.hip)
hipError_t launch_mom_steps(bgk_handle* h, const mom::MomStep& st, int T);
hipError_t launch_mom_stream(bgk_handle* h, const mom::MomStep& st, int T);
int mom_next_steps(const bgk_handle* h, int left, bool adjoint = false);
// Whether a launch has to write the macroscopic fields, `left` steps of the call
// after it: the last one; and the one before a last launch of one step, which takes
// the halo from them, unless that is a ring launch after another one (these keep
// the boundary nodes current).
inline bool mom_write_all(int left, bool ring) { return left == 0 || (left == 1 && !ring); }
int mom_most_steps(const bgk_handle* h, bool adjoint = false);
}  // namespace bgk

#endif  // BGK_MOM_H
