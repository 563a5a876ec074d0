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
// with omega_f = 1 181 (462, three steps per launch).  FP32 moments with three
// steps per launch: 230 (spills), with omega_f = 1 172.
#include <algorithm>

#include "bgk_level.h"

// Every multiply-add below is written out: contraction chosen by the compiler
// could differ between instantiations, and a step has to give the same bits
// whichever launch it is part of.
#pragma clang fp contract(off)

namespace bgk {
namespace {

using namespace level;

struct Macro {
  double *rho, *u, *v, *T;
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

// The initial phi of the ghost columns 0 and Nx+1, which no step changes
// (STEP_7/initialization.f90:15-26: liquid for i <= Nx/40).
constexpr double kPhiWest = 1.0, kPhiEast = -1.0;

// Stores of a strip's nodes through buffer descriptors: a lane that must not
// store gives an offset past the strip.  WIDE: a strip is one row, described from
// the wave's first column ib on (wide_rows).
template <typename R, bool EQF, int HOW, bool WIDE>
struct StoreMom {
  using V4 = typename Vec<R>::V4;
  using C = typename CType<R, EQF>::T;
  __amdgpu_buffer_rsrc_t a, b, c, phi;
  int ib;
  __device__ __forceinline__ StoreMom(const MomOut& out, double* pb, int64_t qs, int n, int first)
      : ib(first) {
    if constexpr (WIDE) {
      qs += ib;
      n = kLanes;
    }
    a = strip_buffer(out.a + qs, n);
    b = strip_buffer(static_cast<V4*>(out.b) + qs, n);
    c = strip_buffer(static_cast<C*>(out.c) + qs, n);
    phi = strip_buffer(pb + qs, n);
  }
  __device__ __forceinline__ void store(int q, bool on, bool on_phi, const Updated& o) const {
    if constexpr (WIDE) q -= ib;
    const int qa = on ? q : kPastStrip;
    buffer_put<HOW>(a, qa, make_double2(o.rho, o.dT));
    if constexpr (EQF) {
      buffer_put<HOW>(b, qa, make4<R>((R)o.u, (R)o.v, (R)o.pgxx, (R)o.pgyy));
      buffer_put<HOW>(c, qa, (R)o.pgxy);
    } else {
      buffer_put<HOW>(b, qa, make4<R>((R)o.u, (R)o.v, (R)o.pfxx, (R)o.pfyy));
      buffer_put<HOW>(c, qa, make4<R>((R)o.pfxy, (R)o.pgxx, (R)o.pgyy, (R)o.pgxy));
    }
    buffer_put<HOW>(phi, on_phi ? q : kPastStrip, o.phi);
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
  MomOut mid;  // kKeep, kKeepProbes
  double *phi_mid, *te_mid;
};

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
// plain loop 40 VGPRs).  The adjoint's runs keep some states: a launch of two
// steps that stores the one between them too costs less than two launches where
// HBM bounds them (2048^2, FP32 moments with omega_f = 1: 142 us, two launches 2 x
// 92; see keeps_between in bgk_adjoint.hip).
enum { kPlain, kProbes, kFinal, kKeep, kKeepProbes };

// One wave's strip.  EDGE: the wave or the strip touches a wall.  But for the
// last launch of a call the loop holds one path for its loads
// and stores: masked lanes and rows store out of the buffer's range, which
// the hardware drops, so that the wait for a row's loads (issued two rows
// ahead) never has to cover stores issued since.  With conditional stores the
// compiler's waits did, and a row cost 2.2 us of store latency on top.
template <int T, typename R, bool EQF, bool EDGE, int MODE, int HOW, bool WIDE>
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
  const StoreMom<R, EQF, HOW, WIDE> out(A.out, A.pb, qs, (j1 - j0 + 1) * (int)P, i0 - T);
  constexpr bool KEEP = MODE == kKeep || MODE == kKeepProbes;
  constexpr bool PROBES = MODE != kPlain && MODE != kKeep;

  // rows of the strip that hold a probe (the flags in column 0 of the probe
  // index plane; at most kMaxRows rows)
  uint64_t probes = 0;
  if (PROBES && A.probe_out)
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
  // full: levels that have completed a row of use; level `full` is only fed
  auto feed_row = [&](int r, Raw<R, EQF>& raw, int full) __attribute__((always_inline)) {
    NodeD nd = widen<R, EQF>(raw);
    __builtin_amdgcn_sched_barrier(0);
    raw = load_raw<R, EQF>(A.in, A.pa, (int64_t)min(r + 2, ny) * P + ic);
    const double te0 = te_row;
    if (EDGE) te_row = te_in[min(r + 1, ny)];
    Updated o;
    double tav = 0.0;  // averaged T of the row fed to the level
#pragma unroll
    for (int t = 0; t < T && t <= full; ++t) {
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
      double f[9], g[9];
      populations<!EQF>(nd.rho, nd.rho, nd.u, nd.v, nd.pfxx, nd.pfyy, nd.pfxy, f);
      populations<true>(nd.th, kTcrit + nd.th, nd.u, nd.v, nd.pgxx, nd.pgyy, nd.pgxy, g);
      feed<EDGE>(L[t], f, g, nd.phi, j, ny, i, nx, has_w, has_e, A.frozen6, A.frozen7, &S, &st,
                 &st2, &pc);
      if (t == full) return;
      o = update<R, EQF>(A.c, S, st, st2, pc);
      tav = kTcrit + (o.dT + o.dT2) * 0.5;
      const int jd = j - 1 - j0;  // (rows outside the strip are its neighbours')
      if (PROBES && jd >= 0 && jd < kMaxRows && ((probes >> jd) & 1) && own)
        record(A, t, j - 1, i, tav);
      if (MODE == kFinal && jd >= 0 && j - 1 <= j1 && own) finish<T>(A, t, j - 1, i, o, tav);
      if (KEEP && t == 0) {
        const bool mine = jd >= 0 && j - 1 <= j1;
        Updated k = o;
        if (EDGE && ghost) k.phi = i == 0 ? kPhiWest : kPhiEast;
        const StoreMom<R, EQF, HOW, WIDE> mid(A.mid, A.phi_mid, qs, (j1 - j0 + 1) * (int)P, i0 - T);
        mid.store(jd * (int)P + i, mine && own, mine && own_phi, k);
        if (EDGE)
          buffer_put(strip_buffer(A.te_mid, ny + 2), mine && own && i == nx ? j - 1 : kPastStrip,
                     tav);
      }
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
    const bool on = jc >= j0 && (!WIDE || jc <= j1);
    const int qo = (jc - j0) * (int)P + i;
    if (EDGE && ghost) o.phi = i == 0 ? kPhiWest : kPhiEast;
    out.store(qo, on && own, on && own_phi, o);
    if (EDGE) buffer_put(te_out, on && jc <= j1 && own && i == nx ? jc : kPastStrip, tav);
  };
  // The first two rows fed to a level complete none that anybody needs: leaving
  // the node update out there (away from the walls) spares 2T of T(h + 2T) updates
  // of a strip of h rows (us per step: FP32 moments 1003 x 777 15.2 -> 14.1, 2048^2
  // 56.0 -> 55.0, 4096^2 202.8 -> 202.8; with omega_f = 1 1003 x 777 13.4 -> 12.2,
  // 8192 x 1026 90.7 -> 89.1; FP64 1003 x 777 16.2 -> 15.6).  The instantiation
  // with the most registers loses by the longer code (FP64 moments with probes,
  // 512^2: 15.1 -> 16.2).
  int r = ra;
  if constexpr (!EDGE && MODE != kFinal && (!PROBES || EQF || sizeof(R) == sizeof(float))) {
#pragma unroll
    for (int t = 0; t < T; ++t, r += 2) {
      feed_row(r, raw0, t);
      feed_row(r + 1, raw1, t);
    }
  }
  for (; r <= rb; r += 2) {
    feed_row(r, raw0, T);
    feed_row(r + 1, raw1, T);
  }
}

template <int T, typename R, bool EQF, int MODE, int HOW, bool WIDE = false>
__global__ __launch_bounds__(kLanes, 2) void k_stream_mom(StreamArgs A) {
  int seg, j0, j1;
  bool edge;
  if (!wave_tile(A.g, A.ny, &seg, &j0, &j1, &edge)) return;
  const int i0 = seg * (kLanes - 2 * T) + 1;
  const int i = i0 - T + (int)threadIdx.x;
  if (edge)
    stream_strip<T, R, EQF, true, MODE, HOW, WIDE>(A, i0, j0, j1, i, i0 - T <= 1,
                                                   i0 - T + kLanes - 1 >= A.nx);
  else
    stream_strip<T, R, EQF, false, MODE, HOW, WIDE>(A, i0, j0, j1, i, false, false);
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
  a.mid = st.mid;
  a.phi_mid = st.phi_mid;
  a.te_mid = st.te_mid;
  // Strips of at most 64 rows with FP32 moments, 16 with FP64; a row beside a
  // wall counts 1.4 (measured at 1.2 / 1.6 / 2.2, us per step: 512^2 8.9 / 9.5
  // / 10.9, 1003 x 777 15.2 / 15.3 / 17.4, 4096^2 210 / 202 / 209; all strips
  // alike, walls in turn: 11.0, 18.5, 210).  FP64 moments at 4096^2 with at most
  // 16 / 32 rows: 323 / 334.
  constexpr int most = sizeof(R) == sizeof(float) ? 64 : 16;
  a.g = make_wave_grid(h->nx, h->ny, kLanes - 2 * T, T, 2 * T, 1.4, most, h->n_cu, h->strip_rows);
  const dim3 grd((unsigned)a.g.nwg);
  // Where the states read and written fit the 256 MB last-level cache but not the
  // L2s, the next launch finds more of what went through the caches than of what
  // went past them (us per step past / through: FP64 moments 724^2, 88 MB, 14.9 /
  // 13.2, 1003 x 777 19.9 / 16.1, 1200^2, 242 MB, 32.5 / 26.7, 1300^2, 284 MB, 36.8
  // / 37.0, 512^2, 44 MB, 8.9 / 9.2; FP32 moments 1448^2, 224 MB, 30.9 / 29.2, 860^2,
  // 79 MB, 15.1 / 15.2).
  const int64_t mb = (int64_t)h->nx * h->ny * 2 *
                     (int64_t)(sizeof(double2) + sizeof(typename Vec<R>::V4) +
                               sizeof(typename CType<R, EQF>::T) + sizeof(double)) >> 20;
  const bool cached = mb >= (sizeof(R) == sizeof(float) ? 96 : 64) && mb < 256;
  if constexpr (T == 1) {
    if (wide_rows(h)) {
      const auto k = st.write_all   ? k_stream_mom<T, R, EQF, kFinal, kNonTemporal, true>
                     : st.probe_out ? k_stream_mom<T, R, EQF, kProbes, kNonTemporal, true>
                                    : k_stream_mom<T, R, EQF, kPlain, kNonTemporal, true>;
      hipLaunchKernelGGL(k, grd, dim3(kLanes), 0, h->stream, a);
      return hipGetLastError();
    }
  }
  if constexpr (T == 2) {
    if (st.mid.a) {
      const auto k = st.probe_out ? k_stream_mom<T, R, EQF, kKeepProbes, kNonTemporal>
                                  : k_stream_mom<T, R, EQF, kKeep, kNonTemporal>;
      hipLaunchKernelGGL(k, grd, dim3(kLanes), 0, h->stream, a);
      return hipGetLastError();
    }
  }
  const auto k = st.write_all   ? k_stream_mom<T, R, EQF, kFinal, kNonTemporal>
                 : st.probe_out ? k_stream_mom<T, R, EQF, kProbes, kNonTemporal>
                 : cached       ? k_stream_mom<T, R, EQF, kPlain, kCached>
                                : k_stream_mom<T, R, EQF, kPlain, kNonTemporal>;
  hipLaunchKernelGGL(k, grd, dim3(kLanes), 0, h->stream, a);
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
