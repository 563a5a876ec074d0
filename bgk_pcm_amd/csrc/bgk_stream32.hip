// bgk_stream32.hip -- T time steps with FP32 population storage in one launch, and
// a step alone with the same arithmetic (k_step32), so that a run does not depend on
// how it is split.
//
// Storage and reference densities as in bgk_fused32.hip (f_k - w_k rho_ref and
// g_k - w_k T_crit in FP32); the walk and the node update are those of
// bgk_level.h.  After the regularised collision the eighteen populations of a
// node are a function of ten moments, so an update needs its pulled
// populations only through their sums and writes them out once: about 300
// FP64 VALU instructions per node and step, where pulling, colliding and
// encoding population by population takes 600.  Between the steps of a launch
// the populations are rounded to what the planes would hold.
//
// What bounds it: both HBM (80 B per node and step, 160 with one step per
// launch; 3.8 TB/s at 4096^2) and VALU issue at two waves per SIMD (65% of the
// time); the rest is the latency of 512-byte row pieces.  Measured in
// stream32.
#include <algorithm>

#include "bgk_level.h"

namespace bgk {
namespace {

using namespace level;

struct Macro {
  double *rho, *u, *v, *T;
};

struct Args32 {
  Planes<float2> A, B;
  const double* pa;
  double* pb;
  const double* te_in;
  double* te_out;
  Macro m;
  StepC c;
  const double* tab;  // reference densities: solid [0, Ny+2), liquid [Ny+2, ..)
  double tin, t_cold, u0, v0, rho0;
  int east_cold;
  int nx, ny;
  int64_t pitch;
  WaveGrid g;
};

// A row as loaded.
struct Raw32 {
  float2 p[9];
  double phi;
};

__device__ __forceinline__ void load_raw(const Args32& A, unsigned off, unsigned offp, int j,
                                         Raw32& r) {
  const int64_t row = (int64_t)j * A.pitch;
#pragma unroll
  for (int k = 0; k < 9; ++k) r.p[k] = at(A.A.row(k, row), off);
  r.phi = at(A.pa + row, offp);
}

// Populations as a launch hands them on: what the planes hold and what they
// stand for.
struct Stored {
  float fs[9], gs[9];
  double f[9], g[9];
};

// Reference density of a node of a row with solid and liquid densities rs, rl
// (bgk_fused32.hip's rho_ref).
__device__ __forceinline__ double ref_density(double rs, double rl, double phi) {
  return fma(fma(0.5, phi, 0.5), rl - rs, rs);
}

__device__ __forceinline__ void encode(const Updated& o, double rr, Stored& p) {
  populations<true>(o.rho, o.rho, o.u, o.v, o.pfxx, o.pfyy, o.pfxy, p.f);
  populations<true>(o.dT, kTcrit + o.dT, o.u, o.v, o.pgxx, o.pgyy, o.pgxy, p.g);
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    p.fs[k] = (float)fma(-kW[k], rr, p.f[k]);
    p.gs[k] = (float)p.g[k];
  }
}
__device__ __forceinline__ void decode(double rr, Stored& p) {
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    p.f[k] = fma(kW[k], rr, (double)p.fs[k]);
    p.g[k] = (double)p.gs[k];
  }
}

// Averaged moments of the stored state (STEP_7/moments.f90:11-25).
__device__ __forceinline__ double averaged_T(const Stored& p, const Updated& o) {
  double s = (double)p.gs[0];
#pragma unroll
  for (int k = 1; k < 9; ++k) s += (double)p.gs[k];
  return kTcrit + (s + o.dT2) * 0.5;
}
struct Avg {
  double rho, T, u, v;
};
__device__ __forceinline__ Avg averaged(const Stored& p, const Updated& o, double rr) {
  double a[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) a[k] = (double)p.fs[k];
  Avg r;
  r.rho = rr + (a[0] + a[1] + a[2] + a[3] + a[4] + a[5] + a[6] + a[7] + a[8]);
  r.T = averaged_T(p, o);
  r.u = ((a[1] - a[3] + a[5] - a[6] - a[7] + a[8]) / r.rho + o.u2) * 0.5;
  r.v = ((a[2] - a[4] + a[5] + a[6] - a[7] - a[8]) / r.rho + o.v2) * 0.5;
  return r;
}

// The halo as BC_f / BC_g leave it at the start of the call's last step, from
// the state that step starts from (row jc).
__device__ __forceinline__ void halo(const Args32& A, int jc, int i, double rho, double T,
                                     double phi) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch, rj = (int64_t)jc * P, rn = (int64_t)(ny + 1) * P;
  const bool s_row = jc == 1, n_row = jc == ny;
  if (s_row) {
    A.m.rho[i] = rho;
    A.m.T[i] = T;
    A.m.u[i] = A.m.v[i] = 0.0;
    A.pb[i] = phi;
  }
  if (n_row) {
    A.m.rho[rn + i] = rho;
    A.m.T[rn + i] = T;
    A.m.u[rn + i] = A.m.v[rn + i] = 0.0;
    A.pb[rn + i] = phi;
  }
  if (i == 1) {
    A.m.T[rj] = A.tin;
    if (s_row) A.m.T[0] = A.tin;
    if (n_row) A.m.T[rn] = A.tin;
    if (s_row) A.pb[0] = A.pa[P];
    if (n_row) A.pb[rn] = A.pa[(int64_t)ny * P];
  }
  if (i == nx) {
    const double te = A.east_cold ? A.t_cold : T;
    A.m.T[rj + nx + 1] = te;
    if (s_row) A.m.T[nx + 1] = te;
    if (n_row) A.m.T[rn + nx + 1] = te;
    if (s_row) A.pb[nx + 1] = A.pa[P + nx + 1];
    if (n_row) A.pb[rn + nx + 1] = A.pa[(int64_t)ny * P + nx + 1];
  }
}

// One wave's strip (see bgk_stream_mom.hip's stream_strip).
template <int T, bool EDGE, bool FINAL>
__device__ __forceinline__ void strip32(const Args32& A, int j0, int j1, int i, bool has_w,
                                        bool has_e) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch;
  const int lane = (int)threadIdx.x;
  const bool own = lane >= T && lane < kLanes - T && i <= nx;
  const bool ghost = EDGE && (i == 0 || i == nx + 1);
  const bool own_phi = own || (ghost && (i == 0 ? has_w : lane <= kLanes - T));
  const unsigned ic = (unsigned)(EDGE ? min(max(i, 0), nx + 1) : i);  // column loaded
  const unsigned off = ic * (unsigned)sizeof(float2), offp = ic * (unsigned)sizeof(double);
  const __amdgpu_buffer_rsrc_t te_out = strip_buffer(A.te_out, ny + 2);
  const scalar_ptr te_in = as_scalar(A.te_in), tab = as_scalar(A.tab);
  // the two corner ghosts no BC_f branch writes (stored against rho0)
  float fr6 = 0.0f, fr7 = 0.0f;
  if (EDGE) {
    fr6 = A.A.row(6, nx + 1)->x;
    fr7 = A.A.row(7, (int64_t)(ny + 1) * P + nx + 1)->x;
  }
  const double frozen6 = fma(kW[6], A.rho0, (double)fr6), frozen7 = fma(kW[7], A.rho0, (double)fr7);

  Level L[T];
#pragma unroll
  for (int t = 0; t < T; ++t) L[t] = Level{};
  const int ra = EDGE ? max(1, j0 - T) : j0 - T, rb = j1 + T;
  Raw32 raw;
  load_raw(A, off, offp, ra, raw);
  double te_row = EDGE ? te_in[ra] : 0.0;
  // reference densities of rows r, r - 1, .. r - T, the next row's loaded ahead
  double rs[T + 1], rl[T + 1];
#pragma unroll
  for (int d = 0; d <= T; ++d) {
    const int j = EDGE ? max(ra - d, 1) : ra - d;
    rs[d] = tab[j];
    rl[d] = tab[ny + 2 + j];
  }
  __builtin_amdgcn_s_waitcnt(kWaitLoads);
  // full: levels that have completed a row of use; level `full` is only fed
  auto feed_row = [&](int r, int full) __attribute__((always_inline)) {
    Stored p;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      p.fs[k] = raw.p[k].x;
      p.gs[k] = raw.p[k].y;
    }
    double phi = taken(raw.phi);
    decode(ref_density(rs[0], rl[0], phi), p);
    __builtin_amdgcn_sched_barrier(0);
    const int jn = min(r + 1, ny);
    load_raw(A, off, offp, jn, raw);
    const double rsn = tab[jn], rln = tab[ny + 2 + jn];
    const double te0 = te_row;
    if (EDGE) te_row = te_in[jn];
    Updated o;
    double tav = 0.0, rr = 0.0;
#pragma unroll
    for (int t = 0; t < T && t <= full; ++t) {
      const int j = r - t;  // row fed to level t
      if (j < j0 - (T - t) || (EDGE && (j < 1 || j > ny + 1))) continue;
      if (EDGE && j <= ny) {
        // ghost columns: no flow populations, thermal equilibria of the wall
        double te = t == 0 ? te0 : from_west(tav);
        if (A.east_cold) te = A.t_cold;
        const double tw = i == 0 ? A.tin : te;
        double gg[9];
        populations<false>(tw - kTcrit, tw, A.u0, A.v0, 0.0, 0.0, 0.0, gg);
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          p.f[k] = ghost ? 0.0 : p.f[k];
          p.g[k] = ghost ? gg[k] : p.g[k];
        }
      }
      PullSums S;
      double st, st2, pc;
      feed<EDGE>(L[t], p.f, p.g, phi, j, ny, i, nx, has_w, has_e, frozen6, frozen7, &S, &st, &st2,
                 &pc);
      if (t == full) break;
      o = update<double, false>(A.c, S, st, st2, pc);
      const int jc = j - 1;
      phi = o.phi;
      if (EDGE && ghost) phi = pc;
      rr = ref_density(rs[t + 1], rl[t + 1], phi);
      encode(o, rr, p);
      if (EDGE) tav = averaged_T(p, o);
      if (FINAL && t == T - 2 && jc >= j0 && jc <= j1 && own) {
        const Avg a = averaged(p, o, rr);
        halo(A, jc, i, a.rho, a.T, phi);
      }
      if (t < T - 1) decode(rr, p);
    }
    if (full == T) {
      const int jc = r - T;  // row completed by the last level
      const bool on = jc >= j0;
      const int64_t qr = (int64_t)jc * P;
      const int qa = on && jc <= j1 && own ? i : kPastRow;
#pragma unroll
      for (int k = 0; k < 9; ++k)
        buffer_put(row_buffer(A.B.row(k, qr), P), qa, make_float2(p.fs[k], p.gs[k]));
      buffer_put(row_buffer(A.pb + qr, P), on && jc <= j1 && own_phi ? i : kPastRow, phi);
      if (EDGE) buffer_put(te_out, on && jc <= j1 && own && i == nx ? jc : kPastRow, tav);
      if (FINAL && on && jc <= j1 && own) {
        const int64_t qg = (int64_t)jc * P + i;
        const Avg a = averaged(p, o, rr);
        A.m.rho[qg] = a.rho;
        A.m.T[qg] = a.T;
        A.m.u[qg] = a.u;
        A.m.v[qg] = a.v;
      }
    }
#pragma unroll
    for (int d = T; d > 0; --d) {
      rs[d] = rs[d - 1];
      rl[d] = rl[d - 1];
    }
    rs[0] = rsn;
    rl[0] = rln;
  };
  // (as in bgk_stream_mom.hip; us per step: 1003 x 777 25.7 -> 23.9, 1448^2 52.5 ->
  // 49.8, 2048^2 90.6 -> 90.4, 4096^2 341.7 -> 338.7)
  int r = ra;
  if constexpr (!EDGE && !FINAL) {
#pragma unroll
    for (int t = 0; t < T; ++t, r += 2) {
      feed_row(r, t);
      feed_row(r + 1, t);
    }
  }
  for (; r <= rb; ++r) feed_row(r, T);
  if (EDGE && own && i == nx) {
    if (j0 == 1) A.B.row(6, nx + 1)->x = fr6;
    if (j1 == ny) A.B.row(7, (int64_t)(ny + 1) * P + nx + 1)->x = fr7;
  }
}

template <int T, bool FINAL>
__global__ __launch_bounds__(kLanes, 2) void k_stream32(Args32 A) {
  int seg, j0, j1;
  bool edge;
  if (!wave_tile(A.g, A.ny, &seg, &j0, &j1, &edge)) return;
  const int i0 = seg * (kLanes - 2 * T) + 1;
  const int i = i0 - T + (int)threadIdx.x;
  if (edge)
    strip32<T, true, FINAL>(A, j0, j1, i, i0 - T <= 1, i0 - T + kLanes - 1 >= A.nx);
  else
    strip32<T, false, FINAL>(A, j0, j1, i, false, false);
}

// One step, one node per thread in the tiles of bgk_device.h, with the arithmetic
// of the walk: an odd step has the bits it has within a launch of two.  A wave with
// a boundary-adjacent node takes one path for all its lanes: ghost columns carry
// no flow populations and the wall's equilibria (at the ghost velocities of m.u
// and m.v), and every lane makes the same loads, from the nearest nodes inside.
// Bound by HBM; past the caches three waves per SIMD instead of the four that the
// registers allow disturb each other less (4096^2, us per call of one step: 586 /
// 559; cached, 727^2, 19.0 / 19.7).  Against k_fused32: 4096^2 578 -> 559, 2048^2
// 151 -> 133, 1003 x 777 30.2 -> 25.4.
template <bool CACHED>
__global__ __launch_bounds__(TILE_W) __attribute__((amdgpu_waves_per_eu(2, CACHED ? 4 : 3)))
void k_step32(Args32 A, TileGrid tg, int write_all) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch;
  int i, j;
  if (!tile_node(tg, Geom{nx, ny, P}, &i, &j)) return;
  const bool edge = i == 1 || i == nx || j == 1 || j == ny;
  const int row[3] = {max(j - 1, 1), j, min(j + 1, ny)};  // south, own, north
  const int64_t q = (int64_t)j * P + i;
  const double* const ps = A.pa + ((int64_t)row[0] * P + i);
  const double* const pc = A.pa + q;
  const double* const pn = A.pa + ((int64_t)row[2] * P + i);
  // taps C, E, N, W, S, NE, NW, SW, SE: of direction OPP[k] at population k's source
  const double tap[9] = {pc[0], pc[1], pn[0], pc[-1], ps[0], pn[1], pn[-1], ps[-1], ps[1]};
  const scalar_ptr tab = as_scalar(A.tab);
  double rs[3], rl[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    rs[d] = tab[row[d]];
    rl[d] = tab[ny + 2 + row[d]];
  }
  double f[9], g[9], own[9] = {}, rho_was = 0.0, T_was = 0.0;
  float fr6 = 0.0f, fr7 = 0.0f;
  PullSums S;
  if (!__any(edge)) {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const float2 v = load_pair<CACHED>(A.A.row(k, q - CX[k] - (int64_t)CY[k] * P));
      f[k] = fma(kW[k], ref_density(rs[1 - CY[k]], rl[1 - CY[k]], tap[OPP[k]]), (double)v.x);
      g[k] = (double)v.y;
    }
    S = pulled_sums<false>(f, g, f, i, j, nx, ny, 0.0, 0.0);
  } else {
    const double r1 = ref_density(rs[1], rl[1], tap[0]);
    fr6 = A.A.row(6, nx + 1)->x;
    fr7 = A.A.row(7, (int64_t)(ny + 1) * P + nx + 1)->x;
    rho_was = A.m.rho[q];
    T_was = A.m.T[q];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int64_t h = (int64_t)row[d] * P;
      const double t = A.east_cold ? A.t_cold : as_scalar(A.te_in)[row[d]];
      double gw[9], ge[9];
      populations<false>(A.tin - kTcrit, A.tin, A.m.u[h], A.m.v[h], 0.0, 0.0, 0.0, gw);
      populations<false>(t - kTcrit, t, A.m.u[h + nx + 1], A.m.v[h + nx + 1], 0.0, 0.0, 0.0, ge);
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        if (1 - CY[k] != d) continue;
        const int si = i - CX[k];
        const float2 v = *A.A.row(k, h + min(max(si, 1), nx));
        const double x = fma(kW[k], ref_density(rs[d], rl[d], tap[OPP[k]]), (double)v.x);
        f[k] = si >= 1 && si <= nx ? x : 0.0;
        g[k] = si < 1 ? gw[k] : si > nx ? ge[k] : (double)v.y;
        if (k > 0) own[k] = fma(kW[k], r1, (double)A.A.row(k, q)->x);
      }
    }
    S = pulled_sums<true>(f, g, own, i, j, nx, ny, fma(kW[6], A.rho0, (double)fr6),
                          fma(kW[7], A.rho0, (double)fr7));
  }
  double st, st2;
  tap_sums(tap, &st, &st2);
  const Updated o = update<double, false>(A.c, S, st, st2, tap[0]);
  const double rr = ref_density(rs[1], rl[1], o.phi);
  Stored p;
  encode(o, rr, p);
#pragma unroll
  for (int k = 0; k < 9; ++k) store_pair<CACHED>(A.B.row(k, q), p.fs[k], p.gs[k]);
  store_one<CACHED>(&A.pb[q], o.phi);
  if (!(edge || write_all)) return;
  const Avg a = averaged(p, o, rr);
  if (edge) {
    halo(A, j, i, rho_was, T_was, tap[0]);
    if (i == 1) A.pb[q - 1] = tap[3];
    if (i == nx) {
      A.pb[q + 1] = tap[1];
      A.te_out[j] = a.T;
      if (j == 1) A.B.row(6, nx + 1)->x = fr6;
      if (j == ny) A.B.row(7, (int64_t)(ny + 1) * P + nx + 1)->x = fr7;
    }
  }
  A.m.rho[q] = a.rho;
  A.m.T[q] = a.T;
  A.m.u[q] = a.u;
  A.m.v[q] = a.v;
}

Args32 args32(const bgk_handle* h) {
  Args32 a;
  const int ca = h->cur, cb = 1 - h->cur;
  a.A = planes_of<float2>(h->f32[ca]);
  a.B = planes_of<float2>(h->f32[cb]);
  a.pa = h->phi[h->pc];
  a.pb = h->phi[1 - h->pc];
  a.te_in = h->teast[h->te_cur];
  a.te_out = h->teast[1 - h->te_cur];
  a.m = Macro{h->rho, h->u, h->v, h->T};
  a.c = step_constants(h->c);
  a.tab = h->rref[h->rc];
  a.tin = h->c.tin;
  a.t_cold = h->c.t_cold;
  a.u0 = h->c.u0;
  a.v0 = h->c.v0;
  a.rho0 = h->c.rho0;
  a.east_cold = h->c.east_cold;
  a.nx = h->nx;
  a.ny = h->ny;
  a.pitch = h->pitch;
  return a;
}

void advanced(bgk_handle* h, int steps) {
  h->cur = 1 - h->cur;
  h->pc = 1 - h->pc;
  h->te_cur = 1 - h->te_cur;
  h->since_rebase += steps;
}

}  // namespace

// Measured, us per step, two steps per launch against k_fused32: 4096^2 354
// (472), 2048^2 90 (135), 1003 x 777 23.9 (27.9), 724^2 22.2 (23.1), 512^2
// 19.6 (14.6).  FP32 collision arithmetic is the general kernel's.
bool sums32(const bgk_handle* h) {
  if (h->prm.fp32_collision || h->pop_variant == 1) return false;
  return h->pop_variant > 1 || (int64_t)h->nx * h->ny >= (int64_t)1 << 19;
}
// (the ghost velocities are the initial ones in strip32)
bool stream32(const bgk_handle* h) { return sums32(h) && h->ghost_uv && !h->recorded; }

hipError_t launch_step32(bgk_handle* h, bool write_all) {
  const TileGrid tg = make_tile_grid(h->geom, 2 * (18 * (int)sizeof(float) + (int)sizeof(double)));
  const auto k = tg.cached ? k_step32<true> : k_step32<false>;
  hipLaunchKernelGGL(k, dim3((unsigned)(tg.per * NXCD)), dim3(TILE_W), 0, h->stream, args32(h), tg,
                     write_all ? 1 : 0);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) advanced(h, 1);
  return e;
}

hipError_t launch_stream32(bgk_handle* h, bool write_all) {
  constexpr int T = kSteps32;
  Args32 a = args32(h);
  // at most 16 rows per strip (measured at 8 / 16 / 24 / 48, us per step: 4096^2
  // 361 / 352 / 352 / 352, 2048^2 103 / 100 / 107 / 118)
  a.g = make_wave_grid(h->nx, h->ny, kLanes - 2 * T, T, 2 * T, 1.4, 16, h->n_cu, h->strip_rows);
  const dim3 grd((unsigned)a.g.nwg);
  if (write_all)
    hipLaunchKernelGGL((k_stream32<T, true>), grd, dim3(kLanes), 0, h->stream, a);
  else
    hipLaunchKernelGGL((k_stream32<T, false>), grd, dim3(kLanes), 0, h->stream, a);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) advanced(h, T);
  return e;
}

}  // namespace bgk
