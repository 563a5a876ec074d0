// bgk_stream64.hip -- T FP64 population time steps in one launch, for the
// no-slip cavity.
//
// The walk of bgk_wave.h with whole populations: every node update takes its
// eighteen pulled populations and nine phi taps in the reference's order of
// operations (compiled with -ffp-contract=off), so results equal STEP_7's bit
// for bit, like bgk_fused.hip's, which does one step per launch.
//
// Level 0 loads the populations of a row already pulled (population k at
// column i - cx_k and row j - cy_k), so a strip of h rows takes h + 2 (T - 1)
// iterations.  A later level gets its row from
// the level below in registers and keeps, between two rows, the twelve
// populations the next two rows pull from it: lane shifts for the columns.
//
// Walls: as bgk_fused.hip describes them.  In a strip that touches one
// (strip_edge) a lane whose source is a ghost takes its own opposite
// population, or the thermal ghost's equilibrium, or the copied row, by
// selects; the loads stay the same for every lane.
//
// What bounds it: HBM (152 B per node and step, 304 with one step per launch);
// a row costs its wave 1330 VALU instructions at two waves per SIMD, 75% of
// its time at the memory rate.  Measured, us per step, against bgk_fused.hip:
// 4096^2 552 (893), 2048^2 152 (228), 1003 x 777 34.9 (38.5), 724^2 27.6
// (26.6), 512^2 18.1 (13.9): below 2^19 nodes one step per launch (stream64).
#include <algorithm>

#include "bgk_pop64.h"
#include "bgk_wave.h"

namespace bgk {
namespace {

using namespace wave;

struct Macro {
  double *rho, *u, *v, *T;
};

struct Args64 {
  Planes<double2> A, B;
  const double* pa;
  double* pb;
  const double* te_in;
  double* te_out;
  Macro m;
  Consts c;
  int nx, ny;
  int64_t pitch;
  WaveGrid g;
};

// A level's registers between two rows (levels 1 and up): of the row waiting
// for its northern neighbours, the populations pulled from the south (2, 5,
// 6) and from its own row (0, 1, 3); the southern share of the row after it;
// phi (west, centre, east) of both rows.
struct Pend {
  double sf[3], sg[3], cf[3], cg[3];
  double nf[3], ng[3];
  double ps[3], pc[3];
  // walls only: own f5, f6 and the northern g of the pending row, the wall
  // temperatures of the row and of the one south of it
  double o5, o6, gn[3], te_s, te_c;
};

// Populations of row j already pulled: population k of node (i - cx_k, j -
// cy_k).  off: byte offset of column i in a row of pairs.
__device__ __forceinline__ void load_pulled(const Args64& A, unsigned off, int j, Row& r) {
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const double2 v = at(A.A.row(k, (int64_t)(j - CY[k]) * A.pitch - CX[k]), off);
    r.f[k] = v.x;
    r.g[k] = v.y;
  }
}

// Thermal ghosts (BC_g.f90:9-31): replaces the populations a lane in column 1
// or Nx pulls from column 0 or Nx+1, in the rows below, beside and above its
// own (ghost rows: the clamped row).  ts, tc, tn: the east wall's temperature
// in those rows.  The ghost columns' velocities are the initial ones.
__device__ __forceinline__ void wall_g(const Args64& A, int i, bool has_w, bool has_e, double ts,
                                       double tc, double tn, double gp[9]) {
  const Consts& c = A.c;
  if (has_w) {
    const bool on = i == 1;
    gp[5] = on ? equilibrium_k(c, 5, c.tin, c.u0, c.v0) : gp[5];
    gp[1] = on ? equilibrium_k(c, 1, c.tin, c.u0, c.v0) : gp[1];
    gp[8] = on ? equilibrium_k(c, 8, c.tin, c.u0, c.v0) : gp[8];
  }
  if (has_e) {
    const bool on = i == A.nx;
    gp[6] = on ? equilibrium_k(c, 6, c.east_cold ? c.t_cold : ts, c.u0, c.v0) : gp[6];
    gp[3] = on ? equilibrium_k(c, 3, c.east_cold ? c.t_cold : tc, c.u0, c.v0) : gp[3];
    gp[7] = on ? equilibrium_k(c, 7, c.east_cold ? c.t_cold : tn, c.u0, c.v0) : gp[7];
  }
}

// Feed row j (1..Ny; Ny+1: nothing more comes) with the level below's output
// `in` (and its averaged T) to a level; gives the pulled row and taps of row
// j - 1.
template <bool EDGE>
__device__ __forceinline__ void feed(const Args64& A, Pend& L, const Done& in, double tav, int j,
                                     int i, bool has_w, bool has_e, double frozen6, double frozen7,
                                     double fp[9], double gp[9], double tap[9]) {
  const int nx = A.nx, ny = A.ny;
  fp[0] = L.cf[0];
  fp[1] = L.cf[1];
  fp[3] = L.cf[2];
  fp[2] = L.sf[0];
  fp[5] = L.sf[1];
  fp[6] = L.sf[2];
  gp[0] = L.cg[0];
  gp[1] = L.cg[1];
  gp[3] = L.cg[2];
  gp[2] = L.sg[0];
  gp[5] = L.sg[1];
  gp[6] = L.sg[2];
  tap[0] = L.pc[1];
  tap[1] = L.pc[2];
  tap[3] = L.pc[0];
  tap[4] = L.ps[1];
  tap[7] = L.ps[0];
  tap[8] = L.ps[2];
  const double te_s = L.te_s, te_c = L.te_c;
  double te_n = tav;
  if (EDGE && j > ny) {
    // row Ny pulls from row Ny+1: bounce-back, copied g and phi
    fp[4] = L.nf[0];
    fp[7] = i == nx ? frozen7 : L.o5;
    fp[8] = L.o6;
    gp[4] = L.gn[0];
    gp[7] = L.gn[1];
    gp[8] = L.gn[2];
    tap[2] = L.pc[1];
    tap[5] = L.pc[2];
    tap[6] = L.pc[0];
    te_n = te_c;
  } else {
    const double pw = from_west(in.phi), pe = from_east(in.phi);
    tap[2] = in.phi;
    tap[5] = pe;
    tap[6] = pw;
    fp[4] = in.f[4];
    fp[7] = from_east(in.f[7]);
    fp[8] = from_west(in.f[8]);
    gp[4] = in.g[4];
    gp[7] = from_east(in.g[7]);
    gp[8] = from_west(in.g[8]);
    double n4 = gp[4], n7 = gp[7], n8 = gp[8];
    if (EDGE) {
      if (has_w) fp[8] = i == 1 ? L.o6 : fp[8];
      if (has_e) fp[7] = i == nx ? L.o5 : fp[7];
    }
    // row j becomes the pending one
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      L.sf[s] = L.nf[s];
      L.sg[s] = L.ng[s];
      L.ps[s] = L.pc[s];
    }
    L.pc[0] = pw;
    L.pc[1] = in.phi;
    L.pc[2] = pe;
    L.cf[0] = in.f[0];
    L.cf[1] = from_west(in.f[1]);
    L.cf[2] = from_east(in.f[3]);
    L.cg[0] = in.g[0];
    L.cg[1] = from_west(in.g[1]);
    L.cg[2] = from_east(in.g[3]);
    L.nf[0] = in.f[2];
    L.nf[1] = from_west(in.f[5]);
    L.nf[2] = from_east(in.f[6]);
    L.ng[0] = in.g[2];
    L.ng[1] = from_west(in.g[5]);
    L.ng[2] = from_east(in.g[6]);
    if (EDGE) {
      L.te_s = L.te_c;
      L.te_c = tav;
      if (j == 1) {  // row 1 pulls from row 0
        L.sf[0] = in.f[4];
        L.sf[1] = in.f[7];
        L.sf[2] = i == nx ? frozen6 : in.f[8];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          L.sg[s] = L.ng[s];
          L.ps[s] = L.pc[s];
        }
        L.te_s = tav;
      }
      if (has_w) {
        if (j != 1) L.sf[1] = i == 1 ? in.f[7] : L.sf[1];
        L.cf[1] = i == 1 ? in.f[3] : L.cf[1];
      }
      if (has_e) {
        if (j != 1) L.sf[2] = i == nx ? in.f[8] : L.sf[2];
        L.cf[2] = i == nx ? in.f[1] : L.cf[2];
      }
      L.o5 = in.f[5];
      L.o6 = in.f[6];
      L.gn[0] = n4;
      L.gn[1] = n7;
      L.gn[2] = n8;
    }
  }
  if (EDGE) wall_g(A, i, has_w, has_e, te_s, te_c, te_n, gp);
}

// The halo as BC_f / BC_g leave it at the start of the call's last step, from
// the state that step starts from (row jc), and the fields after it.
__device__ __forceinline__ void halo(const Args64& A, int jc, int i, const Avg& a, double phi) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch, rj = (int64_t)jc * P, rn = (int64_t)(ny + 1) * P;
  const bool s_row = jc == 1, n_row = jc == ny;
  if (s_row) {
    A.m.rho[i] = a.rho;
    A.m.T[i] = a.T;
    A.m.u[i] = A.m.v[i] = 0.0;
    A.pb[i] = phi;
  }
  if (n_row) {
    A.m.rho[rn + i] = a.rho;
    A.m.T[rn + i] = a.T;
    A.m.u[rn + i] = A.m.v[rn + i] = 0.0;
    A.pb[rn + i] = phi;
  }
  if (i == 1) {
    A.m.T[rj] = A.c.tin;
    if (s_row) A.m.T[0] = A.c.tin;
    if (n_row) A.m.T[rn] = A.c.tin;
    if (s_row) A.pb[0] = A.pa[P];
    if (n_row) A.pb[rn] = A.pa[(int64_t)ny * P];
  }
  if (i == nx) {
    const double te = A.c.east_cold ? A.c.t_cold : a.T;
    A.m.T[rj + nx + 1] = te;
    if (s_row) A.m.T[nx + 1] = te;
    if (n_row) A.m.T[rn + nx + 1] = te;
    if (s_row) A.pb[nx + 1] = A.pa[P + nx + 1];
    if (n_row) A.pb[rn + nx + 1] = A.pa[(int64_t)ny * P + nx + 1];
  }
}

// The stores of a row: nine pair planes, phi, and the macroscopic fields after
// a call's last step.
template <bool FINAL>
struct Store64 {
  __device__ __forceinline__ static void put(const Args64& A, int jc, int j0, int j1, int i,
                                             bool own, bool own_phi, const Done& o) {
    const bool on = jc >= j0 && jc <= j1;
    const int64_t qr = (int64_t)jc * A.pitch;
    const int qa = on && own ? i : kPastRow;
#pragma unroll
    for (int k = 0; k < 9; ++k)
      buffer_put(row_buffer(A.B.row(k, qr), A.pitch), qa, make_double2(o.f[k], o.g[k]));
    buffer_put(row_buffer(A.pb + qr, A.pitch), on && own_phi ? i : kPastRow, o.phi);
    if (FINAL && on && own) {
      const Avg a = averaged(o);
      const int64_t qg = qr + i;
      A.m.rho[qg] = a.rho;
      A.m.T[qg] = a.T;
      A.m.u[qg] = a.u;
      A.m.v[qg] = a.v;
    }
  }
};

// A strip whose waves and levels meet no wall.
template <int T, bool STEP7, bool FINAL>
__device__ __forceinline__ void strip_mid(const Args64& A, int j0, int j1, int i) {
  const int lane = (int)threadIdx.x;
  const bool own = lane >= T && lane < kLanes - T;
  Pend L[T - 1];
#pragma unroll
  for (int t = 0; t < T - 1; ++t) L[t] = Pend{};
  const int ra = j0 - (T - 1), rb = j1 + (T - 1);  // rows of level 0
  const unsigned off = (unsigned)i * (unsigned)sizeof(double2);
  auto phi_row = [&](int j) { return at(A.pa + (int64_t)j * A.pitch, off / 2); };
  Row in;
  load_pulled(A, off, ra, in);
  const double ps = phi_row(ra - 1), pc = phi_row(ra);
  double pn = phi_row(ra + 1);
  __builtin_amdgcn_s_waitcnt(kWaitLoads);
  // taps of the rows below and beside (west, centre, east)
  double s3[3] = {from_west(ps), ps, from_east(ps)}, c3[3] = {from_west(pc), pc, from_east(pc)};
  for (int r = ra; r <= rb; ++r) {
    const double n3[3] = {from_west(pn), pn, from_east(pn)};
    const double tap0[9] = {c3[1], c3[2], n3[1], c3[0], s3[1], n3[2], n3[0], s3[0], s3[2]};
    Done o = node_step<STEP7>(A.c, in.f, in.g, tap0);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      s3[s] = c3[s];
      c3[s] = n3[s];
    }
    // the next row's loads, into the registers level 0 has done with
    __builtin_amdgcn_sched_barrier(0);
    load_pulled(A, off, r + 1, in);
    pn = phi_row(r + 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 1; t < T; ++t) {
      const int j = r - t + 1;  // row fed to level t
      if (j < j0 - (T - t)) continue;
      double fp[9], gp[9], tap[9];
      feed<false>(A, L[t - 1], o, 0.0, j, i, false, false, 0.0, 0.0, fp, gp, tap);
      o = node_step<STEP7>(A.c, fp, gp, tap);
    }
    Store64<FINAL>::put(A, r - (T - 1), j0, j1, i, own, own, o);
  }
}

// A strip that touches a wall.
template <int T, bool STEP7, bool FINAL>
__device__ __forceinline__ void strip_edge(const Args64& A, int j0, int j1, int i, bool has_w,
                                           bool has_e) {
  const int nx = A.nx, ny = A.ny;
  const int64_t P = A.pitch;
  const int lane = (int)threadIdx.x;
  const bool own = lane >= T && lane < kLanes - T && i <= nx;
  const bool ghost = i == 0 || i == nx + 1;
  const bool own_phi = own || (ghost && (i == 0 ? has_w : lane <= kLanes - T));
  unsigned offs[3];
  edge_offsets(i, nx, offs);
  const unsigned offp = (unsigned)min(max(i, 0), nx + 1) * (unsigned)sizeof(double);
  const __amdgpu_buffer_rsrc_t te_out = strip_buffer(A.te_out, ny + 2);
  const scalar_ptr te_in = as_scalar(A.te_in);
  const double frozen6 = A.A.row(6, nx + 1)->x;
  const double frozen7 = A.A.row(7, (int64_t)(ny + 1) * P + nx + 1)->x;
  Pend L[T - 1];
#pragma unroll
  for (int t = 0; t < T - 1; ++t) L[t] = Pend{};
  const int ra = max(1, j0 - (T - 1)), rb = j1 + (T - 1);  // rows of level 0
  auto phi_row = [&](int j) { return at(A.pa + (int64_t)min(max(j, 1), ny) * P, offp); };
  EdgeRow in;
  load_pulled_edge(A.A, P, ny, offs, ra, in);
  const double ps = phi_row(ra - 1), pc = phi_row(ra);
  double pn = phi_row(ra + 1);
  double te_s = te_in[max(ra - 1, 1)], te_c = te_in[ra], te_n = te_in[min(ra + 1, ny)];
  __builtin_amdgcn_s_waitcnt(kWaitLoads);
  double s3[3] = {from_west(ps), ps, from_east(ps)}, c3[3] = {from_west(pc), pc, from_east(pc)};
  for (int r = ra; r <= rb; ++r) {
    Done o{};
    double tav = 0.0;
    if (r <= ny) {
      const double n3[3] = {from_west(pn), pn, from_east(pn)};
      const double tap0[9] = {c3[1], c3[2], n3[1], c3[0], s3[1], n3[2], n3[0], s3[0], s3[2]};
      wall_f(nx, ny, i, r, frozen6, frozen7, in);
      wall_g(A, i, has_w, has_e, te_s, te_c, te_n, in.r.g);
      o = node_step<STEP7>(A.c, in.r.f, in.r.g, tap0);
      tav = averaged_T(o);
      if (ghost) o.phi = c3[1];
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        s3[s] = c3[s];
        c3[s] = n3[s];
      }
    }
    te_s = te_c;
    te_c = te_n;
    te_n = te_in[min(r + 2, ny)];
    __builtin_amdgcn_sched_barrier(0);
    load_pulled_edge(A.A, P, ny, offs, min(r + 1, ny), in);
    pn = phi_row(r + 2);
    __builtin_amdgcn_sched_barrier(0);
    static_assert(T == 2, "level 0 gives the state before the last step");
    if (FINAL && r >= j0 && r <= j1 && own) halo(A, r, i, averaged(o), o.phi);
#pragma unroll
    for (int t = 1; t < T; ++t) {
      const int j = r - t + 1;  // row fed to level t
      if (j < max(1, j0 - (T - t)) || j > ny + 1) continue;
      double fp[9], gp[9], tap[9];
      feed<true>(A, L[t - 1], o, tav, j, i, has_w, has_e, frozen6, frozen7, fp, gp, tap);
      o = node_step<STEP7>(A.c, fp, gp, tap);
      tav = averaged_T(o);
      if (ghost) o.phi = tap[0];
    }
    const int jc = r - (T - 1);  // row completed by the last level
    Store64<FINAL>::put(A, jc, j0, j1, i, own, own_phi, o);
    buffer_put(te_out, jc >= j0 && jc <= j1 && own && i == nx ? jc : kPastRow, tav);
  }
  if (own && i == nx) {
    if (j0 == 1) A.B.row(6, nx + 1)->x = frozen6;
    if (j1 == ny) A.B.row(7, (int64_t)(ny + 1) * P + nx + 1)->x = frozen7;
  }
}

template <int T, bool STEP7, bool FINAL>
__global__ __launch_bounds__(kLanes, 2) void k_stream64(Args64 A) {
  int seg, j0, j1;
  bool edge;
  if (!wave_tile(A.g, A.ny, &seg, &j0, &j1, &edge)) return;
  const int i0 = seg * (kLanes - 2 * T) + 1;
  const int i = i0 - T + (int)threadIdx.x;
  if (edge)
    strip_edge<T, STEP7, FINAL>(A, j0, j1, i, i0 - T <= 1, i0 - T + kLanes - 1 >= A.nx);
  else
    strip_mid<T, STEP7, FINAL>(A, j0, j1, i);
}

}  // namespace

// Below 2^19 nodes one step per launch is faster (it stays in the caches, and the
// few waves of this kernel are bound by the latency of their rows); a handle whose ghost velocities were
// uploaded takes the general kernel.
bool stream64(const bgk_handle* h) {
  if (!h->ghost_uv || h->recorded || h->pop_variant == 1) return false;
  return h->pop_variant > 1 || (int64_t)h->nx * h->ny >= (int64_t)1 << 19;
}

hipError_t launch_stream64(bgk_handle* h, bool write_all) {
  constexpr int T = kSteps64;
  Args64 a;
  const int ca = h->cur, cb = 1 - h->cur;
  a.A = planes_of<double2>(h->f[ca]);
  a.B = planes_of<double2>(h->f[cb]);
  a.pa = h->phi[h->pc];
  a.pb = h->phi[1 - h->pc];
  a.te_in = h->teast[h->te_cur];
  a.te_out = h->teast[1 - h->te_cur];
  a.m = Macro{h->rho, h->u, h->v, h->T};
  a.c = h->c;
  a.nx = h->nx;
  a.ny = h->ny;
  a.pitch = h->pitch;
  // strips of at most 16 rows; a row beside a wall counts 1.6 (measured at 1.2 /
  // 1.6 / 2.2, us per step: 1003 x 777 39 / 36 / 38, 2048^2 150 / 155 / 159,
  // 4096^2 560 / 571 / 577)
  a.g = make_wave_grid(h->nx, h->ny, kLanes - 2 * T, T, 2 * (T - 1), 1.6, 16, h->n_cu,
                       h->strip_rows);
  const dim3 grd((unsigned)a.g.nwg);
  const bool s7 = h->prm.rounding == BGK_ROUND_STEP7;
  if (s7 && write_all)
    hipLaunchKernelGGL((k_stream64<T, true, true>), grd, dim3(kLanes), 0, h->stream, a);
  else if (s7)
    hipLaunchKernelGGL((k_stream64<T, true, false>), grd, dim3(kLanes), 0, h->stream, a);
  else if (write_all)
    hipLaunchKernelGGL((k_stream64<T, false, true>), grd, dim3(kLanes), 0, h->stream, a);
  else
    hipLaunchKernelGGL((k_stream64<T, false, false>), grd, dim3(kLanes), 0, h->stream, a);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) {
    h->cur = cb;
    h->pc = 1 - h->pc;
    h->te_cur = 1 - h->te_cur;
  }
  return e;
}

}  // namespace bgk
