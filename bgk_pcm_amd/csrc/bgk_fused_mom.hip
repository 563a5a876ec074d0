// bgk_fused_mom.hip -- moment storage: the choice of kernel and of the steps
// per launch, the initialization, and the ring kernel, one step per launch
// through LDS, which large lattices take for a step alone (see
// ring_step; every other launch is bgk_stream_mom.hip's).
//
// The node state is the ten moments of bgk_mom.h (rho, T - T_crit in FP64;
// u, v and the scaled non-equilibrium second moments in R = float or
// double), 48 bytes per node with FP32 R (36 with omega_f = 1) instead of
// 144 for FP32 populations, and the pull rebuilds population k of the
// upstream node from its moments.  rho and T stay FP64: the rounding of rho
// (not of u) is what drives the velocity error of FP32 storage, since a
// neighbour's density error enters the momentum balance through
// sum_k c_k w_k rho(x - c_k).  u, v and the non-equilibrium moments carry
// their own relative precision.
//
// Tiling: a workgroup owns W columns and a strip of consecutive rows, and
// walks the strip row by row.  Row r + 1 is fetched from HBM while row r, in
// LDS, is fed to the sums of the rows below, beside and above it (feed_three in
// bgk_level.h; the LDS holds two rows, for one barrier a row), so every node's
// moments and phi are read from HBM once per step (plus the strip's two
// boundary rows and the two halo columns).  The boundary-adjacent nodes run in
// extra workgroups of the same launch with BC_f (no-slip) and BC_g folded in as
// in bgk_fused.hip: ghost rows of g and phi are the clamped rows, own opposite
// populations for bounce-back, the two frozen corner ghosts as constants.  The
// operations and their order are the streaming kernel's, so a step has the same
// bits in either (4096^2, us per step: 364, and 286 with omega_f = 1; rebuilding
// nine upstream nodes' populations at every node, in an order of its own, 362
// and 290).
//
// Arithmetic is FP64 throughout.  STEP_7's FP32 temporaries (ft, gt) cannot
// be represented by moments, so this path follows the clean rounding policy;
// beta follows bgk_params.rounding as everywhere.
#include <algorithm>

#include "bgk_level.h"
#include "bgk_strip.h"

namespace bgk {
namespace {

using namespace level;

constexpr int TX = 64, TY = 4;  // block of the initialization kernel

struct Macro {
  double *rho, *u, *v, *T;
};

// LDS ring of two rows of W + 2 nodes (W columns and the two halo columns).
template <int W, typename R, bool EQF>
struct Ring {
  double2 a[2][W + 2];
  typename Vec<R>::V4 b[2][W + 2];
  typename CType<R, EQF>::T c[2][W + 2];
  double phi[2][W + 2];
};

template <typename R, bool EQF>
__device__ __forceinline__ Node<R, EQF> load_node(const MomIn& in, const double* __restrict__ pa,
                                                  const Geom& gm, int ic, int jr) {
  Node<R, EQF> n;
  n.a = make_double2(0.0, 0.0);
  n.b = make4<R>(R(0), R(0), R(0), R(0));
  n.c = typename CType<R, EQF>::T{};
  n.phi = 0.0;
  const int64_t q = (int64_t)jr * gm.pitch + ic;
  if (ic >= 1 && ic <= gm.nx) {
    n.a = stream_load(in.a + q);
    n.b = nt_load4<R>(static_cast<const typename Vec<R>::V4*>(in.b) + q);
    n.c = c_stream<R, EQF>(in.c, q);
  }
  if (ic >= 0 && ic <= gm.nx + 1) n.phi = pa[q];
  return n;
}

template <int W, typename R, bool EQF>
__device__ __forceinline__ void put(Ring<W, R, EQF>& L, int r, int s, const Node<R, EQF>& n) {
  L.a[r][s] = n.a;
  L.b[r][s] = n.b;
  L.c[r][s] = n.c;
  L.phi[r][s] = n.phi;
}

template <typename R, bool EQF>
__device__ __forceinline__ Pops populations_of(const double2& a, const typename Vec<R>::V4& b,
                                               const typename CType<R, EQF>::T& c) {
  const double u = (double)b.x, v = (double)b.y;
  Pops p;
  if constexpr (EQF) {
    populations<false>(a.x, a.x, u, v, 0.0, 0.0, 0.0, p.f);
    populations<true>(a.y, kTcrit + a.y, u, v, (double)b.z, (double)b.w, (double)c, p.g);
  } else {
    populations<true>(a.x, a.x, u, v, (double)b.z, (double)b.w, (double)c.x, p.f);
    populations<true>(a.y, kTcrit + a.y, u, v, (double)c.y, (double)c.z, (double)c.w, p.g);
  }
  return p;
}

// Node update from its pulled moments and phi_prec sums; stores the node's
// moments and phi.
template <typename R, bool EQF>
__device__ __forceinline__ Updated update_node(const StepC& c, const PullSums& S, double st,
                                               double st2, double pc, const MomOut& out,
                                               double* __restrict__ pb, int64_t q) {
  const Updated o = update<R, EQF>(c, S, st, st2, pc);
  using V4 = typename Vec<R>::V4;
  stream_store(out.a + q, o.rho, o.dT);
  if constexpr (EQF) {
    nt_store4<R>(static_cast<V4*>(out.b) + q, (R)o.u, (R)o.v, (R)o.pgxx, (R)o.pgyy);
    __builtin_nontemporal_store((R)o.pgxy, static_cast<R*>(out.c) + q);
  } else {
    nt_store4<R>(static_cast<V4*>(out.b) + q, (R)o.u, (R)o.v, (R)o.pfxx, (R)o.pfyy);
    nt_store4<R>(static_cast<V4*>(out.c) + q, (R)o.pfxy, (R)o.pgxx, (R)o.pgyy, (R)o.pgxy);
  }
  stream_store(&pb[q], o.phi);
  return o;
}

// The averaged moments after the step (STEP_7/moments.f90:11-25).
__device__ __forceinline__ double averaged_T(const Updated& o) {
  return kTcrit + (o.dT + o.dT2) * 0.5;
}
__device__ __forceinline__ void put_macro(const Macro& m, int64_t q, const Updated& o) {
  m.rho[q] = o.rho;
  m.T[q] = averaged_T(o);
  m.u[q] = (o.u + o.u2) * 0.5;
  m.v[q] = (o.v + o.v2) * 0.5;
}

// Interior nodes (1 < i < Nx, 1 < j < Ny) by row strips, W columns per workgroup.
// A thread feeds its column's node and the two beside it, row after row, to the
// sums of bgk_level.h, so that a row is needed in LDS only while it is fed.
// Workgroups from sg.nmain on serve the boundary-adjacent nodes
// (mom_edge_nodes).
template <int W, typename R, bool EQF>
__device__ __forceinline__ void mom_interior(const MomIn& in, const MomOut& out,
                                             const double* __restrict__ pa,
                                             double* __restrict__ pb, const Macro& m,
                                             const StepC& c, const Geom& gm, const StripGrid& sg,
                                             int write_all) {
  __shared__ Ring<W, R, EQF> L;
  const int nx = gm.nx, ny = gm.ny;
  int strip, seg;
  if (!strip_of(sg, (int)blockIdx.x, &strip, &seg)) return;  // whole workgroup
  const int j0 = strip * sg.rows + 1;
  const int j1 = min(j0 + sg.rows - 1, ny);
  const int t = (int)threadIdx.x;
  const int i0 = seg * W + 1;  // column of slot 1
  const int i = i0 + t;        // this thread's column, slot t + 1
  // threads 0 and 1 also fetch the halo columns i0 - 1 (slot 0) and i0 + W (slot W + 1)
  const int hcol = (t == 0) ? i0 - 1 : i0 + W;
  const int hslot = (t == 0) ? 0 : W + 1;
  auto clampj = [ny](int jj) { return jj < 1 ? 1 : (jj > ny ? ny : jj); };
  const bool col_in = (i > 1 && i < nx);
  Level S = Level{};
  Node<R, EQF> nn = load_node<R, EQF>(in, pa, gm, i, clampj(j0 - 1)), nh;
  if (t < 2) nh = load_node<R, EQF>(in, pa, gm, hcol, clampj(j0 - 1));
  for (int r = j0 - 1; r <= j1 + 1; ++r) {  // row fed
    const int b = r & 1;
    put(L, b, t + 1, nn);
    if (t < 2) put(L, b, hslot, nh);
    __syncthreads();  // (row r + 1 overwrites row r - 1, which nobody reads any more)
    if (r <= j1) {
      nn = load_node<R, EQF>(in, pa, gm, i, clampj(r + 1));
      if (t < 2) nh = load_node<R, EQF>(in, pa, gm, hcol, clampj(r + 1));
    }
    const Pops w = populations_of<R, EQF>(L.a[b][t], L.b[b][t], L.c[b][t]);
    const Pops c0 = populations_of<R, EQF>(L.a[b][t + 1], L.b[b][t + 1], L.c[b][t + 1]);
    const Pops e = populations_of<R, EQF>(L.a[b][t + 2], L.b[b][t + 2], L.c[b][t + 2]);
    PullSums P;
    double st, st2, pc;
    feed_three(S, w, c0, e, L.phi[b][t], L.phi[b][t + 1], L.phi[b][t + 2], &P, &st, &st2, &pc);
    const int j = r - 1;  // row completed
    if (j >= j0 && col_in && j > 1 && j < ny) {
      const int64_t q = (int64_t)j * gm.pitch + i;
      const Updated o = update_node<R, EQF>(c, P, st, st2, pc, out, pb, q);
      if (write_all) put_macro(m, q, o);
    }
  }
}

// The boundary-adjacent nodes, one per thread, with BC_f type 4 and BC_g
// (STEP_7/BC_f.f90:62-68,101-107,125-136,181-192; BC_g.f90:9-64) folded into
// the pulls: bounce-back of the node's own opposite populations, the two
// frozen corner ghosts, W/E thermal ghosts at Tin and at the previous
// step's averaged T(Nx, j), N/S ghost rows of g and phi equal to rows Ny / 1;
// then the halo bookkeeping of the macroscopic fields.
template <typename R, bool EQF>
__device__ __forceinline__ void mom_edge_nodes(const MomIn& in, const MomOut& out,
                                               const double* __restrict__ pa,
                                               double* __restrict__ pb,
                                               const double* __restrict__ te_in,
                                               double* __restrict__ te_out, const Macro& m,
                                               const Consts& c, const StepC& sc, const Geom& gm,
                                               int e) {
  const int nx = gm.nx, ny = gm.ny;
  const int64_t P = gm.pitch;
  int i, j;
  if (!edge_node(e, nx, ny, &i, &j)) return;
  const int64_t q = (int64_t)j * P + i;
  const Pops own = populations_of<R, EQF>(in.a[q], b_at<R, EQF>(in.b, q), c_at<R, EQF>(in.c, q));
  double f[9], g[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int si = i - CX[k], sj = j - CY[k];
    const int sjc = sj < 1 ? 1 : (sj > ny ? ny : sj);
    if (si >= 1 && si <= nx) {
      const int64_t h = (int64_t)sjc * P + si;
      const Pops p =
          populations_of<R, EQF>(in.a[h], b_at<R, EQF>(in.b, h), c_at<R, EQF>(in.c, h));
      f[k] = p.f[k];
      g[k] = p.g[k];
    } else {  // no flow populations, the wall's T and velocity
      const double th = (si == 0 ? c.tin : east_T(c, te_in, sjc)) - kTcrit;
      double p[9];
      populations<true>(th, kTcrit + th, c.u0, c.v0, 0.0, 0.0, 0.0, p);
      f[k] = 0.0;
      g[k] = p[k];
    }
  }
  const int64_t rn = (int64_t)(j < ny ? j + 1 : ny) * P;
  const int64_t rs = (int64_t)(j > 1 ? j - 1 : 1) * P;
  const int64_t r0 = (int64_t)j * P;
  const double tap[9] = {pa[q],          pa[r0 + i + 1], pa[rn + i],     pa[r0 + i - 1], pa[rs + i],
                         pa[rn + i + 1], pa[rn + i - 1], pa[rs + i - 1], pa[rs + i + 1]};
  const PullSums S = pulled_sums<true>(f, g, own.f, i, j, nx, ny, c.frozen6, c.frozen7);
  double st, st2;
  tap_sums(tap, &st, &st2);
  const Updated o = update_node<R, EQF>(sc, S, st, st2, tap[0], out, pb, q);

  // ---- halo bookkeeping: BC_f N/S rows (rho copied, u = v = 0), BC_g
  // T and phi ghosts, the east column's averaged T for the next step
  const bool w_edge = (i == 1), e_edge = (i == nx), s_edge = (j == 1), n_edge = (j == ny);
  if (s_edge) {
    m.rho[i] = m.rho[q];
    m.T[i] = m.T[q];
    m.u[i] = 0.0;
    m.v[i] = 0.0;
    pb[i] = pa[q];
  }
  if (n_edge) {
    const int64_t h = (int64_t)(ny + 1) * P + i;
    m.rho[h] = m.rho[q];
    m.T[h] = m.T[q];
    m.u[h] = 0.0;
    m.v[h] = 0.0;
    pb[h] = pa[q];
  }
  if (w_edge) {
    m.T[r0] = c.tin;
    pb[r0] = pa[r0];
    if (s_edge) {
      m.T[0] = c.tin;
      pb[0] = pa[P];
    }
    if (n_edge) {
      const int64_t h = (int64_t)(ny + 1) * P;
      m.T[h] = c.tin;
      pb[h] = pa[(int64_t)ny * P];
    }
  }
  if (e_edge) {
    const int64_t h = r0 + nx + 1;
    m.T[h] = east_T(c, te_in, j);
    pb[h] = pa[h];
    te_out[j] = averaged_T(o);
    if (s_edge) {
      m.T[nx + 1] = east_T(c, te_in, 1);
      pb[nx + 1] = pa[P + nx + 1];
    }
    if (n_edge) {
      const int64_t hn = (int64_t)(ny + 1) * P + nx + 1;
      m.T[hn] = east_T(c, te_in, ny);
      pb[hn] = pa[(int64_t)ny * P + nx + 1];
    }
  }
  put_macro(m, q, o);
}

template <int W, typename R, bool EQF>
__global__ __launch_bounds__(W) void k_fused_mom(
    MomIn in, MomOut out, const double* __restrict__ pa, double* __restrict__ pb,
    const double* __restrict__ te_in, double* __restrict__ te_out, Macro m, Consts c, StepC sc,
    Geom gm, StripGrid sg, int write_all) {
  if ((int)blockIdx.x >= sg.nmain) {
    const int e = ((int)blockIdx.x - sg.nmain) * W + (int)threadIdx.x;
    mom_edge_nodes<R, EQF>(in, out, pa, pb, te_in, te_out, m, c, sc, gm, e);
    return;
  }
  mom_interior<W, R, EQF>(in, out, pa, pb, m, sc, gm, sg, write_all);
}

// STEP_7/initialization.f90:15-152 for a moment handle: the initial
// populations are equilibria, i.e. moments with zero non-equilibrium part.
template <typename R, bool EQF>
__global__ void k_initialization_mom(MomOut st, Macro m, double* phi, double* phip, Consts c,
                                     Geom gm, int interf, int west_bc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > gm.nx + 1 || j > gm.ny + 1) return;
  const int64_t q = (int64_t)j * gm.pitch + i;
  const NodeInit s0 = initial_node(c, gm, i, j, interf, west_bc);
  st.a[q] = make_double2(s0.rho, s0.T - kTcrit);
  static_cast<typename Vec<R>::V4*>(st.b)[q] = make4<R>((R)s0.u, (R)s0.v, R(0), R(0));
  static_cast<typename CType<R, EQF>::T*>(st.c)[q] = typename CType<R, EQF>::T{};
  m.rho[q] = s0.rho;
  m.u[q] = s0.u;
  m.v[q] = s0.v;
  m.T[q] = s0.T;
  phi[q] = s0.phi;
  phip[q] = s0.phi;
}

template <int W, typename R, bool EQF>
hipError_t launch_ring(bgk_handle* h, const MomStep& st) {
  // resident workgroups per CU of this instantiation (LDS and registers)
  static const int per_cu = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_fused_mom<W, R, EQF>, W, 0) !=
        hipSuccess)
      n = 0;
    return n;
  }();
  const StripGrid sg =
      make_strip_grid(h->nx, h->ny, W, EQF ? 64 : 32, per_cu * h->n_cu, h->strip_rows);
  const int nedge = edge_count(h->nx, h->ny);
  const int64_t nwg = (int64_t)sg.nmain + (nedge + W - 1) / W;
  Macro m{h->rho, h->u, h->v, h->T};
  hipLaunchKernelGGL((k_fused_mom<W, R, EQF>), dim3((unsigned)nwg), dim3(W), 0, h->stream,
                     st.in, st.out, st.pa, st.pb, st.te_in, st.te_out, m, h->c,
                     step_constants(h->c), h->geom, sg, st.write_all ? 1 : 0);
  return hipGetLastError();
}

template <int W, typename R>
hipError_t launch_ring_layout(bgk_handle* h, const MomStep& st) {
  return h->mom_eqf ? launch_ring<W, R, true>(h, st) : launch_ring<W, R, false>(h, st);
}

// Width of the ring kernel's workgroups: the widest that adds at most a quarter to
// the columns, or the widest of those that add least; 0: none adds less than half.
// (The wider, the longer the contiguous pieces of a row; FP64 rows wider than 256
// do not fit the LDS of a resident workgroup twice.)
int ring_width(const bgk_handle* h) {
  const auto columns = [h](int w) { return ((int64_t)h->nx + w - 1) / w * w; };
  int best = 64;
  for (int w = h->prm.precision == BGK_FP32_MOM ? 512 : 256; w >= 64; w /= 2) {
    if (4 * columns(w) <= 5 * (int64_t)h->nx) return w;
    if (columns(w) < columns(best) || (columns(w) == columns(best) && w > best)) best = w;
  }
  return 2 * columns(best) <= 3 * (int64_t)h->nx ? best : 0;
}

// Whether a step alone goes through the ring kernel: its loads go past the caches,
// which leaves these to the macroscopic fields that a call's last step writes;
// its rows are longer pieces than a wave's; and its boundary nodes are a thread
// each, where the streaming kernel walks rows.  Measured, us per call of one
// step, streaming kernel with T = 1 / ring:
//              FP32 moments  omega_f = 1  FP64 moments  omega_f = 1
//   1700^2        85 / 84       71 / 73     151 / 133     105 / 96
//   1850^2       108 / 97       86 / 81     176 / 151     135 / 113
//   2048^2       146 / 107     121 / 89     211 / 172     165 / 129
//   4096^2       551 / 510     475 / 427    812 / 767     631 / 587
//   90 x 40000   157 / 125     136 / 105    215 / 186     170 / 140
//   130 x 40000  228 / 198     207 / 172    320 / 290     253 / 222
//   512 x 1500    30 / 37       25 / 35      42 / 44       32 / 35
//   250 x 2200    31 / 24       28 / 22      37 / 31       31 / 26
//   250 x 1000    15 / 19       14 / 18      17 / 23       15 / 20
//   60 x 60000   132 / 128     110 / 108    188 / 201     144 / 151
//   60 x 2500     16 / 12       15 / 12      17 / 15       16 / 13
//   7 x 3000      14 / 10       14 / 10      15 / 10       15 / 10
//   1 x 3000      14 / 8.2      14 / 8.1     15 / 8.4     15 / 8.3
bool ring_step(const bgk_handle* h) {
  if (h->mom_variant != 0) return h->mom_variant >= 4;
  const int64_t nodes = (int64_t)h->nx * h->ny;
  if (h->nx <= 2) return true;
  if (h->nx <= 64) return nodes <= 160000;
  return nodes >= (h->nx <= 384 ? (int64_t)1 << 19 : (int64_t)3 << 20) && ring_width(h) > 0;
}

// Whether the last two steps of a call go one by one, through the ring kernel: on
// small or narrow lattices of the general layout the launch of two that writes the
// fields takes up to four plain ones' time.  Measured, us per step of calls of two, one
// launch / two ring launches:
//              FP32 moments  FP64 moments
//   16 x 16     9.7 / 6.7     11.2 / 7.1
//   97 x 61     9.5 / 8.7     11.0 / 8.8
//   300^2      11.4 / 9.6     15.9 / 11.0
//   512^2        16 / 26        22 / 22
//   100 x 1500   16 / 11        22 / 15
//   30 x 6000    22 / 20        28 / 22
//   60 x 60000  117 / 128      195 / 198
//   90 x 40000  139 / 121      248 / 184
//   130 x 40000 203 / 188      307 / 279
bool ends_in_singles(const bgk_handle* h) {
  if (h->mom_variant != 0 || h->mom_eqf) return false;
  const int64_t nodes = (int64_t)h->nx * h->ny;
  if (h->nx <= 144) return h->nx > 64 || nodes <= (int64_t)1 << 18;
  return nodes <= (h->prm.precision == BGK_FP64_MOM ? (int64_t)1 << 17 : 100000);
}

template <typename R, bool EQF>
void launch_init(bgk_handle* h, const MomOut& st, dim3 grd) {
  Macro m{h->rho, h->u, h->v, h->T};
  hipLaunchKernelGGL((k_initialization_mom<R, EQF>), grd, dim3(TX, TY), 0, h->stream, st, m,
                     h->phi[h->pc], h->phi[1 - h->pc], h->c, h->geom, h->geom.nx / 40,
                     h->prm.west_bc);
}

}  // namespace

// Most steps per launch.  Two halve the HBM bytes of a step; three pay only
// where a node is large and its update small (FP64 moments with omega_f = 1:
// 4096^2 181 against 240 us per step, 2048^2 50 against 63) and most strips run no
// wall's code (200 x 20000 67 against 75, 130 x 40000 109 against 106, 60 x 60000
// 128 against 64; 60000 x 40 37 against 39, 400000 x 6 68 against 50).
//
// FP32 moments with omega_f = 1 take one step per launch beyond 2^25 nodes although
// two are faster there too (8192^2: 1.14 against 0.68 ms per step).  The reason is
// no measurement but a bound on a ratio: the backward pass is held to three plain
// forward steps at 8192^2, and at 2.87 ms a step (its kernel alone takes 1.80, at
// 89% of a copy's rate) it is four of the faster ones.  BGK_MOM_VARIANT=2 takes two
// at every size; the adjoint's own forward runs (`adjoint`) always do.
int mom_most_steps(const bgk_handle* h, bool adjoint) {
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  const int64_t nodes = (int64_t)h->nx * h->ny;
  if (h->mom_variant >= 4 || wave::wide_rows(h)) return 1;
  if (h->mom_variant > 0) return h->mom_variant == 3 && !(f64 && h->mom_eqf) ? 2 : h->mom_variant;
  if (!adjoint && !f64 && h->mom_eqf && nodes > (int64_t)1 << 25) return 1;
  const bool walls = h->nx <= 160 || h->ny <= 32;
  return f64 && h->mom_eqf && nodes >= (int64_t)1 << 21 && !walls ? 3 : 2;
}

// Of `left` steps, how many the next launch takes: an odd rest first, so that
// a call ends with a launch of several steps (which knows the state before
// the last one, for the halo).
int mom_next_steps(const bgk_handle* h, int left, bool adjoint) {
  const int most = mom_most_steps(h, adjoint);
  return left % most ? left % most : most;
}

hipError_t launch_mom_steps(bgk_handle* h, const MomStep& st, int T) {
  if (!st.ring) return launch_mom_stream(h, st, T);
  const int w = ring_width(h);
  if (h->prm.precision == BGK_FP64_MOM)
    return w == 256   ? launch_ring_layout<256, double>(h, st)
           : w == 128 ? launch_ring_layout<128, double>(h, st)
                      : launch_ring_layout<64, double>(h, st);
  return w == 512   ? launch_ring_layout<512, float>(h, st)
         : w == 256 ? launch_ring_layout<256, float>(h, st)
         : w == 128 ? launch_ring_layout<128, float>(h, st)
                    : launch_ring_layout<64, float>(h, st);
}

hipError_t launch_fused_steps_mom(bgk_handle* h, int nsteps) {
  // With a graph (recorded) the launches have the parity of the steps: what does
  // not fill whole ones, two of them where `most` is even, goes step by step.
  const int most = mom_most_steps(h), group = most % 2 == 0 ? 2 * most : most;
  const int whole = nsteps / group * group;
  const bool alone = ring_step(h), pair = nsteps >= 2 && ends_in_singles(h);
  for (int left = nsteps; left > 0;) {
    const int T = h->recorded          ? (left > whole ? 1 : most)
                  : pair && left == 2 ? 1
                                      : mom_next_steps(h, left);
    left -= T;
    const int a = h->cur, b = 1 - h->cur;
    MomStep st;
    st.in = MomIn{h->ma[a], h->mb[a], h->mc[a]};
    st.out = MomOut{h->ma[b], h->mb[b], h->mc[b]};
    st.pa = h->phi[h->pc];
    st.pb = h->phi[1 - h->pc];
    st.te_in = h->teast[h->te_cur];
    st.te_out = h->teast[1 - h->te_cur];
    // (an odd step before others writes no fields: through the ring only where the
    // lattice is large, 2048^2 103 us for 106, FP64 162 for 170)
    st.ring = T == 1 && (left <= 1 ? alone || pair : alone && h->nx > 384);
    st.write_all = mom_write_all(left, alone || pair);
    st.probe_idx = nullptr;
    st.probe_out = nullptr;
    st.probe_np = 0;
    const hipError_t e = launch_mom_steps(h, st, T);
    if (e != hipSuccess) return e;
    h->cur = b;
    h->pc = 1 - h->pc;
    h->te_cur = 1 - h->te_cur;
  }
  return hipSuccess;
}

hipError_t launch_initialization_mom(bgk_handle* h) {
  const Geom& g = h->geom;
  MomOut st{h->ma[h->cur], h->mb[h->cur], h->mc[h->cur]};
  dim3 grd((unsigned)((g.nx + 2 + TX - 1) / TX), (unsigned)((g.ny + 2 + TY - 1) / TY));
  const bool f64 = h->prm.precision == BGK_FP64_MOM;
  if (h->mom_eqf)
    f64 ? launch_init<double, true>(h, st, grd) : launch_init<float, true>(h, st, grd);
  else
    f64 ? launch_init<double, false>(h, st, grd) : launch_init<float, false>(h, st, grd);
  return hipGetLastError();
}

}  // namespace bgk
