// bgk_fused.hip -- the fused FP64 time step for the no-slip cavity.
//
// One kernel does the whole block STEP_7/main.f90:60-69 for one node per
// thread: pull streaming with BC_f/BC_g folded in, momentsPre, phase_field,
// forces, collision and moments, reading buffer A (cur) and writing buffer
// B (1-cur).  Compiled with -ffp-contract=off; the arithmetic is operand for
// operand the reference's, so results equal STEP_7's bit for bit.
//
// How the boundary routines fold into the pull when all four walls are
// no-slip (BC type 4, STEP_7/BC_f.f90:62-68,101-107,125-136,181-192):
//  * every ghost population the pull reads was written by BC_f from the
//    reading node's own opposite population (half-way bounce-back), except
//    f6(Nx+1,0) and f7(Nx+1,Ny+1), which no BC writes: they keep their
//    initial value.  Those two are read from memory and copied into B.
//  * BC_g (STEP_7/BC_g.f90:9-64) makes the west ghosts the equilibrium at
//    Tin with u(0,j), v(0,j), the east ghosts the equilibrium at the
//    previous step's averaged T(Nx,j) with u(Nx+1,j), v(Nx+1,j), and then
//    copies rows 1 and Ny to rows 0 and Ny+1 for all columns: a pull from
//    row 0 / Ny+1 reads row 1 / Ny (clamped row), and a pull from column 0 /
//    Nx+1 evaluates that equilibrium.  T(Nx,j) of the previous step is kept
//    in the small ping-pong array teast.
//  * phi_prec rows 0 / Ny+1 are BC_g copies of rows 1 / Ny (clamped rows);
//    columns 0 / Nx+1 are never written after initialization and are copied
//    from A to B.
//  * the halo of rho, T, u, v and phi after a step holds what BC_f/BC_g
//    wrote at the start of that step, i.e. previous-step values; the edge
//    nodes write them so a download sees the reference's full arrays.
#include "bgk_pop64.h"

namespace bgk {
namespace {

struct Macro {
  double *rho, *u, *v, *T;
};

// pair view of buffer b: plane k holds (f_k, g_k) per node
inline Pairs64 pairs(double* const* fplanes) {
  Pairs64 r;
  for (int k = 0; k < 9; ++k) r.p[k] = reinterpret_cast<double2*>(fplanes[k]);
  return r;
}

constexpr int kNodeBytes = 2 * (18 + 1) * (int)sizeof(double);  // populations and phi

__global__ void k_teast_prologue(const double* __restrict__ T, double* __restrict__ te, Geom gm) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j > gm.ny + 1) return;
  te[j] = T[(int64_t)j * gm.pitch + gm.nx];
}

// What bounds it on small lattices is latency: a launch every few us whose
// waves make a dozen dependent memory accesses.  So a wave that holds a
// boundary-adjacent node takes one path for all its lanes, with every load
// (ghost velocities and halo values included) issued before the first use
// (us per step: 256^2 9.4 with the ghosts' loads in branches, 7.6 so; with rows in
// bands, make_tile_grid, 6.4; 97 x 61 7.7, 6.1 and 5.7).
template <bool STEP7, bool CACHED>
__global__ __launch_bounds__(TILE_W) void k_fused64(Planes<double2> A, Planes<double2> B,
                                                     const double* __restrict__ pa,
                                                     double* __restrict__ pb,
                                                     const double* __restrict__ te_in,
                                                     double* __restrict__ te_out, Macro m,
                                                     Consts c, Geom gm, TileGrid tg,
                                                     int write_all) {
  const int nx = gm.nx, ny = gm.ny;
  int i, j;
  if (!tile_node(tg, gm, &i, &j)) return;
  const int64_t P = gm.pitch;
  const int64_t q = (int64_t)j * P + i;
  const bool w_edge = (i == 1), e_edge = (i == nx), s_edge = (j == 1), n_edge = (j == ny);
  const bool edge = w_edge || e_edge || s_edge || n_edge;

  // ---- phi_prec taps (STEP_7/phase_field.f90:27-45), rows clamped per BC_g
  const int64_t rn = (int64_t)(j < ny ? j + 1 : ny) * P;
  const int64_t rs = (int64_t)(j > 1 ? j - 1 : 1) * P;
  const int64_t r0 = (int64_t)j * P;
  const double tap[9] = {pa[q],          pa[r0 + i + 1], pa[rn + i],     pa[r0 + i - 1], pa[rs + i],
                         pa[rn + i + 1], pa[rn + i - 1], pa[rs + i - 1], pa[rs + i + 1]};

  // ---- streaming (STEP_7/streaming.f90:7-25) with the boundaries folded in
  Row in;
  double rho_was = 0.0, T_was = 0.0;  // of this node before the step (the halo)
  double frozen6 = 0.0, frozen7 = 0.0;
  if (!__any(edge)) {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const double2 fg = load_pair<CACHED>(A.row(k, q - CX[k] - (int64_t)CY[k] * P));
      in.f[k] = fg.x;
      in.g[k] = fg.y;
    }
  } else {
    using wave::as_scalar;
    unsigned offs[3];
    edge_offsets(i, nx, offs);
    EdgeRow e;
    load_pulled_edge(A, P, ny, offs, j, e);
    rho_was = m.rho[q];
    T_was = m.T[q];
    frozen6 = as_scalar(&A.row(6, nx + 1)->x)[0];
    frozen7 = as_scalar(&A.row(7, (int64_t)(ny + 1) * P + nx + 1)->x)[0];
    // thermal ghosts in the rows below, beside and above (the row j is the
    // workgroup's, so these are scalar loads)
    const int rows[3] = {j > 1 ? j - 1 : 1, j, j < ny ? j + 1 : ny};
    constexpr int KW[3] = {5, 1, 8}, KE[3] = {6, 3, 7};
    double uw[3], vw[3], ue[3], ve[3], te[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const int64_t h = (int64_t)rows[s] * P;
      uw[s] = as_scalar(m.u)[h];
      vw[s] = as_scalar(m.v)[h];
      ue[s] = as_scalar(m.u)[h + nx + 1];
      ve[s] = as_scalar(m.v)[h + nx + 1];
      te[s] = c.east_cold ? c.t_cold : as_scalar(te_in)[rows[s]];
    }
    wall_f(nx, ny, i, j, frozen6, frozen7, e);
    in = e.r;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const double gw = equilibrium_k(c, KW[s], c.tin, uw[s], vw[s]);
      const double ge = equilibrium_k(c, KE[s], te[s], ue[s], ve[s]);
      in.g[KW[s]] = w_edge ? gw : in.g[KW[s]];
      in.g[KE[s]] = e_edge ? ge : in.g[KE[s]];
    }
  }

  // ---- momentsPre .. collision
  const Done o = node_step<STEP7>(c, in.f, in.g, tap);
#pragma unroll
  for (int k = 0; k < 9; ++k) store_pair<CACHED>(B.row(k, q), o.f[k], o.g[k]);
  store_one<CACHED>(&pb[q], o.phi);

  // ---- moments (STEP_7/moments.f90:11-25), where somebody reads them
  if (edge || write_all) {
    const Avg a = averaged(o);
    if (edge) {
      // halo as BC_f / BC_g left it at the start of this step
      if (s_edge) {
        m.rho[i] = rho_was;
        m.T[i] = T_was;
        m.u[i] = 0.0;
        m.v[i] = 0.0;
        pb[i] = tap[0];
      }
      if (n_edge) {
        const int64_t h = (int64_t)(ny + 1) * P + i;
        m.rho[h] = rho_was;
        m.T[h] = T_was;
        m.u[h] = 0.0;
        m.v[h] = 0.0;
        pb[h] = tap[0];
      }
      if (w_edge) {
        m.T[r0] = c.tin;
        pb[r0] = tap[3];
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
        pb[h] = tap[1];
        te_out[j] = a.T;
        if (s_edge) {
          m.T[nx + 1] = east_T(c, te_in, 1);
          pb[nx + 1] = pa[P + nx + 1];
          B.row(6, nx + 1)->x = frozen6;
        }
        if (n_edge) {
          const int64_t hn = (int64_t)(ny + 1) * P + nx + 1;
          m.T[hn] = east_T(c, te_in, ny);
          pb[hn] = pa[(int64_t)ny * P + nx + 1];
          B.row(7, hn)->x = frozen7;
        }
      }
    }
    m.rho[q] = a.rho;
    m.T[q] = a.T;
    m.u[q] = a.u;
    m.v[q] = a.v;
  }
}

// One step for any walls, after BC_f and BC_g (bgk_stage.hip) have written the
// ghosts of A and pa: every pull and tap is a load.  The workgroups past the
// tiles copy the ghosts, of which a boundary type may leave some unwritten, to
// the next step's planes.  304 B per node as k_fused64, where the eight
// subroutines move about 1.1 KB in ten launches (1024 x 512 channel, us per
// step: 149 by subroutines, 48 in two launches, 38 with rows in bands).
template <bool STEP7, bool CACHED>
__global__ __launch_bounds__(TILE_W) void k_general64(Pairs64 A, Pairs64 B,
                                                      const double* __restrict__ pa,
                                                      double* __restrict__ pb, Macro m, Consts c,
                                                      Geom gm, TileGrid tg, int write_all) {
  const int nx = gm.nx, ny = gm.ny;
  const int64_t P = gm.pitch;
  const int64_t past = (int64_t)blockIdx.x - tg.per * NXCD;
  if (past >= 0) {
    // ghost node e: rows 0 and Ny+1, then columns 0 and Nx+1 of rows 1..Ny
    const int64_t e = past * TILE_W + threadIdx.x, row = nx + 2;
    if (e >= 2 * row + 2 * (int64_t)ny) return;
    const int64_t q = e < row       ? e
                      : e < 2 * row ? (int64_t)(ny + 1) * P + (e - row)
                                    : ((e - 2 * row) / 2 + 1) * P + ((e & 1) ? nx + 1 : 0);
#pragma unroll
    for (int k = 0; k < 9; ++k) B.p[k][q] = A.p[k][q];
    pb[q] = pa[q];
    return;
  }
  int i, j;
  if (!tile_node(tg, gm, &i, &j)) return;
  const int64_t q = (int64_t)j * P + i;
  double fp[9], gp[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const double2 fg = load_pair<CACHED>(&A.p[k][q - CX[k] - (int64_t)CY[k] * P]);
    fp[k] = fg.x;
    gp[k] = fg.y;
  }
  const double tap[9] = {pa[q],         pa[q + 1],     pa[q + P],     pa[q - 1], pa[q - P],
                         pa[q + 1 + P], pa[q - 1 + P], pa[q - 1 - P], pa[q + 1 - P]};
  const Done o = node_step<STEP7>(c, fp, gp, tap);
#pragma unroll
  for (int k = 0; k < 9; ++k) store_pair<CACHED>(&B.p[k][q], o.f[k], o.g[k]);
  store_one<CACHED>(&pb[q], o.phi);
  // BC_f and BC_g read the moments of the boundary-adjacent nodes
  if (write_all || i == 1 || i == nx || j == 1 || j == ny) {
    const Avg a = averaged(o);
    m.rho[q] = a.rho;
    m.T[q] = a.T;
    m.u[q] = a.u;
    m.v[q] = a.v;
  }
}

}  // namespace

hipError_t launch_teast_prologue(bgk_handle* h) {
  if (h->te_ok && !h->recorded) return hipSuccess;
  const Geom& g = h->geom;
  hipLaunchKernelGGL(k_teast_prologue, dim3((unsigned)((g.ny + 2 + 255) / 256)), dim3(256), 0,
                     h->stream, h->T, h->teast[h->te_cur], g);
  const hipError_t e = hipGetLastError();
  h->te_ok = e == hipSuccess;
  return e;
}

hipError_t launch_fused_step64(bgk_handle* h, bool write_all) {
  const Geom& g = h->geom;
  const TileGrid tg = make_tile_grid(g, kNodeBytes);
  dim3 blk(TILE_W);
  dim3 grd((unsigned)(tg.per * NXCD));
  Macro m{h->rho, h->u, h->v, h->T};
  const double* te_in = h->teast[h->te_cur];
  double* te_out = h->teast[1 - h->te_cur];
  const int a = h->cur, b = 1 - h->cur;
  const Planes<double2> A = wave::planes_of<double2>(h->f[a]), B = wave::planes_of<double2>(h->f[b]);
  const bool s7 = h->prm.rounding == BGK_ROUND_STEP7;
  const auto k = s7 ? (tg.cached ? k_fused64<true, true> : k_fused64<true, false>)
                    : (tg.cached ? k_fused64<false, true> : k_fused64<false, false>);
  hipLaunchKernelGGL(k, grd, blk, 0, h->stream, A, B, h->phi[h->pc], h->phi[1 - h->pc], te_in,
                     te_out, m, h->c, g, tg, write_all ? 1 : 0);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) {
    h->cur = b;
    h->pc = 1 - h->pc;
    h->te_cur = 1 - h->te_cur;
  }
  return e;
}

hipError_t launch_general_step64(bgk_handle* h, bool write_all) {
  hipError_t e = launch_bc(h, true, true);
  if (e != hipSuccess) return e;
  const Geom& g = h->geom;
  const TileGrid tg = make_tile_grid(g, kNodeBytes);
  const int64_t ghosts = 2 * ((int64_t)g.nx + 2) + 2 * (int64_t)g.ny;
  const dim3 grd((unsigned)(tg.per * NXCD + (ghosts + TILE_W - 1) / TILE_W));
  Macro m{h->rho, h->u, h->v, h->T};
  const int a = h->cur, b = 1 - h->cur;
  const bool s7 = h->prm.rounding == BGK_ROUND_STEP7;
  const auto k = s7 ? (tg.cached ? k_general64<true, true> : k_general64<true, false>)
                    : (tg.cached ? k_general64<false, true> : k_general64<false, false>);
  hipLaunchKernelGGL(k, grd, dim3(TILE_W), 0, h->stream, pairs(h->f[a]), pairs(h->f[b]),
                     h->phi[h->pc], h->phi[1 - h->pc], m, h->c, g, tg, write_all ? 1 : 0);
  e = hipGetLastError();
  if (e == hipSuccess) {
    h->cur = b;
    h->pc = 1 - h->pc;
  }
  return e;
}

}  // namespace bgk
