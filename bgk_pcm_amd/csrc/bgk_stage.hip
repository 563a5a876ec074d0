// bgk_stage.hip -- one kernel (or kernel pair) per reference subroutine.
//
// This is the per-subroutine path of the drop-in boundary: bgk_bc_f,
// bgk_bc_g, bgk_streaming, ... each launch the kernels below on the handle's
// stream, on the same fields the reference's `module shared` holds.  It
// serves every boundary type of the reference and is the path bgk_step takes
// when the walls are not all no-slip.  Compiled with -ffp-contract=off: the
// FP64 results equal the reference's bit for bit.
#include <algorithm>

#include "bgk_internal.h"

namespace bgk {
namespace {

struct Macro {
  double *rho, *u, *v, *T, *rho2, *u2, *v2, *T2;
};

inline Macro macro_of(bgk_handle* h) {
  return Macro{h->rho, h->u, h->v, h->T, h->rho2, h->u2, h->v2, h->T2};
}

inline Pops64 pops(double* const* p) {
  Pops64 r;
  for (int k = 0; k < 9; ++k) r.p[k].base = p[k];
  return r;
}

// pair view: plane k holds (f_k, g_k) per node.  One 16-byte access serves both
// members; as two stride-2 accesses each cache line was requested twice.  A step
// by subroutines, us, before and after pairs, merged boundary launches and no
// copy of phi: 64^2 40 / 32, 512^2 90 / 79, 1024 x 512 151 / 130, 2048 x 1024
// 610 / 530.
inline Pairs64 pairs(double* const* fplanes) {
  Pairs64 r;
  for (int k = 0; k < 9; ++k) r.p[k] = reinterpret_cast<double2*>(fplanes[k]);
  return r;
}
__device__ __forceinline__ void load_pairs(const Pairs64& p, int64_t q, double a[9],
                                           double b[9]) {
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const double2 v = p.p[k][q];
    a[k] = v.x;
    b[k] = v.y;
  }
}

constexpr int TX = 64, TY = 4;

inline dim3 interior_grid(const Geom& g) {
  return dim3((unsigned)((g.nx + TX - 1) / TX), (unsigned)((g.ny + TY - 1) / TY));
}

// ------------------------------------------------------------ initialization
// STEP_7/initialization.f90:15-152, one thread per node including the halo.
__global__ void k_initialization(Pops64 f, Pops64 g, Macro m, double* phi, double* phip,
                                 Consts c, Geom gm, int interf, int west_bc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > gm.nx + 1 || j > gm.ny + 1) return;
  const int64_t q = (int64_t)j * gm.pitch + i;
  const NodeInit s0 = initial_node(c, gm, i, j, interf, west_bc);
  const double T = s0.T, rho = s0.rho, u = s0.u, v = s0.v;
  double eq[9];
  equilibria(c, rho, u, v, eq);
#pragma unroll
  for (int k = 0; k < 9; ++k) f.p[k][q] = eq[k];
  equilibria(c, T, u, v, eq);
#pragma unroll
  for (int k = 0; k < 9; ++k) g.p[k][q] = eq[k];
  m.rho[q] = rho;
  m.u[q] = u;
  m.v[q] = v;
  m.T[q] = T;
  m.rho2[q] = 0.0;
  m.u2[q] = 0.0;
  m.v2[q] = 0.0;
  m.T2[q] = 0.0;
  phi[q] = s0.phi;
  phip[q] = s0.phi;
}

// Boundary types of the four sides (input.dat).
struct Walls {
  int west, east, north, south;
};

// ----------------------------------------------------------------------- BC_f
// West and east sides, row j = 0..Ny+1 (STEP_7/BC_f.f90:9-104).
__device__ __forceinline__ void bc_f_we(const Pops64& F, const Macro& m, const Consts& c,
                                        const Geom& gm, const Walls& w, int j) {
  const int nx = gm.nx, ny = gm.ny, wbc = w.west, ebc = w.east;
  const int64_t P = gm.pitch;
  auto at = [&](int i, int jj) { return (int64_t)jj * P + i; };
  const Strided2<double>* f = F.p;
  const bool inner = (j >= 1 && j <= ny);
  double uu, vv, uv, upv, umv;
  // WEST
  if (wbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][at(0, j)] = f[k][at(nx, j)];
  } else if (wbc == 1) {
    if (inner) {
      const double u0 = c.u0, v0 = c.v0;
      uu = u0 * u0; vv = v0 * v0; uv = 1.5 * (uu + vv); upv = u0 + v0; umv = u0 - v0;
      const double r1 = m.rho[at(1, j)];
      f[1][at(0, j)] = c.w[1] * r1 * (1.0 + 3.0 * u0 + 4.5 * uu - uv);
      f[5][at(0, j)] = c.w[5] * r1 * (1.0 + 3.0 * upv + 4.5 * upv * upv - uv);
      f[8][at(0, j)] = c.w[8] * r1 * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv);
      m.u[at(0, j)] = u0;
      m.v[at(0, j)] = v0;
      m.rho[at(0, j)] = r1;
    }
  } else if (wbc == 2) {
    const double uw = m.u[at(0, j)], v0 = c.v0;
    uu = uw * uw; vv = v0 * v0; uv = 1.5 * (uu + vv); upv = uw + v0; umv = uw - v0;
    const double r1 = m.rho[at(1, j)];
    f[1][at(0, j)] = c.w[1] * r1 * (1.0 + 3.0 * uw + 4.5 * uu - uv);
    f[5][at(0, j)] = c.w[5] * r1 * (1.0 + 3.0 * upv + 4.5 * upv * upv - uv);
    f[8][at(0, j)] = c.w[8] * r1 * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv);
  } else if (wbc == 3) {
    const double u1 = m.u[at(1, j)], v1 = m.v[at(1, j)];
    uu = u1 * u1; vv = v1 * v1; uv = 1.5 * (uu + vv); upv = u1 + v1; umv = u1 - v1;
    f[1][at(0, j)] = c.w[1] * c.rho1 * (1.0 + 3.0 * u1 + 4.5 * uu - uv);
    f[5][at(0, j)] = c.w[5] * c.rho1 * (1.0 + 3.0 * upv + 4.5 * upv * upv - uv);
    f[8][at(0, j)] = c.w[8] * c.rho1 * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv);
    m.u[at(0, j)] = u1;
    m.v[at(0, j)] = v1;
    m.rho[at(0, j)] = c.rho1;
  } else if (wbc == 4) {
    if (inner) {
      f[1][at(0, j)] = f[3][at(1, j)];
      f[8][at(0, j)] = f[6][at(1, j - 1)];
      f[5][at(0, j)] = f[7][at(1, j + 1)];
    }
  }
  // EAST
  if (ebc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][at(nx + 1, j)] = f[k][at(1, j)];
  } else if (ebc == 3) {
    if (inner) {
      const double ue = m.u[at(nx, j)], ve = m.v[at(nx, j)];
      uu = ue * ue; vv = ve * ve; uv = 1.5 * (uu + vv); upv = ue + ve; umv = ue - ve;
      f[3][at(nx + 1, j)] = c.w[3] * c.rho0 * (1.0 - 3.0 * ue + 4.5 * uu - uv);
      f[6][at(nx + 1, j)] = c.w[6] * c.rho0 * (1.0 - 3.0 * umv + 4.5 * umv * umv - uv);
      f[7][at(nx + 1, j)] = c.w[7] * c.rho0 * (1.0 - 3.0 * upv + 4.5 * upv * upv - uv);
      m.u[at(nx + 1, j)] = ue;
      m.v[at(nx + 1, j)] = ve;
      m.rho[at(nx + 1, j)] = c.rho0;
    }
  } else if (ebc == 4) {
    if (inner) {
      f[3][at(nx + 1, j)] = f[1][at(nx, j)];
      f[6][at(nx + 1, j)] = f[8][at(nx, j + 1)];
      f[7][at(nx + 1, j)] = f[5][at(nx, j - 1)];
    }
  }
}

// North and south sides, column i = 0..Nx+1 (STEP_7/BC_f.f90:108-196), after
// bc_f_we.
__device__ __forceinline__ void bc_f_ns(const Pops64& F, const Macro& m, const Consts& c,
                                        const Geom& gm, const Walls& w, int i) {
  const int nx = gm.nx, ny = gm.ny, nbc = w.north, sbc = w.south;
  const int64_t P = gm.pitch;
  auto at = [&](int ii, int jj) { return (int64_t)jj * P + ii; };
  const Strided2<double>* f = F.p;
  const bool inner = (i >= 1 && i <= nx);
  // NORTH
  if (nbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][at(i, ny + 1)] = f[k][at(i, 1)];
  } else if (nbc == 4) {
    if (inner) {
      f[4][at(i, ny + 1)] = f[2][at(i, ny)];
      f[7][at(i, ny + 1)] = f[5][at(i - 1, ny)];
      f[8][at(i, ny + 1)] = f[6][at(i + 1, ny)];
      m.rho[at(i, ny + 1)] = m.rho[at(i, ny)];
      m.u[at(i, ny + 1)] = 0.0;
      m.v[at(i, ny + 1)] = 0.0;
    }
    if (i == 0) f[8][at(0, ny + 1)] = f[6][at(1, ny)];
  } else if (nbc == 5) {
    f[4][at(i, ny + 1)] = f[2][at(i, ny - 1)];
    f[7][at(i, ny + 1)] = f[6][at(i, ny - 1)];
    f[8][at(i, ny + 1)] = f[5][at(i, ny - 1)];
  } else if (nbc == 6) {
    f[4][at(i, ny + 1)] = f[4][at(i, ny)];
    f[7][at(i, ny + 1)] = f[7][at(i, ny)];
    f[8][at(i, ny + 1)] = f[8][at(i, ny)];
  } else if (nbc == 1) {
    const double u0 = c.u0, v0 = c.v0;
    const double uu = u0 * u0, vv = v0 * v0, uv = 1.5 * (uu + vv), upv = u0 + v0, umv = u0 - v0;
    const double rn = m.rho[at(i, ny)];
    f[4][at(i, ny + 1)] = c.w[4] * rn * (1.0 - 3.0 * v0 + 4.5 * vv - uv);
    f[7][at(i, ny + 1)] = c.w[7] * rn * (1.0 - 3.0 * upv + 4.5 * upv * upv - uv);
    f[8][at(i, ny + 1)] = c.w[8] * rn * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv);
  }
  // SOUTH
  if (sbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][at(i, 0)] = f[k][at(i, ny)];
  } else if (sbc == 4) {
    if (inner) {
      f[2][at(i, 0)] = f[4][at(i, 1)];
      f[5][at(i, 0)] = f[7][at(i + 1, 1)];
      f[6][at(i, 0)] = f[8][at(i - 1, 1)];
      m.rho[at(i, 0)] = m.rho[at(i, 1)];
      m.u[at(i, 0)] = 0.0;
      m.v[at(i, 0)] = 0.0;
    }
    if (i == 0) f[5][at(0, 0)] = f[7][at(1, 1)];
  } else if (sbc == 6) {
    f[2][at(i, 0)] = f[2][at(i, 1)];
    f[5][at(i, 0)] = f[5][at(i, 1)];
    f[6][at(i, 0)] = f[6][at(i, 1)];
  }
}

// ----------------------------------------------------------------------- BC_g
// West and east, row j = 1..Ny (STEP_7/BC_g.f90:9-31).
__device__ __forceinline__ void bc_g_we(const Pops64& G, const Macro& m, const Consts& c,
                                        const Geom& gm, int j) {
  const int nx = gm.nx;
  const int64_t P = gm.pitch;
  auto at = [&](int ii, int jj) { return (int64_t)jj * P + ii; };
  const Strided2<double>* g = G.p;
  {
    const double uw = m.u[at(0, j)], vw = m.v[at(0, j)];
    const double uu = uw * uw, vv = vw * vw, uv = 1.5 * (uu + vv), upv = uw + vw, umv = uw - vw;
    g[1][at(0, j)] = c.w[1] * c.tin * (1.0 + 3.0 * uw + 4.5 * uu - uv);
    g[5][at(0, j)] = c.w[5] * c.tin * (1.0 + 3.0 * upv + 4.5 * upv * upv - uv);
    g[8][at(0, j)] = c.w[8] * c.tin * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv);
    m.T[at(0, j)] = c.tin;
  }
  {
    // the averaged T(Nx, j), or the cold-wall extension's fixed temperature
    const double ue = m.u[at(nx + 1, j)], ve = m.v[at(nx + 1, j)];
    const double te = c.east_cold ? c.t_cold : m.T[at(nx, j)];
    const double uu = ue * ue, vv = ve * ve, uv = 1.5 * (uu + vv), upv = ue + ve, umv = ue - ve;
    g[3][at(nx + 1, j)] = c.w[3] * te * (1.0 - 3.0 * ue + 4.5 * uu - uv);
    g[6][at(nx + 1, j)] = c.w[6] * te * (1.0 - 3.0 * umv + 4.5 * umv * umv - uv);
    g[7][at(nx + 1, j)] = c.w[7] * te * (1.0 - 3.0 * upv + 4.5 * upv * upv - uv);
    m.T[at(nx + 1, j)] = te;
  }
}

// North and south zero-gradient copies, column i = 0..Nx+1
// (STEP_7/BC_g.f90:36-64), after bc_g_we.
__device__ __forceinline__ void bc_g_ns(const Pops64& G, const Macro& m, double* phi,
                                        const Geom& gm, int i) {
  const int ny = gm.ny;
  const int64_t P = gm.pitch;
  const int64_t qn = (int64_t)ny * P + i, qn1 = (int64_t)(ny + 1) * P + i;
  const int64_t q1 = P + i, q0 = i;
#pragma unroll
  for (int k = 0; k < 9; ++k) G.p[k][qn1] = G.p[k][qn];
  m.T[qn1] = m.T[qn];
  phi[qn1] = phi[qn];
#pragma unroll
  for (int k = 0; k < 9; ++k) G.p[k][q0] = G.p[k][q1];
  m.T[q0] = m.T[q1];
  phi[q0] = phi[q1];
}

// BC_f and/or BC_g.  The sides depend on each other in the reference's order
// (west and east, then north and south; f before g).  PHASE 0: all of it by one
// workgroup, which waits between the four parts; 1..4: one part, one thread per
// node, for lattices whose sides one workgroup would walk too slowly.  What
// bounds a part is the latency of a launch or of a few dependent accesses, so
// one launch of one workgroup beats four.
constexpr int kBcThreads = 1024;
struct BcArgs {
  Pops64 F, G;
  Macro m;
  double* phi;
  Consts c;
  Geom gm;
  Walls w;
  int do_f, do_g;
};
template <int PHASE>
__global__ __launch_bounds__(kBcThreads) void k_bc(BcArgs a) {
  const int nx = a.gm.nx, ny = a.gm.ny;
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const int step = PHASE == 0 ? kBcThreads : nx + ny + 4;  // (1..4: one node each)
  if ((PHASE == 0 && a.do_f) || PHASE == 1)
    for (int j = t0; j <= ny + 1; j += step) bc_f_we(a.F, a.m, a.c, a.gm, a.w, j);
  if (PHASE == 0 && a.do_f) __syncthreads();
  if ((PHASE == 0 && a.do_f) || PHASE == 2)
    for (int i = t0; i <= nx + 1; i += step) bc_f_ns(a.F, a.m, a.c, a.gm, a.w, i);
  if (PHASE == 0 && a.do_f && a.do_g) __syncthreads();
  if ((PHASE == 0 && a.do_g) || PHASE == 3)
    for (int j = t0 + 1; j <= ny; j += step) bc_g_we(a.G, a.m, a.c, a.gm, j);
  if (PHASE == 0 && a.do_g) __syncthreads();
  if ((PHASE == 0 && a.do_g) || PHASE == 4)
    for (int i = t0; i <= nx + 1; i += step) bc_g_ns(a.G, a.m, a.phi, a.gm, i);
}

// ------------------------------------------------------------------ streaming
// Pull of f and g into fp and gp, STEP_7/streaming.f90:5-27.
__global__ void k_streaming(Pairs64 f, Pairs64 fp, Geom gm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
  if (i > gm.nx || j > gm.ny) return;
  const int64_t P = gm.pitch;
  const int64_t q = (int64_t)j * P + i;
#pragma unroll
  for (int k = 0; k < 9; ++k) fp.p[k][q] = f.p[k][q - CX[k] - (int64_t)CY[k] * P];
}

// ----------------------------------------------------------------- momentsPre
// STEP_7/momentsPre.f90:8-21.
__global__ void k_moments_pre(Pairs64 fp, Macro m, Geom gm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
  if (i > gm.nx || j > gm.ny) return;
  const int64_t q = (int64_t)j * gm.pitch + i;
  double a[9], b[9];
  load_pairs(fp, q, a, b);
  const double r = a[0] + a[1] + a[2] + a[3] + a[4] + a[5] + a[6] + a[7] + a[8];
  const double t = b[0] + b[1] + b[2] + b[3] + b[4] + b[5] + b[6] + b[7] + b[8];
  const double irho = 1.0 / r;
  const double u = irho * (a[1] - a[3] + a[5] - a[6] - a[7] + a[8]);
  const double v = irho * (a[2] - a[4] + a[5] + a[6] - a[7] - a[8]);
  m.rho[q] = r;
  m.T[q] = t;
  m.u[q] = u;
  m.v[q] = v;
  m.rho2[q] = r;
  m.T2[q] = t;
  m.u2[q] = u;
  m.v2[q] = v;
}

// ---------------------------------------------------------------- phase_field
// STEP_7/phase_field.f90:19-55.  The copy phi_prec(:,:) = phi(:,:) of :19 is the
// exchange of the two planes: pp holds the old phi, and the new one goes to the
// other plane, with the halo nodes (which the update leaves) copied along.
__global__ void k_phase_field(double* phi, const double* pp, const double* T, Consts c,
                              Geom gm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > gm.nx + 1 || j > gm.ny + 1) return;
  const int64_t P = gm.pitch;
  const int64_t q = (int64_t)j * P + i;
  if (i < 1 || i > gm.nx || j < 1 || j > gm.ny) {
    phi[q] = pp[q];
    return;
  }
  const double tap[9] = {pp[q],         pp[q + 1],     pp[q + P],     pp[q - 1], pp[q - P],
                         pp[q + 1 + P], pp[q - 1 + P], pp[q - 1 - P], pp[q + 1 - P]};
  phi[q] = phase_update(c, T[q], tap);
}

// --------------------------------------------------------------------- forces
// STEP_7/forces.f90:15-26.
__global__ void k_forces(Macro m, const double* phi, const double* pp, Consts c, Geom gm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
  if (i > gm.nx || j > gm.ny) return;
  const int64_t q = (int64_t)j * gm.pitch + i;
  const double ph = phi[q];
  const double rho = m.rho[q];
  const double t = m.T[q] - (c.dt_st * (ph - pp[q]) / 2.0);
  double fy = buoyancy(c, rho, t, ph);
  const double u = m.u[q], v = m.v[q];
  const double fx = -(u * (1.0 - ph) * 0.5);
  fy = fy - v * (1.0 - ph) * 0.5;
  m.T[q] = t;
  m.u[q] = u + fx / (c.omega_f * rho);
  m.v[q] = v + fy / (c.omega_f * rho);
}

// ------------------------------------------------------------------ collision
// STEP_7/collision.f90:14-152.
template <bool STEP7>
__global__ void k_collision(Pairs64 fp, Pairs64 f, Macro m, const double* __restrict__ phi,
                            Consts c, Geom gm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
  if (i > gm.nx || j > gm.ny) return;
  const int64_t q = (int64_t)j * gm.pitch + i;
  const double u = m.u[q], v = m.v[q];
  double a[9], b[9], fo[9], go[9];
  load_pairs(fp, q, a, b);
  regularised_bgk<STEP7>(c, c.omega_f, m.rho[q], u, v, a, fo);
  regularised_bgk<STEP7>(c, omega_g_at(c, phi[q]), m.T[q], u, v, b, go);
#pragma unroll
  for (int k = 0; k < 9; ++k) f.p[k][q] = make_double2(fo[k], go[k]);
}

// -------------------------------------------------------------------- moments
// STEP_7/moments.f90:11-25.
__global__ void k_moments(Pairs64 f, Macro m, Geom gm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;
  if (i > gm.nx || j > gm.ny) return;
  const int64_t q = (int64_t)j * gm.pitch + i;
  double a[9], b[9];
  load_pairs(f, q, a, b);
  const double r = a[0] + a[1] + a[2] + a[3] + a[4] + a[5] + a[6] + a[7] + a[8];
  const double irho = 1.0 / r;
  const double tt = b[0] + b[1] + b[2] + b[3] + b[4] + b[5] + b[6] + b[7] + b[8];
  const double tu = irho * (a[1] - a[3] + a[5] - a[6] - a[7] + a[8]);
  const double tv = irho * (a[2] - a[4] + a[5] + a[6] - a[7] - a[8]);
  m.rho[q] = r;
  m.T[q] = (tt + m.T2[q]) * 0.5;
  m.u[q] = (tu + m.u2[q]) * 0.5;
  m.v[q] = (tv + m.v2[q]) * 0.5;
}

inline unsigned blocks1d(int n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// ------------------------------------------------------------------ launchers

hipError_t launch_initialization(bgk_handle* h) {
  const Geom& g = h->geom;
  dim3 blk(TX, TY);
  dim3 grd((unsigned)((g.nx + 2 + TX - 1) / TX), (unsigned)((g.ny + 2 + TY - 1) / TY));
  hipLaunchKernelGGL(k_initialization, grd, blk, 0, h->stream, pops(h->f[h->cur]),
                     pops(h->g[h->cur]), macro_of(h), h->phi[h->pc], h->phi[1 - h->pc], h->c,
                     g, g.nx / 40, h->prm.west_bc);
  return hipGetLastError();
}

hipError_t launch_bc(bgk_handle* h, bool do_f, bool do_g) {
  const Geom& g = h->geom;
  BcArgs a{pops(h->f[h->cur]), pops(h->g[h->cur]), macro_of(h), h->phi[h->pc], h->c, g,
           Walls{h->prm.west_bc, h->prm.east_bc, h->prm.north_bc, h->prm.south_bc},
           do_f ? 1 : 0, do_g ? 1 : 0};
  // one workgroup up to four rounds of its threads on a side
  if (std::max(g.nx, g.ny) + 2 <= 4 * kBcThreads) {
    hipLaunchKernelGGL(k_bc<0>, dim3(1), dim3(kBcThreads), 0, h->stream, a);
    return hipGetLastError();
  }
  const dim3 we(blocks1d(g.ny + 2, 256)), ns(blocks1d(g.nx + 2, 256));
  if (do_f) {
    hipLaunchKernelGGL(k_bc<1>, we, dim3(256), 0, h->stream, a);
    hipLaunchKernelGGL(k_bc<2>, ns, dim3(256), 0, h->stream, a);
  }
  if (do_g) {
    hipLaunchKernelGGL(k_bc<3>, we, dim3(256), 0, h->stream, a);
    hipLaunchKernelGGL(k_bc<4>, ns, dim3(256), 0, h->stream, a);
  }
  return hipGetLastError();
}

hipError_t launch_bc_f(bgk_handle* h) { return launch_bc(h, true, false); }
hipError_t launch_bc_g(bgk_handle* h) { return launch_bc(h, false, true); }

hipError_t launch_streaming(bgk_handle* h) {
  hipLaunchKernelGGL(k_streaming, interior_grid(h->geom), dim3(TX, TY), 0, h->stream,
                     pairs(h->f[h->cur]), pairs(h->f[1 - h->cur]), h->geom);
  return hipGetLastError();
}

hipError_t launch_moments_pre(bgk_handle* h) {
  hipLaunchKernelGGL(k_moments_pre, interior_grid(h->geom), dim3(TX, TY), 0, h->stream,
                     pairs(h->f[1 - h->cur]), macro_of(h), h->geom);
  return hipGetLastError();
}

hipError_t launch_phase_field(bgk_handle* h) {
  const Geom& g = h->geom;
  const dim3 grd((unsigned)((g.nx + 2 + TX - 1) / TX), (unsigned)((g.ny + 2 + TY - 1) / TY));
  hipLaunchKernelGGL(k_phase_field, grd, dim3(TX, TY), 0, h->stream, h->phi[1 - h->pc],
                     h->phi[h->pc], h->T, h->c, g);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) h->pc = 1 - h->pc;
  return e;
}

hipError_t launch_forces(bgk_handle* h) {
  hipLaunchKernelGGL(k_forces, interior_grid(h->geom), dim3(TX, TY), 0, h->stream, macro_of(h),
                     h->phi[h->pc], h->phi[1 - h->pc], h->c, h->geom);
  return hipGetLastError();
}

hipError_t launch_collision(bgk_handle* h) {
  if (h->prm.rounding == BGK_ROUND_STEP7)
    hipLaunchKernelGGL(k_collision<true>, interior_grid(h->geom), dim3(TX, TY), 0, h->stream,
                       pairs(h->f[1 - h->cur]), pairs(h->f[h->cur]), macro_of(h), h->phi[h->pc],
                       h->c, h->geom);
  else
    hipLaunchKernelGGL(k_collision<false>, interior_grid(h->geom), dim3(TX, TY), 0, h->stream,
                       pairs(h->f[1 - h->cur]), pairs(h->f[h->cur]), macro_of(h), h->phi[h->pc],
                       h->c, h->geom);
  return hipGetLastError();
}

hipError_t launch_moments(bgk_handle* h) {
  hipLaunchKernelGGL(k_moments, interior_grid(h->geom), dim3(TX, TY), 0, h->stream,
                     pairs(h->f[h->cur]), macro_of(h), h->geom);
  return hipGetLastError();
}

}  // namespace bgk
