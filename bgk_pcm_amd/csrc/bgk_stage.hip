// bgk_stage.hip -- one kernel (or kernel pair) per reference subroutine.
//
// This is the per-subroutine path of the drop-in boundary: bgk_bc_f,
// bgk_bc_g, bgk_streaming, ... each launch the kernels below on the handle's
// stream, on the same fields the reference's `module shared` holds.  It
// serves every boundary type of the reference; bgk_step takes its boundary
// launch when the walls are not all no-slip.  Compiled with -ffp-contract=off: the
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
// by subroutines, us, before and after pairs, one boundary launch each and no
// copy of phi: 64^2 40 / 31, 512^2 90 / 65, 1024 x 512 151 / 106, 2048 x 1024
// 610 / 462.
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
// Each routine below reads everything first and writes after: the planes may
// alias for all the compiler knows, and a load behind a store waits for both
// (channel 1024 x 512, us per step: 75 interleaved, 71 so).

// The equilibria of directions a, b, d (one side's) for density r and velocity
// (u, v), in the operand order of BC_f.f90.
struct Three {
  double a, b, d;
};
__device__ __forceinline__ Three west_eq(const Consts& c, double r, double u, double v) {
  const double uu = u * u, vv = v * v, uv = 1.5 * (uu + vv), upv = u + v, umv = u - v;
  return Three{c.w[1] * r * (1.0 + 3.0 * u + 4.5 * uu - uv),
               c.w[5] * r * (1.0 + 3.0 * upv + 4.5 * upv * upv - uv),
               c.w[8] * r * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv)};
}
__device__ __forceinline__ Three east_eq(const Consts& c, double r, double u, double v) {
  const double uu = u * u, vv = v * v, uv = 1.5 * (uu + vv), upv = u + v, umv = u - v;
  return Three{c.w[3] * r * (1.0 - 3.0 * u + 4.5 * uu - uv),
               c.w[6] * r * (1.0 - 3.0 * umv + 4.5 * umv * umv - uv),
               c.w[7] * r * (1.0 - 3.0 * upv + 4.5 * upv * upv - uv)};
}
__device__ __forceinline__ Three north_eq(const Consts& c, double r, double u, double v) {
  const double uu = u * u, vv = v * v, uv = 1.5 * (uu + vv), upv = u + v, umv = u - v;
  return Three{c.w[4] * r * (1.0 - 3.0 * v + 4.5 * vv - uv),
               c.w[7] * r * (1.0 - 3.0 * upv + 4.5 * upv * upv - uv),
               c.w[8] * r * (1.0 + 3.0 * umv + 4.5 * umv * umv - uv)};
}

// West and east sides, row j = 0..Ny+1 (STEP_7/BC_f.f90:9-104).
__device__ __forceinline__ void bc_f_we(const Pops64& F, const Macro& m, const Consts& c,
                                        const Geom& gm, const Walls& w, int j) {
  const int nx = gm.nx, ny = gm.ny, wbc = w.west, ebc = w.east;
  const int64_t P = gm.pitch;
  auto at = [&](int i, int jj) { return (int64_t)jj * P + i; };
  const Strided2<double>* f = F.p;
  const bool inner = (j >= 1 && j <= ny);
  // ---- read
  double fw[9], fe[9];  // periodic
  Three w3{}, e3{};     // directions 1, 5, 8 of the west, 3, 6, 7 of the east
  double ru = 0.0, rv = 0.0, rr = 0.0, eu = 0.0, ev = 0.0;
  if (wbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) fw[k] = f[k][at(nx, j)];
  } else if (wbc == 1) {
    if (inner) {
      rr = m.rho[at(1, j)];
      ru = c.u0;
      rv = c.v0;
      w3 = west_eq(c, rr, ru, rv);
    }
  } else if (wbc == 2) {
    w3 = west_eq(c, m.rho[at(1, j)], m.u[at(0, j)], c.v0);
  } else if (wbc == 3) {
    ru = m.u[at(1, j)];
    rv = m.v[at(1, j)];
    rr = c.rho1;
    w3 = west_eq(c, rr, ru, rv);
  } else if (wbc == 4) {
    if (inner) w3 = Three{f[3][at(1, j)], f[7][at(1, j + 1)], f[6][at(1, j - 1)]};
  }
  if (ebc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) fe[k] = f[k][at(1, j)];
  } else if (ebc == 3) {
    if (inner) {
      eu = m.u[at(nx, j)];
      ev = m.v[at(nx, j)];
      e3 = east_eq(c, c.rho0, eu, ev);
    }
  } else if (ebc == 4) {
    if (inner) e3 = Three{f[1][at(nx, j)], f[8][at(nx, j + 1)], f[5][at(nx, j - 1)]};
  }
  // ---- write
  if (wbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][at(0, j)] = fw[k];
  } else if (wbc == 2 || wbc == 3 || inner) {
    f[1][at(0, j)] = w3.a;
    f[5][at(0, j)] = w3.b;
    f[8][at(0, j)] = w3.d;
    if (wbc == 1 || wbc == 3) {
      m.u[at(0, j)] = ru;
      m.v[at(0, j)] = rv;
      m.rho[at(0, j)] = rr;
    }
  }
  if (ebc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][at(nx + 1, j)] = fe[k];
  } else if (inner) {
    f[3][at(nx + 1, j)] = e3.a;
    f[6][at(nx + 1, j)] = e3.b;
    f[7][at(nx + 1, j)] = e3.d;
    if (ebc == 3) {
      m.u[at(nx + 1, j)] = eu;
      m.v[at(nx + 1, j)] = ev;
      m.rho[at(nx + 1, j)] = c.rho0;
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
  // ---- read
  double fn[9], fs[9];  // periodic
  Three n3{}, s3{};     // directions 4, 7, 8 of the north, 2, 5, 6 of the south
  double nr = 0.0, sr = 0.0;
  if (nbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) fn[k] = f[k][at(i, 1)];
  } else if (nbc == 4) {
    if (inner) {
      n3 = Three{f[2][at(i, ny)], f[5][at(i - 1, ny)], f[6][at(i + 1, ny)]};
      nr = m.rho[at(i, ny)];
    }
    if (i == 0) n3.d = f[6][at(1, ny)];
  } else if (nbc == 5) {
    n3 = Three{f[2][at(i, ny - 1)], f[6][at(i, ny - 1)], f[5][at(i, ny - 1)]};
  } else if (nbc == 6) {
    n3 = Three{f[4][at(i, ny)], f[7][at(i, ny)], f[8][at(i, ny)]};
  } else if (nbc == 1) {
    n3 = north_eq(c, m.rho[at(i, ny)], c.u0, c.v0);
  }
  if (sbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) fs[k] = f[k][at(i, ny)];
  } else if (sbc == 4) {
    if (inner) {
      s3 = Three{f[4][at(i, 1)], f[7][at(i + 1, 1)], f[8][at(i - 1, 1)]};
      sr = m.rho[at(i, 1)];
    }
    if (i == 0) s3.b = f[7][at(1, 1)];
  } else if (sbc == 6) {
    s3 = Three{f[2][at(i, 1)], f[5][at(i, 1)], f[6][at(i, 1)]};
  }
  // ---- write
  const int64_t n = at(i, ny + 1), s = at(i, 0);
  if (nbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][n] = fn[k];
  } else if (nbc == 4) {
    if (inner) {
      f[4][n] = n3.a;
      f[7][n] = n3.b;
      m.rho[n] = nr;
      m.u[n] = 0.0;
      m.v[n] = 0.0;
    }
    if (inner || i == 0) f[8][n] = n3.d;
  } else {
    f[4][n] = n3.a;
    f[7][n] = n3.b;
    f[8][n] = n3.d;
  }
  if (sbc == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k][s] = fs[k];
  } else if (sbc == 4) {
    if (inner) {
      f[2][s] = s3.a;
      f[6][s] = s3.d;
      m.rho[s] = sr;
      m.u[s] = 0.0;
      m.v[s] = 0.0;
    }
    if (inner || i == 0) f[5][s] = s3.b;
  } else {
    f[2][s] = s3.a;
    f[5][s] = s3.b;
    f[6][s] = s3.d;
  }
}

// ----------------------------------------------------------------------- BC_g
// West and east, row j = 1..Ny (STEP_7/BC_g.f90:9-31).
__device__ __forceinline__ void bc_g_we(const Pops64& G, const Macro& m, const Consts& c,
                                        const Geom& gm, int j) {
  const int nx = gm.nx;
  const int64_t w = (int64_t)j * gm.pitch, e = w + nx + 1;
  const Strided2<double>* g = G.p;
  const double uw = m.u[w], vw = m.v[w], ue = m.u[e], ve = m.v[e];
  // the averaged T(Nx, j), or the cold-wall extension's fixed temperature
  const double te = c.east_cold ? c.t_cold : m.T[w + nx];
  const Three w3 = west_eq(c, c.tin, uw, vw), e3 = east_eq(c, te, ue, ve);
  g[1][w] = w3.a;
  g[5][w] = w3.b;
  g[8][w] = w3.d;
  m.T[w] = c.tin;
  g[3][e] = e3.a;
  g[6][e] = e3.b;
  g[7][e] = e3.d;
  m.T[e] = te;
}

// North and south zero-gradient copies, column i = 0..Nx+1
// (STEP_7/BC_g.f90:36-64), after bc_g_we.
__device__ __forceinline__ void bc_g_ns(const Pops64& G, const Macro& m, double* phi,
                                        const Geom& gm, int i) {
  const int64_t P = gm.pitch;
  const int64_t qn = (int64_t)gm.ny * P + i, q1 = P + i;
  double gn[9], gs[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    gn[k] = G.p[k][qn];
    gs[k] = G.p[k][q1];
  }
  const double tn = m.T[qn], ts = m.T[q1], pn = phi[qn], ps = phi[q1];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    G.p[k][qn + P] = gn[k];
    G.p[k][i] = gs[k];
  }
  m.T[qn + P] = tn;
  m.T[i] = ts;
  phi[qn + P] = pn;
  phi[i] = ps;
}

// BC_f and/or BC_g in one launch.  The sides depend on each other in the
// reference's order (west and east, then north and south; f before g), but
// only in the columns 0, 1, Nx, Nx+1 and the rows 0, 1, Ny-1, Ny, Ny+1: the first
// workgroup does these (each once, where they coincide), waiting between the four
// parts; every other row of the west and east and column of the north and south
// is a thread of its own elsewhere, f before g.
// What bounds it: the latency of a launch and of a few dependent accesses.
// Measured, us per step of a channel (this launch and k_general64): 2048 x 1024
// 186 with one workgroup for all, 132 so; 1024 x 512 71 / 48; 64^2 13.3 / 12.8.
constexpr int kBcThreads = 256;
struct BcArgs {
  Pops64 F, G;
  Macro m;
  double* phi;
  Consts c;
  Geom gm;
  Walls w;
  int do_f, do_g;
};
__global__ __launch_bounds__(kBcThreads) void k_bc(BcArgs a) {
  const int nx = a.gm.nx, ny = a.gm.ny;
  if (blockIdx.x > 0) {
    int t = ((int)blockIdx.x - 1) * kBcThreads + (int)threadIdx.x;
    const int rows = max(ny - 3, 0);
    if (t < rows) {
      const int j = t + 2;  // 2..Ny-2
      if (a.do_f) bc_f_we(a.F, a.m, a.c, a.gm, a.w, j);
      if (a.do_g) bc_g_we(a.G, a.m, a.c, a.gm, j);
    } else if ((t -= rows) < nx - 2) {
      const int i = t + 2;  // 2..Nx-1
      if (a.do_f) bc_f_ns(a.F, a.m, a.c, a.gm, a.w, i);
      if (a.do_g) bc_g_ns(a.G, a.m, a.phi, a.gm, i);
    }
    return;
  }
  // this thread's row (0, 1, Ny-1..Ny+1) and column (0, 1, Nx, Nx+1) of the first
  // workgroup; -1: none
  const int e = (int)threadIdx.x;
  const int row = e < 2 ? e : e < 5 && ny - 3 + e > 1 ? ny - 3 + e : -1;
  const int col = e < 2 ? e : e < 4 && nx - 2 + e > 1 ? nx - 2 + e : -1;
  if (a.do_f) {
    if (row >= 0) bc_f_we(a.F, a.m, a.c, a.gm, a.w, row);
    __syncthreads();
    if (col >= 0) bc_f_ns(a.F, a.m, a.c, a.gm, a.w, col);
    __syncthreads();
  }
  if (a.do_g) {
    if (row >= 1 && row <= ny) bc_g_we(a.G, a.m, a.c, a.gm, row);
    __syncthreads();
    if (col >= 0) bc_g_ns(a.G, a.m, a.phi, a.gm, col);
  }
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
  // rows 2..Ny-2 and columns 2..Nx-1
  const unsigned rest = blocks1d(std::max(g.ny - 3, 0) + std::max(g.nx - 2, 0), kBcThreads);
  hipLaunchKernelGGL(k_bc, dim3(1 + rest), dim3(kBcThreads), 0, h->stream, a);
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
  const bool copy = h->recorded;  // (the exchange would change the buffers)
  if (copy) {
    const hipError_t e = launch_copy64(h, h->phi[h->pc], 1, h->phi[1 - h->pc], 1);
    if (e != hipSuccess) return e;
  }
  const int to = copy ? h->pc : 1 - h->pc;
  hipLaunchKernelGGL(k_phase_field, grd, dim3(TX, TY), 0, h->stream, h->phi[to], h->phi[1 - to],
                     h->T, h->c, g);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) h->pc = to;
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

hipError_t launch_stages64(bgk_handle* h) {
  for (const auto launch : {launch_bc_f, launch_bc_g, launch_streaming, launch_moments_pre,
                            launch_phase_field, launch_forces, launch_collision, launch_moments}) {
    const hipError_t e = launch(h);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace bgk
