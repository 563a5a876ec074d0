// bgk_pop64.h -- the FP64 population step of one node, shared by the kernels that
// fuse it (bgk_fused.hip, bgk_stream64.hip).  For translation units compiled
// with -ffp-contract=off: operand for operand the reference's arithmetic.
#ifndef BGK_POP64_H
#define BGK_POP64_H

#include "bgk_wave.h"

namespace bgk {

using wave::Planes;

struct Done {
  double f[9], g[9], phi;
  double T2, u2, v2;  // momentsPre, for the averages
};

// momentsPre .. collision of one node (STEP_7/momentsPre.f90:8-21,
// phase_field.f90:24-52, forces.f90:18-26, collision.f90:14-150).
template <bool STEP7>
__device__ __forceinline__ Done node_step(const Consts& c, const double fp[9], const double gp[9],
                                          const double tap[9]) {
  Done o;
  const double rho = fp[0] + fp[1] + fp[2] + fp[3] + fp[4] + fp[5] + fp[6] + fp[7] + fp[8];
  double T = gp[0] + gp[1] + gp[2] + gp[3] + gp[4] + gp[5] + gp[6] + gp[7] + gp[8];
  const double irho = 1.0 / rho;
  double u = irho * (fp[1] - fp[3] + fp[5] - fp[6] - fp[7] + fp[8]);
  double v = irho * (fp[2] - fp[4] + fp[5] + fp[6] - fp[7] - fp[8]);
  o.T2 = T;
  o.u2 = u;
  o.v2 = v;
  o.phi = phase_update(c, T, tap);
  T = T - (c.dt_st * (o.phi - tap[0]) / 2.0);
  double fy = buoyancy(c, rho, T, o.phi);
  const double fx = -(u * (1.0 - o.phi) * 0.5);
  fy = fy - v * (1.0 - o.phi) * 0.5;
  u = u + fx / (c.omega_f * rho);
  v = v + fy / (c.omega_f * rho);
  regularised_bgk<STEP7>(c, c.omega_f, rho, u, v, fp, o.f);
  regularised_bgk<STEP7>(c, omega_g_at(c, o.phi), T, u, v, gp, o.g);
  return o;
}

struct Avg {
  double rho, T, u, v;
};
// STEP_7/moments.f90:11-25
__device__ __forceinline__ double averaged_T(const Done& o) {
  const double* g = o.g;
  const double tt = g[0] + g[1] + g[2] + g[3] + g[4] + g[5] + g[6] + g[7] + g[8];
  return (tt + o.T2) * 0.5;
}
__device__ __forceinline__ Avg averaged(const Done& o) {
  const double* f = o.f;
  Avg a;
  a.rho = f[0] + f[1] + f[2] + f[3] + f[4] + f[5] + f[6] + f[7] + f[8];
  const double irho = 1.0 / a.rho;
  const double tu = irho * (f[1] - f[3] + f[5] - f[6] - f[7] + f[8]);
  const double tv = irho * (f[2] - f[4] + f[5] + f[6] - f[7] - f[8]);
  a.T = averaged_T(o);
  a.u = (tu + o.u2) * 0.5;
  a.v = (tv + o.v2) * 0.5;
  return a;
}

// populations a row pulls
struct Row {
  double f[9], g[9];
};

// The populations of row j beside a wall, already pulled (population k of node
// (i - cx_k, j - cy_k)).  Sources outside the lattice are taken from the nearest
// column and row in it (right for g in the copied rows 0 and Ny+1); own: the
// node's own f, for the bounce-back (wall_f).  Every lane makes the same loads,
// all in flight at once.  offs: the byte offsets of columns i - 1, i, i + 1,
// each within 1..Nx.
struct EdgeRow {
  Row r;
  double own[9];
};
__device__ __forceinline__ void edge_offsets(int i, int nx, unsigned offs[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d)
    offs[d] = (unsigned)min(max(i + d - 1, 1), nx) * (unsigned)sizeof(double2);
}
__device__ __forceinline__ void load_pulled_edge(const Planes<double2>& A, int64_t pitch, int ny,
                                                 const unsigned offs[3], int j, EdgeRow& e) {
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int sj = min(max(j - CY[k], 1), ny);
    const double2 v = wave::at(A.row(k, (int64_t)sj * pitch), offs[1 - CX[k]]);
    e.r.f[k] = v.x;
    e.r.g[k] = v.y;
    if (k > 0) e.own[k] = wave::at(&A.row(k, (int64_t)j * pitch)->x, offs[1]);
  }
}

// Bounce-back (BC_f type 4): a population whose source is a ghost is the node's
// own opposite one, but for the two corner ghosts no BC_f branch writes.
__device__ __forceinline__ void wall_f(int nx, int ny, int i, int j, double frozen6,
                                       double frozen7, EdgeRow& e) {
#pragma unroll
  for (int k = 1; k < 9; ++k) {
    const bool row = (CY[k] > 0 && j == 1) || (CY[k] < 0 && j == ny);
    const bool col = (CX[k] > 0 && i == 1) || (CX[k] < 0 && i == nx);
    double b = e.own[OPP[k]];
    if (k == 6 && j == 1) b = i == nx ? frozen6 : b;
    if (k == 7 && j == ny) b = i == nx ? frozen7 : b;
    e.r.f[k] = row || col ? b : e.r.f[k];
  }
}

}  // namespace bgk

#endif  // BGK_POP64_H
