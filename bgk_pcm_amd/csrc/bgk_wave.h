// bgk_wave.h -- building blocks of the wave-streaming kernels: the steps of several
// levels per launch (bgk_stream_mom.hip, bgk_stream32.hip, bgk_stream64.hip) and the
// adjoint (bgk_adjoint.hip).
//
// One wavefront owns 64 neighbouring columns and walks up a strip of rows.
// Lane L holds column i0 - T + L of the row being processed, so a pull from
// the column to the west or east is a shift by one lane (v_mov_b32 with the
// DPP control wave_shr:1 / wave_shl:1, full rate, no LDS and no barrier), and
// a pull from the row below or above is a value kept in registers while the
// walk goes on.  A launch of T steps feeds each row through T levels: level t
// completes row r - t - 1 when row r arrives, and hands it to level t + 1 in
// the same iteration.  T lanes at each end of the wave and T rows at each end
// of a strip are recomputed by the neighbour, so HBM sees the state once in
// and once out per T steps.
#ifndef BGK_WAVE_H
#define BGK_WAVE_H

#include <algorithm>

#include "bgk_internal.h"

namespace bgk {
namespace wave {

constexpr int kLanes = 64;
constexpr int kDppShr1 = 0x138;  // lane L reads lane L - 1
constexpr int kDppShl1 = 0x130;  // lane L reads lane L + 1

// The value of the lane to the west (column i - 1); 0 in lane 0.
__device__ __forceinline__ double from_west(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kDppShr1, 0xf,
                                                            0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kDppShr1,
                                                            0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// The value of the lane to the east (column i + 1); 0 in lane 63.
__device__ __forceinline__ double from_east(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kDppShl1, 0xf,
                                                            0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kDppShl1,
                                                            0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float from_west(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                               kDppShr1, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_east(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                               kDppShl1, 0xf, 0xf, true));
}

// Buffer descriptor of n elements at p (wave-uniform), and a store of one
// element at offset q that the hardware drops where q >= n.  kPastStrip times
// an element's size (4 to 32 bytes) stays within 32 bits and past any strip
// (kMaxStrip elements, see make_wave_grid).  Where a row alone is more (wide_rows),
// the moment kernels count columns from the wave's first one.  The population
// kernels store row by row, elements of at most 16 bytes: row_buffer and kPastRow,
// just below 2^32 bytes, hold for any row that fits a device.
constexpr int kPastStrip = 0x07ffffff, kPastRow = -16;
constexpr int kMaxStrip = 0x03ffffff;
inline bool wide_rows(const bgk_handle* h) { return h->pitch > kMaxStrip; }
template <typename E>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t strip_buffer(E* p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, n * (int)sizeof(E), 0x00020000);
}
template <typename E>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(E* p, int64_t n) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)((unsigned)n * (unsigned)sizeof(E)),
                                           0x00020000);
}
constexpr int kCached = 0, kNonTemporal = 2;
template <int HOW = kNonTemporal, typename E>
__device__ __forceinline__ void buffer_put(__amdgpu_buffer_rsrc_t r, int q, const E& x) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const int off = (int)((unsigned)q * (unsigned)sizeof(E));
  if constexpr (sizeof(E) == 4) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, off, 0, HOW);
  } else if constexpr (sizeof(E) == 8) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, off, 0, HOW);
  } else if constexpr (sizeof(E) == 16) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, off, 0, HOW);
  } else {
    static_assert(sizeof(E) == 32, "element size");
    struct Two {
      u32x4 lo, hi;
    };
    const Two t = __builtin_bit_cast(Two, x);
    __builtin_amdgcn_raw_buffer_store_b128(t.lo, r, off, 0, HOW);
    __builtin_amdgcn_raw_buffer_store_b128(t.hi, r, off + 16, 0, HOW);
  }
}

// An element at a lane's 32-bit byte offset from a uniform address.
template <typename E>
__device__ __forceinline__ E at(const E* base, unsigned off) {
  return *reinterpret_cast<const E*>(reinterpret_cast<const char*>(base) + off);
}

// A copy of x in registers of its own, so that a load issued next can reuse
// x's (otherwise the compiler loads into others and moves them, with a wait,
// at the end of the loop).
__device__ __forceinline__ double taken(double x) {
  double y;
  asm("v_mov_b64 %0, %1" : "=v"(y) : "v"(x));
  return y;
}
__device__ __forceinline__ float taken(float x) {
  float y;
  asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
  return y;
}

// Nine pair planes at one spacing (a handle's planes of one buffer are carved
// alike).  A kernel forms a plane's row address where it uses it, from the
// row's: nine pointers or buffer descriptors held across the row loop spill
// scalar registers (100 of 720 instructions per row of the FP32 kernel).
template <typename P2>
struct Planes {
  P2* base;
  int64_t stride;  // pairs
  __device__ __forceinline__ P2* row(int k, int64_t q) const { return base + (q + k * stride); }
};
template <typename P2, typename E>
inline Planes<P2> planes_of(E* const* p) {
  P2* const b = reinterpret_cast<P2*>(p[0]);
  return Planes<P2>{b, reinterpret_cast<P2*>(p[1]) - b};
}

// s_waitcnt operand: all loads and stores done (vmcnt 0; the others free).  Set
// before a loop whose loads stay in flight across its back edge, so that the
// waits inside need not cover the loop's entry.
constexpr int kWaitLoads = 0x0f70;

// A read-only array through the scalar cache (uniform index).
typedef const __attribute__((address_space(4))) double* scalar_ptr;
__device__ __forceinline__ scalar_ptr as_scalar(const double* p) {
  return (scalar_ptr)(uintptr_t)p;
}

// Work split of a launch: column segments of `cols` output columns, and for
// each segment strips of rows, one wave (and workgroup) per strip.  Waves that
// meet a wall (the first segment, the last one or two, and the lowest and
// highest strip of the others) run the walls' code and take longer per row:
// their strips are shorter, and they are dispatched first, so that none of
// them is left when the others are done.
constexpr int kMaxRows = 64;
struct WaveGrid {
  int nseg, nright;  // segments; those that meet the east wall
  int ne;            // segments whose every strip runs the walls' code: 1 + nright, or all
  int re, nse;       // rows per strip of those, strips
  int ra;            // rows of the lowest and highest strip of the others
  int rows, nmid;    // rows per strip between them, strips
  int nedge;         // workgroups of the walls
  int nwg;           // all, the others padded to a multiple of 8 (the XCDs)
};

// Segment and rows j0..j1 of this workgroup; false for the padding.  Workgroup
// b runs on XCD b % 8: of the strips away from the walls each XCD takes a
// contiguous run of (strip, segment) pairs, so the columns and rows that
// neighbours share are hits in its L2.
__device__ __forceinline__ bool wave_tile(const WaveGrid& g, int ny, int* seg, int* j0, int* j1,
                                          bool* edge) {
  int b = (int)blockIdx.x;
  *edge = b < g.nedge;
  if (*edge) {
    if (b < g.ne * g.nse) {
      const int e = b % g.ne;
      *seg = e == 0 ? 0 : g.nseg - g.ne + e;
      *j0 = b / g.ne * g.re + 1;
      *j1 = min(*j0 + g.re - 1, ny);
    } else {
      b -= g.ne * g.nse;
      *seg = 1 + b / 2;
      *j0 = b % 2 == 0 ? 1 : ny - g.ra + 1;
      *j1 = *j0 + g.ra - 1;
    }
    return true;
  }
  b -= g.nedge;
  const int inner = g.nseg - g.ne, per = (g.nwg - g.nedge) / NXCD;
  const int k = b % NXCD * per + b / NXCD;
  *seg = 1 + k % inner;
  *j0 = g.ra + 1 + k / inner * g.rows;
  *j1 = min(*j0 + g.rows - 1, ny - g.ra);
  return k / inner < g.nmid;
}

// The split with strips of h rows (walls: of equal duration, at `slow` times
// the cost per row iteration).  A strip of h rows takes h + extra iterations.
// most: the rows that a strip may have; where the T + 1 rows that keep the others
// off the walls are more, every strip runs the walls' code.
inline WaveGrid split_waves(int nx, int ny, int cols, int T, int extra, double slow, int h,
                            int most) {
  WaveGrid g{};
  g.nseg = (nx + cols - 1) / cols;
  const int last = nx - (g.nseg - 1) * cols;  // columns of the last segment
  g.nright = last <= T ? 2 : 1;
  g.re = std::max(1, std::min({ny, h, (int)((h + extra) / slow) - extra}));
  g.ra = std::max(g.re, T + 1);
  g.ne = g.nseg <= 1 + g.nright || ny <= 2 * g.ra || g.ra > most ? g.nseg : 1 + g.nright;
  g.nse = (ny + g.re - 1) / g.re;
  g.rows = h;
  const int64_t inner = g.nseg - g.ne;
  g.nmid = inner > 0 ? (ny - 2 * g.ra + h - 1) / h : 0;
  g.nedge = (int)((int64_t)g.ne * g.nse + 2 * inner);
  g.nwg = g.nedge + (int)((inner * g.nmid + NXCD - 1) / NXCD * NXCD);
  return g;
}

// The strip height, 1..most, by a model of the launch.  Up to one wave per SIMD
// (4 n_cu) all run at once at full speed; two waves on a SIMD slow each other
// by 1.2 to 1.6 (measured, large to small lattices); beyond 8 n_cu waves (4
// n_cu where the registers hold one wave, `deep` = 1) the launch takes its work
// at that rate, plus half a strip for the last waves.  Taller strips repeat
// fewer rows.  rows_override > 0 fixes the height.
inline WaveGrid make_wave_grid(int nx, int ny, int cols, int T, int extra, double slow, int most,
                               int n_cu, int rows_override, int deep = 2) {
  // (offsets within a strip stay below kMaxStrip elements)
  const int room = (int)std::max((int64_t)1, kMaxStrip / ((int64_t)nx + 256));
  most = std::min({most, ny, kMaxRows, room});
  if (rows_override > 0)
    return split_waves(nx, ny, cols, T, extra, slow, std::min(rows_override, most), room);
  WaveGrid best{};
  double cost = -1.0;
  for (int h = 1; h <= most; ++h) {
    const WaveGrid g = split_waves(nx, ny, cols, T, extra, slow, h, room);
    const double inner = g.nseg - g.ne, slots = 4.0 * deep * n_cu;
    const double shared = deep > 1 ? 1.35 : 1.0;
    const double waves = g.nedge + inner * g.nmid;
    const double te = slow * (std::max(g.re, inner > 0 ? g.ra : 0) + extra);
    const double longest = std::max(te, g.nmid > 0 ? (double)(h + extra) : 0.0);
    const double work = slow * ((double)g.ne * g.nse * (g.re + extra) + 2 * inner * (g.ra + extra)) +
                        inner * g.nmid * (h + extra);
    const double c = waves <= 4.0 * n_cu ? longest
                     : waves <= slots      ? shared * longest
                                           : shared * (work / slots + 0.5 * longest);
    if (cost < 0.0 || c < cost) {
      cost = c;
      best = g;
    }
  }
  return best;
}

}  // namespace wave
}  // namespace bgk

#endif  // BGK_WAVE_H
