// Lid-driven cavity flow of npbench's cavity_flow
// (npbench/benchmarks/cavity_flow/cavity_flow_numpy.py:13-83), FP64, bitwise
// the NumPy reference.
//
// A time step is a chain of whole-grid phases -- build b; nit pressure-Poisson
// Jacobi iterations; update u, v -- on grids of ~10^4 points (the paper preset
// is 101 x 101 with 700 steps of 50 iterations: 37,000 phases).  A launch per
// phase would be bound by launches, so two forms cut their number:
//
// * cavity_pressure advances the pressure by up to kMaxDepth iterations per
//   launch (temporal blocking): a workgroup holds its block and a halo of one
//   cell per iteration in registers, so it needs nothing from other
//   workgroups until the launch ends; cavity_velocity does the velocity update
//   of one step and the source of the next in one launch.  A step of 20
//   iterations is 2 launches spread over the chip.
// * cavity_flow_lds runs every phase of the call in one workgroup with a
//   barrier between phases, both pressure buffers in LDS and b in registers:
//   no launches, but one CU.  It stays for the small grids where a phase
//   costs less than its share of a launch (use_lds below).
//
// Divisions are by five uniform divisors whose reciprocals are prepared once
// (division.h).  b needs no zeroing: only its interior is read, and each step
// writes it first.
//
// The four boundary statements after each iteration (:30-33), applied in the
// reference's order, leave row 0, column 0 and column nx-1 equal to this
// iteration's interior next to them (the corners (0,0) and (0,nx-1) take
// (1,1) and (1,nx-2)) and the last row 0.  So whoever computes an interior
// point next to one of those edges also knows the edge's value, and an
// iteration is a single phase.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "common.h"
#include "division.h"
#include "lanes.h"

namespace npbx {
namespace {

constexpr int kThreadsC = 1024;
constexpr int kLdsPoints = 10240;  // two FP64 pressure buffers: all 160 KiB of LDS

// The reference's scalar expressions, computed on the host as Python computes
// them (x**2 is the C library's pow, which CPython's float power calls).
struct CavityArgs {
  double* u;
  double* v;
  double* p;
  double* un;
  double* vn;
  double* pn;
  double* b;
  int nx, ny, nt, nit;
  double rho, nu;
  double inv_dt;    // 1 / dt
  double two_dx;    // 2 * dx
  double two_dy;    // 2 * dy
  double dx2, dy2;  // dx**2, dy**2
  double den;       // 2 * (dx**2 + dy**2)
  double cb;        // dx**2 * dy**2 / (2 * (dx**2 + dy**2))
  double dt, dx, dy;
  double cpu;       // dt / (2 * rho * dx)
  double cpv;       // dt / (2 * rho * dy)
  double cdx2;      // dt / dx**2
  double cdy2;      // dt / dy**2
};

// The kernel's divisors, prepared once per launch and held in scalar
// registers: every division of the time step is by one of them.  Only their
// reciprocals and one common no-rescale range of |m| stay live, so the
// kernel's uniform values fit the scalar register file.
struct CavityDivisors {
  Divisor den, two_dx, two_dy, dx, dy;
  double lo, hi;  // |m| in [lo, hi) for every division of a chunk: exact
};

// Walks this thread's interior points k = t, t + kThreadsC, ... in row-major
// order of the (ny-2) x (nx-2) interior without a division per point, C
// points at a time: f receives their flat grid indices a, edge flags and
// validity (past the end, a is a safe interior index to read, not to write).
// Handing a chunk to f at once lets it issue every load of the chunk before
// its first store, so the loads' latencies overlap.
enum : int { kRow1 = 1, kCol1 = 2, kColLast = 4 };  // interior row 0, column 0, column w-1

struct InteriorWalk {
  int i0, j0, si, sj, w, h, nx;
  __device__ InteriorWalk(int t, int nx_, int ny_) : nx(nx_) {
    w = nx_ - 2;
    h = ny_ - 2;
    i0 = t / w;
    j0 = t - i0 * w;
    si = kThreadsC / w;
    sj = kThreadsC - si * w;
  }
  template <int C, class F>
  __device__ __forceinline__ void each(F&& f) const {
    int i = i0, j = j0;
    while (i < h) {
      int a[C], fl[C];
      bool ok[C];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        ok[c] = i < h;
        a[c] = ok[c] ? (i + 1) * nx + j + 1 : nx + 1;
        fl[c] = (i == 0 ? kRow1 : 0) | (j == 0 ? kCol1 : 0) | (j == w - 1 ? kColLast : 0);
        i += si;
        j += sj;
        if (j >= w) {
          j -= w;
          ++i;
        }
      }
      f(a, fl, ok);
    }
  }
};

constexpr int kChunkV = 2;  // velocity points per chunk (14 loads each)
constexpr int kMaxPts = 4;  // most interior points per thread, in the one-workgroup form

// The point computations take their division as a policy (ShortDiv or
// FullDiv, run by chunk_eval).

// build_up_b (:13-21) from the velocities east, west, north (row + 1) and
// south (row - 1) of a point.
template <class Div>
__device__ __forceinline__ double source_from(const CavityArgs& g, const CavityDivisors& dv,
                                              double ue, double uw, double un, double us,
                                              double ve, double vw, double vn, double vs,
                                              Div& div) {
  const double dudx = div(ue - uw, dv.two_dx);
  const double dvdy = div(vn - vs, dv.two_dy);
  const double t1 = g.inv_dt * (dudx + dvdy);
  const double t2 = dudx * dudx;
  const double t3 = 2.0 * div(div(un - us, dv.two_dy) * (ve - vw), dv.two_dx);
  const double t4 = dvdy * dvdy;
  return g.rho * (((t1 - t2) - t3) - t4);
}

// The same at interior point x of the fields.
template <class Div>
__device__ __forceinline__ double source_at(const CavityArgs& g, const CavityDivisors& dv, int x,
                                            Div& div) {
  const int nx = g.nx;
  const double* u = g.u;
  const double* v = g.v;
  return source_from(g, dv, u[x + 1], u[x - 1], u[x + nx], u[x - nx], v[x + 1], v[x - 1],
                     v[x + nx], v[x - nx], div);
}

// One pressure iterate (:30-33) at interior point x, with b there.
template <class P, class Div>
__device__ __forceinline__ double pressure_at(const CavityArgs& g, const CavityDivisors& dv,
                                              const P* src, int x, double bx, Div& div) {
  const int nx = g.nx;
  return div((src[x + 1] + src[x - 1]) * g.dy2 + (src[x + nx] + src[x - nx]) * g.dx2, dv.den) -
         g.cb * bx;
}

// Stores an iterate at interior point x and, for points next to the edges,
// the copies the boundary statements (:35-37) make of it.
template <class P>
__device__ __forceinline__ void store_pressure(P* dst, int x, int fl, int nx, double val) {
  dst[x] = val;
  if (!fl) return;                                // most points have no edge copy
  if (fl & kRow1) dst[x - nx] = val;              // row 0 = row 1
  if (fl & kCol1) {
    dst[x - 1] = val;                             // column 0 = column 1
    if (fl & kRow1) dst[x - nx - 1] = val;        // corner (0,0) = (1,1)
  }
  if (fl & kColLast) {
    dst[x + 1] = val;                             // column nx-1 = column nx-2
    if (fl & kRow1) dst[x - nx + 1] = val;        // corner (0,nx-1) = (1,nx-2)
  }
}

// u and v (:53-73) at interior point x from un, vn and the pressure p.
template <class P, class Div>
__device__ __forceinline__ void velocity_at(const CavityArgs& g, const CavityDivisors& dv,
                                            const P* p, int x, double& nu, double& nv, Div& div) {
  const int nx = g.nx;
  const double* un = g.un;
  const double* vn = g.vn;
  const double uc = un[x], vc = vn[x];
  const double udx = div(uc * g.dt, dv.dx);  // un * dt / dx
  const double vdy = div(vc * g.dt, dv.dy);  // vn * dt / dy
  const double x1 = udx * (uc - un[x - 1]);
  const double x2 = vdy * (uc - un[x - nx]);
  const double x3 = g.cpu * (p[x + 1] - p[x - 1]);
  const double x4 = g.nu * (g.cdx2 * (un[x + 1] - 2.0 * uc + un[x - 1]) +
                            g.cdy2 * (un[x + nx] - 2.0 * uc + un[x - nx]));
  nu = ((uc - x1 - x2) - x3) + x4;
  const double y1 = udx * (vc - vn[x - 1]);
  const double y2 = vdy * (vc - vn[x - nx]);
  const double y3 = g.cpv * (p[x + nx] - p[x - nx]);
  const double y4 = g.nu * (g.cdx2 * (vn[x + 1] - 2.0 * vc + vn[x - 1]) +
                            g.cdy2 * (vn[x + nx] - 2.0 * vc + vn[x - nx]));
  nv = ((vc - y1 - y2) - y3) + y4;
}

// The velocity boundary conditions (:75-82): the lid row is 1, corners
// included, every other edge point 0.
__device__ __forceinline__ void velocity_boundaries(const CavityArgs& g, int t) {
  const int nx = g.nx, ny = g.ny;
  for (int k = t; k < 2 * nx + 2 * ny; k += kThreadsC) {
    int a;
    if (k < nx) a = k;                                    // row 0
    else if (k < 2 * nx) a = (ny - 1) * nx + (k - nx);    // row ny-1
    else if (k < 2 * nx + ny) a = (k - 2 * nx) * nx;      // column 0
    else a = (k - 2 * nx - ny) * nx + nx - 1;             // column nx-1
    g.u[a] = a >= (ny - 1) * nx ? 1.0 : 0.0;
    g.v[a] = 0.0;
  }
}

// un = u.copy(); vn = v.copy() (:47-48), loads ahead of stores.
__device__ __forceinline__ void copy_velocities(const CavityArgs& g, int t, int np) {
  constexpr int U = 4;
  for (int k0 = t; k0 < np; k0 += U * kThreadsC) {
    double uu[U], vv[U];
#pragma unroll
    for (int c = 0; c < U; ++c) {
      const int k = min(k0 + c * kThreadsC, np - 1);
      uu[c] = g.u[k];
      vv[c] = g.v[k];
    }
#pragma unroll
    for (int c = 0; c < U; ++c) {
      const int k = k0 + c * kThreadsC;
      if (k < np) {
        g.un[k] = uu[c];
        g.vn[k] = vv[c];
      }
    }
  }
}

__device__ __forceinline__ CavityDivisors cavity_divisors(const CavityArgs& g) {
  double lo = 0.0, hi = INFINITY;
  CavityDivisors dv;
  dv.den = prepare_divisor(g.den, lo, hi);
  dv.two_dx = prepare_divisor(g.two_dx, lo, hi);
  dv.two_dy = prepare_divisor(g.two_dy, lo, hi);
  dv.dx = prepare_divisor(g.dx, lo, hi);
  dv.dy = prepare_divisor(g.dy, lo, hi);
  dv.lo = uniform_double(lo);
  dv.hi = uniform_double(hi);
  return dv;
}

// ---- blocked form: a chip-wide launch per group of pressure iterations -----
//
// cavity_pressure<R>: 16 waves stacked along y, each holding R rows x 64
// columns of p and cb b in registers (one column per lane).  A workgroup
// advances its region `depth` iterations; next to other blocks the outer
// `depth` cells are halo, computed redundantly and one cell less valid per
// iteration; at the grid's edges the region ends with the interior, where the
// edge points hold copies of their interior neighbours (the last row: 0) and
// need no registers.  West and east are the adjacent lanes (DPP shifts; the
// outer lanes get themselves back, which at the grid's edge is the copy),
// north and south the wave's own rows, the two edge rows of a wave go through
// LDS (one barrier per iteration).  So every block runs the same code.  Only
// an iteration from memory reads the stored edge (the first of a call may
// hold anything there): its outer neighbours are loaded beside the region.
// NARROW: grids narrower than a region (fewer than 64 interior columns or
// 16 R rows), where the edges fall inside it and are selected per point.
//
// The division by den is the short form with its residual negated twice
// (r = fma(den, m, -n), q = fma(-r, y, m)): the same value, and for n = +-0
// the quotient keeps n's sign, so exact zeros -- a flow at rest has many --
// need no fallback.  It is exact where nothing in the IEEE sequence rescales:
// den in [2^-100, 2^100] and every n zero or of magnitude 2^-900 .. 2^300.
// The upper side is checked once: |p|, |cb b| < 2^100 on load bound every
// iterate by 2^100 (1 + depth) and rounding, because an iterate's weights sum
// to one.  The lower side is the smallest exponent of n over all iterations
// (frexp gives 0 for n = 0).  A workgroup that leaves the range anywhere
// starts over from global memory with the division operator.
//
// Bound by FP64 issue and the exchange: 15 VALU instructions per point and
// iteration at four cycles each (9 arithmetic, 4 lane shifts, 1.5 for the
// range), then the waves' common wait for LDS and the barrier.  201 x 201,
// 20 iterations in one launch of 140 blocks: 14.2 us (0.6 us an iteration;
// one workgroup for the whole grid took 33 us).  Sixteen waves of 3 rows
// measured faster than eight of 6 or four of 12 (1.86, 1.92, 2.04 ms for 100
// steps): more waves hide more of the shifts' and LDS latencies than the
// smaller exchange saves.
constexpr int kWavesP = 16;
constexpr int kMaxDepth = 24;
constexpr int kMinExpN = -898;  // |n| >= 2^-899

struct PressureDiv {  // den, its reciprocal
  double d, y;
};

template <bool FULL>
__device__ __forceinline__ double pressure_quotient(double n, const PressureDiv& v, int& emin) {
  if constexpr (FULL) {
    return n / v.d;
  } else {
    emin = min(emin, __builtin_amdgcn_frexp_exp(n));
    const double m = n * v.y;
    const double r = __builtin_fma(v.d, m, -n);
    return __builtin_fma(-r, v.y, m);
  }
}

// One iteration of the wave's rows x into y (:30-37): ring[r] holds the
// values west of lane 0 and east of lane 63, `top` and `bottom` the rows
// outside the region (waves 0 and 15).
template <int R, bool NARROW, bool FULL>
__device__ __forceinline__ void pressure_step(const double (&x)[R], double (&y)[R],
                                              const double (&bb)[R], const double (&ring)[R],
                                              double top, double bottom, double (*edge)[2][64],
                                              int lane, int w, int gi0, int gj,
                                              const CavityArgs& g, const PressureDiv& v,
                                              bool settled, int& emin) {
  edge[w][0][lane] = x[0];
  edge[w][1][lane] = x[R - 1];
  __syncthreads();
  double above = edge[max(w - 1, 0)][1][lane];
  double below = edge[min(w + 1, kWavesP - 1)][0][lane];
  if (w == 0) above = top;
  if (w == kWavesP - 1) below = bottom;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const double c = x[r];
    double north = r == 0 ? above : x[r - 1];
    double south = r == R - 1 ? below : x[r + 1];
    double west = lane_from_left_or(ring[r], c), east = lane_from_right_or(ring[r], c);
    if constexpr (NARROW) {
      west = settled && gj == 1 ? c : west;
      east = settled && gj == g.nx - 2 ? c : east;
      if (settled && gi0 + r == 1) north = c;
      if (settled && gi0 + r == g.ny - 2) south = 0.0;
    }
    const double n = (east + west) * g.dy2 + (south + north) * g.dx2;
    y[r] = pressure_quotient<FULL>(n, v, emin) - bb[r];
  }
}

template <int R, bool NARROW, bool FULL>
__device__ __forceinline__ void pressure_steps(double (&x)[R], const double (&bb)[R],
                                               const double (&ring)[R], double top, double bottom,
                                               double (*edge)[kWavesP][2][64], int lane, int w,
                                               int gi0, int gj, const CavityArgs& g,
                                               const PressureDiv& v, int depth, int& emin) {
  double y[R];
  pressure_step<R, NARROW, FULL>(x, y, bb, ring, top, bottom, edge[0], lane, w, gi0, gj, g, v,
                                 false, emin);
  int k = 1;
  for (; k + 2 <= depth; k += 2) {
    pressure_step<R, NARROW, FULL>(y, x, bb, y, y[0], 0.0, edge[1], lane, w, gi0, gj, g, v, true,
                                   emin);
    pressure_step<R, NARROW, FULL>(x, y, bb, x, x[0], 0.0, edge[0], lane, w, gi0, gj, g, v, true,
                                   emin);
  }
  if (k < depth) {
    pressure_step<R, NARROW, FULL>(y, x, bb, y, y[0], 0.0, edge[1], lane, w, gi0, gj, g, v, true,
                                   emin);
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = y[r];
  }
}

template <int R, bool NARROW>
__global__ __launch_bounds__(64 * kWavesP) void cavity_pressure(CavityArgs g,
                                                                const double* __restrict__ src,
                                                                double* __restrict__ dst,
                                                                int depth, int tiles_x,
                                                                int tiles_y) {
  __shared__ double edge[2][kWavesP][2][64];
  const int lane = threadIdx.x % 64;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int nx = g.nx, ny = g.ny;
  const Span sx = span_of(blockIdx.x % tiles_x, tiles_x, nx - 2, 64, depth);
  const Span sy = span_of(blockIdx.x / tiles_x, tiles_y, ny - 2, R * kWavesP, depth);
  const int gj = sx.origin + lane, gi0 = sy.origin + w * R;
  const PressureDiv v{g.den, uniform_double(division_reciprocal(g.den))};
  const bool den_ok = g.den >= 0x1p-100 && g.den <= 0x1p100;

  // p clamped into the grid, cb b into the interior: every load lands on a
  // value that exists (clamped ones only in a NARROW grid's unused rows and
  // lanes)
  double x[R], bb[R], ring[R], top, bottom;
  const int gjp = min(gj, nx - 1), gjb = min(gj, nx - 2);
  const int gjr = lane == 0 ? gj - 1 : min(gj + 1, nx - 1);
  bool bad = !den_ok;
  auto load_p = [&] {
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = src[min(gi0 + r, ny - 1) * nx + gjp];
#pragma unroll
    for (int r = 0; r < R; ++r) ring[r] = src[min(gi0 + r, ny - 1) * nx + gjr];
    top = src[(sy.origin - 1) * nx + gjp];
    bottom = src[min(sy.origin + R * kWavesP, ny - 1) * nx + gjp];
  };
  load_p();
#pragma unroll
  for (int r = 0; r < R; ++r) bb[r] = g.b[min(gi0 + r, ny - 2) * nx + gjb];
  auto in_range = [](double a) { return fabs(a) < 0x1p100; };
#pragma unroll
  for (int r = 0; r < R; ++r)
    bad = bad || !in_range(x[r]) || !in_range(bb[r]) || !in_range(ring[r]);
  bad = bad || !in_range(top) || !in_range(bottom);
  int emin = 0;
  pressure_steps<R, NARROW, false>(x, bb, ring, top, bottom, edge, lane, w, gi0, gj, g, v, depth,
                                   emin);
  bad = bad || emin < kMinExpN;
  if (__syncthreads_or(bad)) {
    load_p();
    pressure_steps<R, NARROW, true>(x, bb, ring, top, bottom, edge, lane, w, gi0, gj, g, v, depth,
                                    emin);
  }

  // the block's interior points, with the edge copies the boundary statements
  // make of them
  if (lane < sx.lo || lane >= sx.hi || gj > nx - 2) return;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int gi = gi0 + r, k = w * R + r;
    if (k < sy.lo || k >= sy.hi || gi > ny - 2) continue;
    const int at = gi * nx + gj;
    store_pressure(dst, at, (gi == 1 ? kRow1 : 0) | (gj == 1 ? kCol1 : 0) |
                                (gj == nx - 2 ? kColLast : 0), nx, x[r]);
    if (gi == ny - 2) {  // p[-1, :] = 0, the corners with it
      dst[at + nx] = 0.0;
      if (gj == 1) dst[at + nx - 1] = 0.0;
      if (gj == nx - 2) dst[at + nx + 1] = 0.0;
    }
  }
}

// The velocity update of one step (VEL; otherwise u, v are taken as they are)
// and the source cb b of the next (SRC), one point per thread: a workgroup
// computes the new u, v of 16 x 64 points, exchanges them through LDS and
// forms b for the 14 x 62 inside.  un, vn -> u, v are separate arrays (the
// reference's copies); boundary points take the boundary conditions
// (:75-82), the same value from every workgroup that holds them.
constexpr int kTileVI = 14, kTileVJ = 62;

template <bool VEL, bool SRC>
__global__ __launch_bounds__(1024) void cavity_velocity(CavityArgs g, const double* __restrict__ p,
                                                        int tiles_x) {
  __shared__ double su[16][64], sv[16][64];
  const int lane = threadIdx.x % 64;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int nx = g.nx, ny = g.ny;
  const int gi = static_cast<int>(blockIdx.x) / tiles_x * kTileVI + w;
  const int gj = static_cast<int>(blockIdx.x) % tiles_x * kTileVJ + lane;
  const bool inside = gi < ny && gj < nx;
  const bool interior = gi >= 1 && gi <= ny - 2 && gj >= 1 && gj <= nx - 2;
  const bool owned = interior && w >= 1 && w <= kTileVI && lane >= 1 && lane <= kTileVJ;
  const CavityDivisors dv = cavity_divisors(g);
  const int at = gi * nx + gj;
  double nu = 0.0, nv = 0.0;
  if (VEL && interior) {
    double un1[1];
    chunk_eval(dv, un1, [&](int, auto& div) {
      double uu;
      velocity_at(g, dv, p, at, uu, nv, div);
      return uu;
    });
    nu = un1[0];
  } else if (VEL) {
    nu = gi == ny - 1 ? 1.0 : 0.0;
  } else if (inside) {
    nu = g.un[at];
    nv = g.vn[at];
  }
  if (inside && (owned || !interior) && g.u != g.un) {
    g.u[at] = nu;
    g.v[at] = nv;
  }
  if constexpr (SRC) {
    su[w][lane] = nu;
    sv[w][lane] = nv;
    __syncthreads();
    if (!owned) return;
    double bv[1];
    chunk_eval(dv, bv, [&](int, auto& div) {
      return source_from(g, dv, su[w][lane + 1], su[w][lane - 1], su[w + 1][lane],
                         su[w - 1][lane], sv[w][lane + 1], sv[w][lane - 1], sv[w + 1][lane],
                         sv[w - 1][lane], div);
    });
    g.b[at] = g.cb * bv[0];
  }
}

// Grids of up to kLdsPoints points, PTS (2 or kMaxPts) interior points a thread:
// both pressure buffers live in LDS for the whole run, each thread keeps its (at
// most PTS) interior points' indices, edge flags and b values in registers -- it
// computes b for the same points it then iterates -- so a pressure iteration
// touches LDS only.
template <int PTS>
__global__ __launch_bounds__(kThreadsC) void cavity_flow_lds(CavityArgs g) {
  __shared__ double lp[2 * kLdsPoints];
  const int t = threadIdx.x, nx = g.nx, ny = g.ny;
  const int np = nx * ny;
  const CavityDivisors dv = cavity_divisors(g);
  const InteriorWalk walk(t, nx, ny);
  int pa[PTS];  // past cnt: the safe interior index nx + 1, read and never written
#pragma unroll
  for (int m = 0; m < PTS; ++m) pa[m] = nx + 1;
  int pfl = 0;  // 3 edge-flag bits per point
  int cnt = 0;
  walk.each<PTS>([&](const int(&a)[PTS], const int(&fl)[PTS],
                         const bool(&ok)[PTS]) {
#pragma unroll
    for (int m = 0; m < PTS; ++m) {
      pa[m] = a[m];
      pfl |= (ok[m] ? fl[m] : 0) << (3 * m);
      cnt += ok[m] ? 1 : 0;
    }
  });
  for (int k = t; k < np; k += kThreadsC) lp[k] = g.p[k];
  double* cur = lp;  // the current pressure
  double* nxt = lp + kLdsPoints;
  __syncthreads();
  for (int step = 0; step < g.nt; ++step) {
    // the indices are opaque to the compiler here, so it recomputes the
    // neighbours' addresses each step instead of holding every one of them
    // in registers across the loop
#pragma unroll
    for (int m = 0; m < PTS; ++m) asm volatile("" : "+v"(pa[m]));
    asm volatile("" : "+v"(pfl), "+v"(cnt));
    copy_velocities(g, t, np);
    double bq[PTS];
#pragma unroll
    for (int m0 = 0; m0 < PTS; m0 += kChunkV) {
      double bc[kChunkV] = {};
      if (m0 < cnt)  // whole waves skip the chunks past their points
        chunk_eval(dv, bc, [&](int c, auto& div) { return source_at(g, dv, pa[m0 + c], div); });
#pragma unroll
      for (int c = 0; c < kChunkV; ++c) bq[m0 + c] = bc[c];
      asm volatile("" ::: "memory");  // keeps the next chunk's loads behind this one's
    }
    __syncthreads();  // un and vn complete
    for (int q = 0; q < g.nit; ++q) {
      // opaque here too, with the flags and the count: the lane masks the
      // compiler would otherwise hoist out of this loop overflow the scalar
      // registers
#pragma unroll
      for (int m = 0; m < PTS; ++m) asm volatile("" : "+v"(pa[m]));
      asm volatile("" : "+v"(pfl), "+v"(cnt));
#pragma unroll
      for (int m0 = 0; m0 < PTS; m0 += PTS / 2) {
        if (m0 >= cnt) continue;
        double val[PTS / 2];
        chunk_eval(dv, val, [&](int c, auto& div) {
          return pressure_at(g, dv, cur, pa[m0 + c], bq[m0 + c], div);
        });
#pragma unroll
        for (int c = 0; c < PTS / 2; ++c)
          if (m0 + c < cnt) store_pressure(nxt, pa[m0 + c], (pfl >> (3 * (m0 + c))) & 7, nx, val[c]);
      }
      for (int k = t; k < nx; k += kThreadsC) nxt[(ny - 1) * nx + k] = 0.0;  // p[-1, :] = 0
      __syncthreads();
      double* tmp = cur;
      cur = nxt;
      nxt = tmp;
    }
#pragma unroll
    for (int m0 = 0; m0 < PTS; m0 += kChunkV) {
      if (m0 >= cnt) continue;
      double nu[kChunkV], nv[kChunkV];
      chunk_eval(dv, nu, [&](int c, auto& div) {
        double uu;
        velocity_at(g, dv, cur, pa[m0 + c], uu, nv[c], div);
        return uu;
      });
#pragma unroll
      for (int c = 0; c < kChunkV; ++c) {
        if (m0 + c < cnt) {
          g.u[pa[m0 + c]] = nu[c];
          g.v[pa[m0 + c]] = nv[c];
        }
      }
    }
    velocity_boundaries(g, t);
    __syncthreads();
  }
  for (int k = t; k < np; k += kThreadsC) g.p[k] = cur[k];
}

// Shape of the pressure launches: rows per wave and iterations per launch
// with the smallest modelled time for a step.  A launch costs about 4 us
// (gap, loads, stores) and an iteration 0.1 us (exchange, barrier) plus
// 0.1 us per row of a wave and per workgroup a CU has to run.
struct PressurePlan {
  int rows, depth, rounds;
};

PressurePlan plan_pressure(int nx, int ny, int nit) {
  PressurePlan best{};
  double best_us = INFINITY;
  for (const int rows : {2, 3, 4, 6}) {
    for (int rounds = static_cast<int>(cdiv(nit, kMaxDepth)); rounds <= nit; ++rounds) {
      const int depth = static_cast<int>(cdiv(nit, rounds));
      if (64 - 2 * depth < 8 || rows * kWavesP - 2 * depth < 8) continue;
      const int tx = span_count(nx - 2, 64, depth), ty = span_count(ny - 2, rows * kWavesP, depth);
      const double us = rounds * 4.0 + nit * (0.1 + 0.1 * rows * cdiv(int64_t(tx) * ty, 256));
      if (us < best_us) {
        best_us = us;
        best = {rows, depth, rounds};
      }
      if (depth <= 4) break;  // shallower launches only add launches
    }
  }
  return best;
}

template <int R>
void launch_rows(const CavityArgs& g, const double* src, double* dst, int depth,
                 hipStream_t stream) {
  // a shallower last round has fewer blocks
  const int tx = span_count(g.nx - 2, 64, depth), ty = span_count(g.ny - 2, R * kWavesP, depth);
  const dim3 grid(static_cast<unsigned>(tx) * ty), block(64 * kWavesP);
  if (g.nx - 2 < 64 || g.ny - 2 < R * kWavesP)
    hipLaunchKernelGGL((cavity_pressure<R, true>), grid, block, 0, stream, g, src, dst, depth,
                       tx, ty);
  else
    hipLaunchKernelGGL((cavity_pressure<R, false>), grid, block, 0, stream, g, src, dst, depth,
                       tx, ty);
}

int launch_pressure(const CavityArgs& g, int rows, const double* src, double* dst, int depth,
                    hipStream_t stream) {
  switch (rows) {
    case 2: launch_rows<2>(g, src, dst, depth, stream); break;
    case 3: launch_rows<3>(g, src, dst, depth, stream); break;
    case 4: launch_rows<4>(g, src, dst, depth, stream); break;
    default: launch_rows<6>(g, src, dst, depth, stream); break;
  }
  NPBX_LAUNCHED("cavity_pressure");
  return NPBX_OK;
}

// The whole call in chip-wide launches: the source of the first step, then
// per step its pressure rounds and one launch for its velocities and the next
// step's source.  u, v and p alternate with scratch copies; where an odd
// number of updates would leave them there, the first launch starts from a
// copy so that the last one lands in the caller's arrays.
int blocked_flow(const CavityArgs& a, hipStream_t stream) {
  const PressurePlan pl = a.nit > 0 ? plan_pressure(a.nx, a.ny, a.nit) : PressurePlan{};
  const int tiles_x = static_cast<int>(cdiv(a.nx - 2, kTileVJ));
  const int64_t tiles = int64_t(tiles_x) * cdiv(a.ny - 2, kTileVI);
  NPBX_REQUIRE(tiles < (int64_t(1) << 31), "cavity_flow: grid too large");
  const size_t bytes = static_cast<size_t>(a.nx) * a.ny * sizeof(double);
  const dim3 grid(static_cast<unsigned>(tiles)), block(1024);
  double *ucur = a.u, *vcur = a.v, *ualt = a.un, *valt = a.vn;
  double *pcur = a.p, *palt = a.pn;
  if (static_cast<int64_t>(a.nt) * pl.rounds % 2) {
    NPBX_HIP(hipMemcpyAsync(palt, pcur, bytes, hipMemcpyDeviceToDevice, stream));
    std::swap(pcur, palt);
  }
  CavityArgs g = a;
  g.un = ucur, g.vn = vcur;
  if (a.nt % 2) std::swap(ucur, ualt), std::swap(vcur, valt);
  g.u = ucur, g.v = vcur;
  hipLaunchKernelGGL((cavity_velocity<false, true>), grid, block, 0, stream, g, pcur, tiles_x);
  NPBX_LAUNCHED("cavity_velocity");
  for (int step = 0; step < a.nt; ++step) {
    for (int done = 0; done < a.nit; done += pl.depth) {
      NPBX_TRY(launch_pressure(a, pl.rows, pcur, palt, std::min(pl.depth, a.nit - done), stream));
      std::swap(pcur, palt);
    }
    g.un = ucur, g.vn = vcur, g.u = ualt, g.v = valt;
    if (step + 1 < a.nt)
      hipLaunchKernelGGL((cavity_velocity<true, true>), grid, block, 0, stream, g, pcur, tiles_x);
    else
      hipLaunchKernelGGL((cavity_velocity<true, false>), grid, block, 0, stream, g, pcur,
                         tiles_x);
    NPBX_LAUNCHED("cavity_velocity");
    std::swap(ucur, ualt);
    std::swap(vcur, valt);
  }
  return NPBX_OK;
}

// The one-workgroup form where an iteration costs less than its share of the
// blocked form's launches: up to some 1500 interior points, and more where there
// are few iterations.  us a step, one workgroup | blocks:
//   iterations        1            5             10          20          50
//   20 x 20       3.2 |  9.7    4.8 | 10.8   6.7 | 12.7  10.7 | 20.9  22.4 | 46.9
//   33 x 33       6.3 | 10.6    8.6 | 11.2  11.5 | 13.4  17.2 | 21.6  34.4 | 48.5
//   40 x 40       6.7 | 10.0    9.5 | 11.5  13.2 | 13.1  20.3 | 21.9  41.9 | 48.7
//   45 x 45       7.2 | 10.3   10.9 | 11.5  15.7 | 13.3  25.1 | 22.0  53.3 | 49.3
//   50 x 50       8.2 | 10.3   12.3 | 12.3  17.3 | 13.8  27.3 | 22.0
//   400 wide, 3   4.3 |  8.7    5.9 | 10.0   7.9 | 12.2  11.8 | 20.5  23.6 | 47.6
//   2000 wide, 3 10.2 |  9.1   14.0 | 10.3  18.7 | 12.4  28.2 | 20.8  56.5 | 47.7
// Without iterations (velocities only) 400 x 3 takes 3.8 | 4.7, 32 x 32 5.5 | 5.3
// and 1000 x 3 7.0 | 4.6.
bool use_lds(int64_t nx, int64_t ny, int64_t nit) {
  const int64_t points = nx * ny, interior = (nx - 2) * (ny - 2);
  if (points <= 1024) return true;
  static_assert(2600 <= kMaxPts * kThreadsC);
  if (points > kLdsPoints || interior > 2600) return false;
  if (nit == 0) return interior <= 600;
  return interior <= 1500 || (nit <= (interior <= 2048 ? 4 : 2) && points <= 4000);
}

}  // namespace
}  // namespace npbx

extern "C" int npbx_cavity_flow(int dtype, int64_t nx, int64_t ny, int64_t nt, int64_t nit,
                                void* u, void* v, double dt, double dx, double dy, void* p,
                                double rho, double nu, void* stream) {
  using namespace npbx;
  NPBX_REQUIRE(dtype == NPBX_F64, "cavity_flow: dtype %s not supported (f64)",
               dtype_name(dtype));
  NPBX_REQUIRE(nx >= 3 && ny >= 3 && nx * ny <= (int64_t(1) << 26),
               "cavity_flow: grid %lld x %lld out of range (3 x 3 .. 2^26 points)",
               static_cast<long long>(ny), static_cast<long long>(nx));
  NPBX_REQUIRE(nt >= 0 && nit >= 0 && nt <= (int64_t(1) << 30) && nit <= (int64_t(1) << 30),
               "cavity_flow: negative or huge step counts");
  if (nt == 0) return NPBX_OK;
  NPBX_REQUIRE(u && v && p && u != v && v != p && u != p, "cavity_flow: u, v, p must be distinct non-null arrays");
  const int64_t np = nx * ny;
  void* ws = nullptr;
  NPBX_TRY(workspace(static_cast<size_t>(4 * np) * sizeof(double), &ws));
  CavityArgs g;
  g.u = static_cast<double*>(u);
  g.v = static_cast<double*>(v);
  g.p = static_cast<double*>(p);
  g.un = static_cast<double*>(ws);
  g.vn = g.un + np;
  g.pn = g.vn + np;
  g.b = g.pn + np;
  g.nx = static_cast<int>(nx);
  g.ny = static_cast<int>(ny);
  g.nt = static_cast<int>(nt);
  g.nit = static_cast<int>(nit);
  g.rho = rho;
  g.nu = nu;
  g.dt = dt;
  g.dx = dx;
  g.dy = dy;
  g.inv_dt = 1.0 / dt;
  g.two_dx = 2.0 * dx;
  g.two_dy = 2.0 * dy;
  // CPython's x**2 calls the C library's pow; an opaque exponent keeps the
  // compiler from folding the call into x * x
  volatile double two = 2.0;
  g.dx2 = std::pow(dx, static_cast<double>(two));
  g.dy2 = std::pow(dy, static_cast<double>(two));
  g.den = 2.0 * (g.dx2 + g.dy2);
  g.cb = g.dx2 * g.dy2 / g.den;
  g.cpu = dt / (2.0 * rho * dx);
  g.cpv = dt / (2.0 * rho * dy);
  g.cdx2 = dt / g.dx2;
  g.cdy2 = dt / g.dy2;
  if (!use_lds(nx, ny, nit)) return blocked_flow(g, as_stream(stream));
  // A time step depends on u, v and p only (b, un, vn are rebuilt each step),
  // so the steps split into launches of about 50 ms of work each: no launch
  // runs for long, whatever nt is.
  const int64_t per_launch = std::max<int64_t>(1, int64_t(150000000) / (np * (nit + 3)));
  for (int64_t done = 0; done < nt; done += per_launch) {
    g.nt = static_cast<int>(std::min<int64_t>(per_launch, nt - done));
    const auto kernel =
        (nx - 2) * (ny - 2) <= 2 * kThreadsC ? cavity_flow_lds<2> : cavity_flow_lds<kMaxPts>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kThreadsC), 0, as_stream(stream), g);
    NPBX_LAUNCHED("cavity_flow_lds");
  }
  return NPBX_OK;
}
