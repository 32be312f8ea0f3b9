// Single-rectangle levels that fit one work-group's LDS (gfx950).
//
// A level of a few thousand cells is a microsecond of work, but a red-black
// sweep of it as a grid launch takes 4 to 10 us: the launch, a round trip to
// the other XCDs' data and the tile's serial steps.  What bounds the sweeps
// of such a level is that latency, so these kernels keep the level where the
// next sweep reads it: one work-group holds the iterate in LDS and every
// cell's right-hand side, coefficients and reciprocal diagonal in registers,
// and any number of sweeps (k_box_lds_rbgs in box_small.hip) or the whole lower part of a
// multigrid V-cycle (k_mg_bottom in mg_bottom.hip) is one launch whose steps are separated by
// work-group barriers.
//
// LDS holds the two colours apart: colour c of row (j, k) has its cells
// i = p, p + 2, ... at consecutive slots (p the parity of its first cell), so
// lanes that update neighbouring cells of one colour read and write
// consecutive words.  With slot t of a cell, its neighbours are, in the other
// colour's array, t - 1 + p and t + p along x, t -+ (slots of a row) along y
// and t -+ (slots of a plane) along z.
//
// The values are those of the grid-parallel kernels (box_kernels.hip) bit for
// bit: updates of one colour are independent, the update is the same
// expression, and the physical Robin ghost is formed from the cell's own
// value, the one a ghost fill of the current state writes there.
//
// Measured, us per sweep with the early-exit test, FP64, in place of one launch
// of k_box_rbgs: 64 x 64 constant D 1.52 (4.69), 31 x 23 1.00 (4.70), 16^3
// variable D 3.05 (9.35), 9^3 1.28 (8.65).
#pragma once

#include <cmath>

#include "box_device.h"

namespace sfac {
namespace {

// Threads of the work-group: with coefficients (up to 18 registers a cell in
// FP64) 512, which leave each thread up to 256 registers, four cells of each
// colour; without 1024, whose wavefronts hide more of the LDS and arithmetic
// latency (64 x 64, FP64: 1.5 us a sweep, 2.1 with
// 512 threads and four cells each).
constexpr int kSmallThreads(bool coefs) { return coefs ? 512 : 1024; }

// The homogeneous Robin ghost of every boundary side as c1 u / c2 (robin_ghost).
// exact: every side's coefficients are powers of two (Dirichlet and Neumann
// data on grids of such spacing), so that u times their ratio, then in rc, has
// the same bits; else rc is the reciprocal of c2, and with `quick` every
// side's quotient may be formed with it.  One choice for all sides: made side
// by side inside the ghosts it cost more than the quotient saves (64 sweeps of
// 5^3 83 us, 55 us so, 67 us with plain divisions).
template <typename T>
struct SmallRobin {
  T c1[6], c2[6], rc[6];
  int exact, quick;
};

template <typename T>
SmallRobin<T> small_robin(const BoxLevel& G, const RobinDev& bc) {
  SmallRobin<T> R{};
  const T half = (T)0.5;
  R.exact = R.quick = 1;
  for (int loc = 0; loc < 2 * G.dim; ++loc) {
    const T h = (T)G.dx[loc >> 1], av = (T)bc.a[loc], bv = (T)bc.b[loc];
    R.c1[loc] = bv - half * h * av;
    R.c2[loc] = bv + half * h * av;
    const double m = std::fabs((double)R.c2[loc]);
    int ex;
    if (!(m > 1e-8 && m < 1e8)) R.quick = 0;
    if (std::fabs(std::frexp((double)R.c1[loc], &ex)) != 0.5 || std::frexp(m, &ex) != 0.5)
      R.exact = 0;
  }
  if (!R.quick) R.exact = 0;
  for (int loc = 0; loc < 2 * G.dim; ++loc)
    R.rc[loc] = R.exact ? R.c1[loc] / R.c2[loc] : (R.quick ? (T)1 / R.c2[loc] : (T)0);
  return R;
}

// Values whose ghosts the quick quotient forms: no step overflows or loses
// bits for 1e-8 < |c2| < 1e8.
__device__ inline bool quick_range(double u) {
  const double a = fabs(u);
  return (a > 1e-250 && a < 1e250) || a == 0.0;
}
__device__ inline bool quick_range(float u) {
  const float a = fabsf(u);
  return (a > 1e-20f && a < 1e20f) || a == 0.0f;
}
__device__ inline double fused(double a, double b, double c) { return fma(a, b, c); }
__device__ inline float fused(float a, float b, float c) { return fmaf(a, b, c); }

// c1 u / c2 for a u in quick_range: correctly rounded from rc = 1 / c2
// correctly rounded by a quotient estimate and two residual corrections with
// fused multiply-adds, the second of which rounds correctly (Markstein, IBM
// J. Res. Dev. 34, 1990).
template <int DIM, typename T>
__device__ inline T quick_ghost(const SmallRobin<T>& R, int loc, T u) {
  const T p = DIM == 3 ? (T)0 + u * R.c1[loc] : u * R.c1[loc];
  T q = p * R.rc[loc];
  q = fused(fused(-q, R.c2[loc], p), R.rc[loc], q);
  return fused(fused(-q, R.c2[loc], p), R.rc[loc], q);
}
template <int DIM, typename T>
__device__ inline T full_ghost(const SmallRobin<T>& R, int loc, T u) {
  const T p = DIM == 3 ? (T)0 + u * R.c1[loc] : u * R.c1[loc];
  return p / R.c2[loc];
}
template <int DIM, typename T>
__device__ inline T small_ghost(const SmallRobin<T>& R, int loc, T u) {
  if (R.exact) return u * R.rc[loc];
  if (R.quick && quick_range(u)) return quick_ghost<DIM>(R, loc, u);
  return full_ghost<DIM>(R, loc, u);
}

// Slots of a level's colour arrays in LDS: `row` per row, `plane` per plane,
// `count` per colour; `pad` slots on both sides of each array keep the
// neighbour indices of boundary cells (whose values are not used) inside.
//
// Threads take the slots in another order, the first and last of every row
// (where the cells on the x boundary are) after all others: a Robin ghost
// costs as much as the update itself, and so only the wavefronts that hold
// boundary cells form it.  `core` is the number of the other slots and
// `units` the number of all, the core padded to whole wavefronts.
struct Slots {
  int row, plane, count, pad, stride, core, units;
};
__host__ __device__ inline Slots slots_of(const BoxLevel& G) {
  Slots s;
  s.row = (G.n[0] + 1) / 2;
  s.plane = s.row * G.n[1];
  s.count = s.plane * (G.dim == 3 ? G.n[2] : 1);
  s.pad = G.dim == 3 ? s.plane : s.row;
  s.stride = s.count + 2 * s.pad;
  const int rows = s.count / s.row;
  s.core = s.row > 2 ? rows * (s.row - 2) : 0;
  s.units = (s.core + 63) / 64 * 64 + (s.row > 2 ? 2 * rows : s.count);
  return s;
}
__device__ inline int colour_parity(const BoxLevel& G) {
  return G.lo[0] + G.lo[1] + (G.dim == 3 ? G.lo[2] : 0) + G.shift;
}

// One thread's cells of a level: units threadIdx.x + v blockDim.x of both
// colours.  flags: bits 0-5 faces on the physical boundary, 6 the slot is a
// cell, 7 in the last patch, from 8 on the cell's natural index.  k holds the
// right-hand side, 1/dx times the face coefficients (the first product of
// each flux) and C.
template <typename T, int NC>
struct SmallCells {
  int slot[NC];
  int flags[2][NC];
  int left[2][NC];  // the lower x neighbour's slot in the other colour
  T u[2][NC], dudr[2][NC];
  Coef<T> k[2][NC];
};

// A level's constants for the updates.
template <typename T>
struct SmallConst {
  T dxi, dyi, dzi, cc, dudr;
  T kx, ky, kz;  // 1/dx times the constant D
};
template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline SmallConst<T> small_const(const BoxLevel& G, const BoxArraysT<T>& A) {
  SmallConst<T> s;
  s.dxi = (T)(1.0 / G.dx[0]);
  s.dyi = (T)(1.0 / G.dx[1]);
  s.dzi = DIM == 3 ? (T)(1.0 / G.dx[2]) : (T)0;
  const T dc = (T)A.dconst;
  s.kx = s.dxi * dc;
  s.ky = s.dyi * dc;
  s.kz = s.dzi * dc;
  s.cc = (T)A.cconst;
  s.dudr = (!DVAR && CMODE != 2) ? cell_dudr<DIM, DVAR, CMODE>(Coef<T>{}, G, A) : (T)0;
  return s;
}

template <int DIM, bool DVAR, int CMODE, typename T, int NC>
__device__ inline void small_load(const BoxLevel& G, const BoxArraysT<T>& A, const Slots& S,
                                  const SmallConst<T>& s, SmallCells<T, NC>& q) {
  const int n0 = G.n[0], n1 = G.n[1], n2 = DIM == 3 ? G.n[2] : 1;
  const int par = colour_parity(G);
  const int core = (S.core + 63) / 64 * 64;
#pragma unroll
  for (int v = 0; v < NC; ++v) {
    const int w = threadIdx.x + v * blockDim.x;
    int rw, m;
    bool live;
    if (w < core) {
      live = w < S.core;
      rw = w / (S.row - 2);
      m = 1 + w - rw * (S.row - 2);
    } else if (S.row > 2) {
      live = w < S.units;
      rw = (w - core) >> 1;
      m = (w & 1) ? S.row - 1 : 0;
    } else {
      live = w < S.units;
      rw = w / S.row;
      m = w - rw * S.row;
    }
    if (!live) rw = m = 0;
    const int j = rw % n1, k = DIM == 3 ? rw / n1 : 0;
    // a unit that is no cell reads slot 0 and writes nothing
    q.slot[v] = rw * S.row + m;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int p = pos2(par + j + k + c), i = 2 * m + p;
      q.flags[c][v] = 0;
      q.left[c][v] = rw * S.row + m - 1 + p;
      q.u[c][v] = (T)0;
      q.k[c][v] = Coef<T>{};
      q.dudr[c][v] = (T)0;
      if (live && i < n0) {
        const bool lp = i >= G.lp_lo[0] && i <= G.lp_hi[0] && j >= G.lp_lo[1] && j <= G.lp_hi[1] &&
                        (DIM == 2 || (k >= G.lp_lo[2] && k <= G.lp_hi[2]));
        q.flags[c][v] = 64 | (i == 0 ? 1 : 0) | (i == n0 - 1 ? 2 : 0) | (j == 0 ? 4 : 0) |
                        (j == n1 - 1 ? 8 : 0) |
                        (DIM == 3 ? (k == 0 ? 16 : 0) | (k == n2 - 1 ? 32 : 0) : 0) |
                        (lp ? 128 : 0) | (i + n0 * (j + n1 * k)) << 8;
        q.k[c][v] = load_coef<DIM, DVAR, 0>(G, A, i, j, k);
        // a constant C may come as C mode 2 without an array (k_mg_bottom)
        if (CMODE == 2) q.k[c][v].c = A.C ? A.C[i + n0 * (j + n1 * k)] : (T)A.cconst;
      }
    }
  }
  if (DVAR || CMODE == 2) {
#pragma unroll
    for (int v = 0; v < NC; ++v)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        if (q.flags[c][v]) {
          Coef<T>& k = q.k[c][v];
          q.dudr[c][v] = cell_dudr<DIM, DVAR, CMODE>(k, G, A);
          k.xl = s.dxi * k.xl;
          k.xh = s.dxi * k.xh;
          k.yl = s.dyi * k.yl;
          k.yh = s.dyi * k.yh;
          k.zl = s.dzi * k.zl;
          k.zh = s.dzi * k.zh;
        }
  }
}

// A cell's neighbours (x, y, z; lower then upper).
template <typename T>
struct SmallNbr {
  T v[6];
};

// Residuals of N of a thread's cells of colour c from unit v0 on, their
// neighbours read from the other colour's array (cell_update's expression
// order).  The LDS reads of the N cells are issued first and only the ghosts
// are formed under branches, so that the cells' latencies overlap.
template <int DIM, bool DVAR, int CMODE, int N, typename T, int NC>
__device__ inline void small_residuals(const T* E, int c, int v0, const Slots& S,
                                       const SmallCells<T, NC>& q, const SmallConst<T>& s,
                                       const SmallRobin<T>& R, T* res) {
  const T* o = E + (c ^ 1) * S.stride + S.pad;
  SmallNbr<T> n[N];
#pragma unroll
  for (int v = 0; v < N; ++v) {
    const T* x = o + q.left[c][v0 + v];
    const T* y = o + q.slot[v0 + v];
    n[v].v[0] = x[0];
    n[v].v[1] = x[1];
    n[v].v[2] = y[-S.row];
    n[v].v[3] = y[S.row];
    n[v].v[4] = DIM == 3 ? y[-S.plane] : (T)0;
    n[v].v[5] = DIM == 3 ? y[S.plane] : (T)0;
  }
  // the ghosts of boundary cells
#pragma unroll
  for (int v = 0; v < N; ++v) {
    int fl = q.flags[c][v0 + v];
    // the conditions are formed anew in every sweep: kept across the sweeps
    // they are pairs of scalar registers, more than there are
    asm volatile("" : "+v"(fl));
    if (fl & 63) {
      const T uc = q.u[c][v0 + v];
      if (R.exact) {
#pragma unroll
        for (int loc = 0; loc < 2 * DIM; ++loc)
          if (fl & (1 << loc)) n[v].v[loc] = uc * R.rc[loc];
      } else if (R.quick && !__any(!quick_range(uc))) {
#pragma unroll
        for (int loc = 0; loc < 2 * DIM; ++loc)
          if (fl & (1 << loc)) n[v].v[loc] = quick_ghost<DIM>(R, loc, uc);
      } else {
#pragma unroll
        for (int loc = 0; loc < 2 * DIM; ++loc)
          if (fl & (1 << loc)) n[v].v[loc] = full_ghost<DIM>(R, loc, uc);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < N; ++v) {
    const T uc = q.u[c][v0 + v];
    const Coef<T>& k = q.k[c][v0 + v];
    const T fxl = (DVAR ? k.xl : s.kx) * (uc - n[v].v[0]);
    const T fxh = (DVAR ? k.xh : s.kx) * (n[v].v[1] - uc);
    const T fyl = (DVAR ? k.yl : s.ky) * (uc - n[v].v[2]);
    const T fyh = (DVAR ? k.yh : s.ky) * (n[v].v[3] - uc);
    T div = s.dxi * (fxh - fxl) + s.dyi * (fyh - fyl);
    if (DIM == 3) {
      const T fzl = (DVAR ? k.zl : s.kz) * (uc - n[v].v[4]);
      const T fzh = (DVAR ? k.zh : s.kz) * (n[v].v[5] - uc);
      div = div + s.dzi * (fzh - fzl);
    }
    // without a C term nothing is subtracted (0 u is 0 for every finite u)
    res[v] = CMODE == 0 ? k.f - div : k.f - div - (CMODE == 2 ? k.c : s.cc) * uc;
  }
}

// One colour of a sweep; with check, returns the largest |residual| in the
// last patch.  Two cells at a time in 3-D with FP64 coefficients (four do not
// fit the registers).
template <int DIM, bool DVAR, int CMODE, typename T, int NC>
__device__ inline T small_colour(T* E, int c, const Slots& S, SmallCells<T, NC>& q,
                                 const SmallConst<T>& s, const SmallRobin<T>& R, bool check) {
  constexpr int N = DIM == 3 && (DVAR || CMODE == 2) && sizeof(T) == 8 && NC > 2 ? 2 : NC;
  T* own = E + c * S.stride + S.pad;
  T mr = (T)0;
#pragma unroll
  for (int v0 = 0; v0 < NC; v0 += N) {
    T res[N];
    small_residuals<DIM, DVAR, CMODE, N>(E, c, v0, S, q, s, R, res);
#pragma unroll
    for (int v = 0; v < N; ++v) {
      const int w = v0 + v;
      const T du = -res[v] * ((DVAR || CMODE == 2) ? q.dudr[c][w] : s.dudr);
      q.u[c][w] = q.u[c][w] + du;
      if (q.flags[c][w]) own[q.slot[w]] = q.u[c][w];
      if (check && (q.flags[c][w] & 128)) mr = (T)fmax(mr, (T)fabs(res[v]));
    }
  }
  return mr;
}

// Start values of a thread's cells into registers and LDS (nullptr: 0).
template <typename T, int NC>
__device__ inline void small_start(T* E, const T* uin, const Slots& S, SmallCells<T, NC>& q) {
#pragma unroll
  for (int v = 0; v < NC; ++v)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if (q.flags[c][v]) {
        q.u[c][v] = uin ? uin[q.flags[c][v] >> 8] : (T)0;
        E[c * S.stride + S.pad + q.slot[v]] = q.u[c][v];
      }
}

inline int small_threads(const BoxLevel& G, bool coefs) {
  const int c = slots_of(G).units, most = kSmallThreads(coefs);
  return c >= most ? most : (c + 63) / 64 * 64;
}

}  // namespace
}  // namespace sfac
