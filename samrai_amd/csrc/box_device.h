// Device code shared by the kernels of the single-rectangle levels
// (box_kernels.hip, box_small.hip): per-cell coefficients, the Gauss-Seidel
// update and the Robin ghost, typed by storage precision.
#pragma once

#include "box_kernels.h"

namespace sfac {
namespace {

inline void check_launch() {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw e;
}

__device__ inline int pos2(int x) { return x & 1; }  // parity of any int (two's complement)

// Robin face ghost from its interior neighbour (settype1cells, homogeneous
// or not), location loc = 2*axis + side.
template <int DIM, typename T>
__device__ inline T robin_ghost(const BoxLevel& G, const RobinDev& bc, int homogeneous, int loc,
                                T uin) {
  const int n = loc >> 1;
  const T h = (T)G.dx[n], av = (T)bc.a[loc], bv = (T)bc.b[loc], g = (T)bc.g[loc];
  const T half = (T)0.5;
  if (DIM == 3)
    return ((homogeneous ? (T)0 : h * g) + uin * (bv - half * h * av)) / (bv + half * h * av);
  if (homogeneous) return (uin * (bv - half * h * av)) / (bv + half * h * av);
  return (h * g + uin * (bv - half * h * av)) / (bv + half * h * av);
}

// Box arrays typed by their storage precision.
template <typename T>
inline BoxArraysT<T> typed(const BoxArrays& A) {
  BoxArraysT<T> t;
  t.ein = reinterpret_cast<const T*>(A.ein);
  t.eout = reinterpret_cast<T*>(A.eout);
  t.r = reinterpret_cast<const T*>(A.r);
  for (int a = 0; a < 3; ++a) t.D[a] = reinterpret_cast<const T*>(A.D[a]);
  t.C = reinterpret_cast<const T*>(A.C);
  t.dconst = A.dconst;
  t.cmode = A.cmode;
  t.cconst = A.cconst;
  return t;
}

// Per-cell inputs of one Gauss-Seidel update that do not change during a
// sweep: right-hand side, the six face coefficients (variable D) and C.
template <typename T>
struct Coef {
  T f, xl, xh, yl, yh, zl, zh, c;
};

template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline Coef<T> load_coef(const BoxLevel& G, const BoxArraysT<T>& A, int i, int j,
                                    int k) {
  Coef<T> q{};
  const int n0 = G.n[0], n1 = G.n[1];
  const long c = (long)i + (long)n0 * (j + (long)n1 * k);
  q.f = A.r[c];
  if (DVAR) {
    const long ox = (long)i + (long)(n0 + 1) * (j + (long)n1 * k);
    const long oy = (long)i + (long)n0 * (j + (long)(n1 + 1) * k);
    q.xl = A.D[0][ox];
    q.xh = A.D[0][ox + 1];
    q.yl = A.D[1][oy];
    q.yh = A.D[1][oy + n0];
    if (DIM == 3) {
      q.zl = A.D[2][c];
      q.zh = A.D[2][c + (long)n0 * n1];
    }
  }
  if (CMODE == 2) q.c = A.C[c];
  return q;
}

// 1 / diagonal of a cell's stencil, in the expression order of
// rbgswithfluxmax*.  It depends only on the cell's coefficients, which do
// not change during a solve: callers compute it once per cell (once per
// launch when D and C are constant) and pass it to cell_update, with the
// same bits as forming it inside every update.
template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline T cell_dudr(const Coef<T>& k, const BoxLevel& G, const BoxArraysT<T>& A) {
  const T dxi = (T)(1.0 / G.dx[0]), dyi = (T)(1.0 / G.dx[1]);
  const T dzi = DIM == 3 ? (T)(1.0 / G.dx[2]) : (T)0;
  const T dxi2 = dxi * dxi, dyi2 = dyi * dyi, dzi2 = dzi * dzi;
  const T dc = (T)A.dconst;
  T scal;
  if (CMODE == 2) scal = k.c;
  else scal = CMODE == 1 ? (T)A.cconst : (T)0;
  T diag;
  if (DIM == 3) {
    if (DVAR)
      diag = (dxi2 * (k.xh + k.xl) + dyi2 * (k.yh + k.yl) + dzi2 * (k.zh + k.zl)) - scal;
    else
      diag = (dxi2 * (dc + dc) + dyi2 * (dc + dc) + dzi2 * (dc + dc)) - scal;
  } else {
    if (DVAR)
      diag = (dxi * dxi * (k.xh + k.xl) + dyi * dyi * (k.yh + k.yl)) - scal;
    else
      diag = (dxi * dxi * (dc + dc) + dyi * dyi * (dc + dc)) - scal;
  }
  return (T)1 / diag;
}

// Gauss-Seidel update of one cell held in LDS at q (neighbours at q -+ 1,
// q -+ SY, q - SZd and q + SZu), in the expression order of
// rbgswithfluxmax*, with dudr = cell_dudr of the cell.  Returns |residual|.
// bmask (optional): bit 2a+side set when the face of axis a on that side
// is on the physical boundary; that neighbour is then the Robin ghost of the
// cell's own value, formed here (the value a ghost fill of the current state
// writes there, since the cell is the ghost's only interior neighbour)
// instead of read from U.
template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline T cell_update(T* U, int q, int SY, int SZd, int SZu, const Coef<T>& k,
                                const BoxLevel& G, const BoxArraysT<T>& A, T dudr,
                                int bmask = 0, const RobinDev* bc = nullptr,
                                int homogeneous = 1) {
  const T dxi = (T)(1.0 / G.dx[0]), dyi = (T)(1.0 / G.dx[1]);
  const T dzi = DIM == 3 ? (T)(1.0 / G.dx[2]) : (T)0;
  const T dc = (T)A.dconst;
  const T uc = U[q];
  T uxl = U[q - 1], uxh = U[q + 1], uyl = U[q - SY], uyh = U[q + SY];
  T uzl = DIM == 3 ? U[q - SZd] : (T)0, uzh = DIM == 3 ? U[q + SZu] : (T)0;
  if (bmask != 0) {
    // a branch, not selects: few cells are on the boundary
    if (bmask & 1) uxl = robin_ghost<DIM>(G, *bc, homogeneous, 0, uc);
    if (bmask & 2) uxh = robin_ghost<DIM>(G, *bc, homogeneous, 1, uc);
    if (bmask & 4) uyl = robin_ghost<DIM>(G, *bc, homogeneous, 2, uc);
    if (bmask & 8) uyh = robin_ghost<DIM>(G, *bc, homogeneous, 3, uc);
    if (DIM == 3 && (bmask & 16)) uzl = robin_ghost<DIM>(G, *bc, homogeneous, 4, uc);
    if (DIM == 3 && (bmask & 32)) uzh = robin_ghost<DIM>(G, *bc, homogeneous, 5, uc);
  }
  T Dxl, Dxh, Dyl, Dyh, Dzl = 0, Dzh = 0;
  if (DVAR) {
    Dxl = k.xl;
    Dxh = k.xh;
    Dyl = k.yl;
    Dyh = k.yh;
    if (DIM == 3) {
      Dzl = k.zl;
      Dzh = k.zh;
    }
  } else {
    Dxl = Dxh = Dyl = Dyh = Dzl = Dzh = dc;
  }
  const T fxl = dxi * Dxl * (uc - uxl);
  const T fxh = dxi * Dxh * (uxh - uc);
  const T fyl = dyi * Dyl * (uc - uyl);
  const T fyh = dyi * Dyh * (uyh - uc);
  T fzl = 0, fzh = 0;
  if (DIM == 3) {
    fzl = dzi * Dzl * (uc - uzl);
    fzh = dzi * Dzh * (uzh - uc);
  }
  T scal;
  if (CMODE == 2) scal = k.c;
  else scal = CMODE == 1 ? (T)A.cconst : (T)0;
  const T fv = k.f;
  T residual;
  if (DIM == 3)
    residual = fv - (dxi * (fxh - fxl) + dyi * (fyh - fyl) + dzi * (fzh - fzl)) - scal * uc;
  else
    residual = fv - (dxi * (fxh - fxl) + dyi * (fyh - fyl)) - scal * uc;
  const T du = -residual * dudr;
  U[q] = uc + du * (T)1;
  return fabs(residual);
}

// Raise the word at p (the bits of a non-negative double) to m.  Hundreds of
// work-groups raise one word and most of them to less than it holds: those
// only read it.
__device__ inline void raise_max(unsigned long long* p, double m) {
  const unsigned long long bits = (unsigned long long)__double_as_longlong(m);
  if (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < bits) atomicMax(p, bits);
}

// DIM, DVAR and CMODE of a level's arrays as template arguments of F::run.
template <template <int, bool, int> class F, typename T, class... Args>
void dispatch3(const BoxLevel& G, const BoxArraysT<T>& A, Args&&... args) {
  const bool dvar = A.D[0] != nullptr;
  if (G.dim == 3) {
    if (dvar) {
      if (A.cmode == 2) F<3, true, 2>::run(G, A, args...);
      else if (A.cmode == 1) F<3, true, 1>::run(G, A, args...);
      else F<3, true, 0>::run(G, A, args...);
    } else {
      if (A.cmode == 2) F<3, false, 2>::run(G, A, args...);
      else if (A.cmode == 1) F<3, false, 1>::run(G, A, args...);
      else F<3, false, 0>::run(G, A, args...);
    }
  } else {
    if (dvar) {
      if (A.cmode == 2) F<2, true, 2>::run(G, A, args...);
      else if (A.cmode == 1) F<2, true, 1>::run(G, A, args...);
      else F<2, true, 0>::run(G, A, args...);
    } else {
      if (A.cmode == 2) F<2, false, 2>::run(G, A, args...);
      else if (A.cmode == 1) F<2, false, 1>::run(G, A, args...);
      else F<2, false, 0>::run(G, A, args...);
    }
  }
}

template <typename T>
const T* as(const double* p) { return reinterpret_cast<const T*>(p); }
template <typename T>
T* as(double* p) { return reinterpret_cast<T*>(p); }

}  // namespace
}  // namespace sfac
