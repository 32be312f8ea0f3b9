// The lower part of a multigrid V-cycle (box_small.h).
//
// From the first level of at most kMGDenseCells cells on, a V-cycle is a chain
// of more than a hundred tiny steps (the smallest grid alone takes 60 sweeps),
// each a microsecond of latency on one work-group and most of the machine idle.
// It is also a linear map of the level's right-hand side, e = B f, and it is
// applied up to coarse_solver_max_iterations times per coarse solve with the
// same coefficients.  So a coarse solve that may take several V-cycles forms B
// once, one work-group per column (k_mg_bottom on the unit vectors, all
// columns at once), and a V-cycle's lower part is one matrix-vector product.
// In one work-group, as a coarse solve of few V-cycles takes it, the lower part
// from 8^3 on is 45 us a V-cycle (as launches per step 76), from 10^3 on 81 us
// (105); the product takes 4.  The FAC solve of the 54 M cell hierarchy goes from
// 309 to 296 ms with it, of a 2-D one whose smallest grid is 31 x 23 from 37.8 to
// 29.3 ms.
#include <cstddef>
#include <type_traits>

#include "box_small.h"

namespace sfac {
namespace {

// ------------------------------------------------------------------------
// The lower part of a multigrid V-cycle: levels 0 (of at most kMGDenseCells
// cells) to n - 1 (the smallest) of P, their errors and right-hand sides in LDS.
constexpr int kBottomLevels = 8;
constexpr int kBottomLds = 3584;  // values: 28 KB of FP64, five work-groups a CU
constexpr int kBottomThreads = 512;
constexpr int kBottomSlots = 2;   // per thread and colour on the first level
template <typename T>
struct Bottom {
  int n, pre, post, last;  // levels; sweeps before, after and on the smallest
  int res;                 // LDS offsets: residual, per level error and right-hand side
  int e[kBottomLevels], f[kBottomLevels];
  BoxLevel G[kBottomLevels];
  BoxArraysT<T> A[kBottomLevels];
  SmallRobin<T> R[kBottomLevels];
};

// One level's descriptors, read from the kernel's argument segment (the first
// argument is at its start): uniform loads into scalar registers, where an
// index into the by-value argument would copy it to scratch memory.
typedef const __attribute__((address_space(4))) int* kernarg_ptr;
template <class S>
__device__ inline S kernarg(size_t byte) {
  constexpr int N = sizeof(S) / 4;
  static_assert(sizeof(S) % 4 == 0, "whole words");
  const kernarg_ptr w = (kernarg_ptr)__builtin_amdgcn_kernarg_segment_ptr() + byte / 4;
  struct Words {
    int v[N];
  } t;
#pragma unroll
  for (int i = 0; i < N; ++i) t.v[i] = w[i];
  return __builtin_bit_cast(S, t);
}
template <typename T>
struct BottomLevel {
  BoxLevel G;
  BoxArraysT<T> A;
  SmallRobin<T> R;
  int e, f;
  __device__ explicit BottomLevel(int l)
      : G(kernarg<BoxLevel>(offsetof(Bottom<T>, G) + l * sizeof(BoxLevel))),
        A(kernarg<BoxArraysT<T>>(offsetof(Bottom<T>, A) + l * sizeof(BoxArraysT<T>))),
        R(kernarg<SmallRobin<T>>(offsetof(Bottom<T>, R) + l * sizeof(SmallRobin<T>))),
        e(kernarg<int>(offsetof(Bottom<T>, e) + l * sizeof(int))),
        f(kernarg<int>(offsetof(Bottom<T>, f) + l * sizeof(int))) {}
};

// Error of level G in LDS at index (i, j, k), with homogeneous Robin ghosts
// one cell beyond the domain applied axis by axis (mg_at).
template <int DIM, typename T>
__device__ inline T small_at(const T* E, const BoxLevel& G, const Slots& S, int par,
                             const SmallRobin<T>& R, int i, int j, int k) {
  const int ci = min(max(i, 0), G.n[0] - 1), cj = min(max(j, 0), G.n[1] - 1);
  const int ck = DIM == 3 ? min(max(k, 0), G.n[2] - 1) : 0;
  const int c = pos2(par + ci + cj + ck);
  T v = E[c * S.stride + S.pad + (ci >> 1) + S.row * cj + (DIM == 3 ? S.plane * ck : 0)];
  if (i != ci) v = small_ghost<DIM>(R, i < 0 ? 0 : 1, v);
  if (j != cj) v = small_ghost<DIM>(R, j < 0 ? 2 : 3, v);
  if (DIM == 3 && k != ck) v = small_ghost<DIM>(R, k < 0 ? 4 : 5, v);
  return v;
}

// k_mg_prolong_add (box_kernels.hip) of one cell, from LDS.
template <int DIM, typename T>
__device__ inline T small_prolong(const T* E, const BoxLevel& G, const Slots& S,
                                  const SmallRobin<T>& R, int i, int j, int k) {
  const int par = colour_parity(G);
  const int I = i >> 1, J = j >> 1, K = k >> 1;
  const int sx = (i & 1) ? 1 : -1, sy = (j & 1) ? 1 : -1, sz = (k & 1) ? 1 : -1;
  const T w3 = (T)0.75, w1 = (T)0.25;
  auto at = [&](int a, int b, int c) { return small_at<DIM>(E, G, S, par, R, a, b, c); };
  auto face = [&](int c) {
    return w3 * (w3 * at(I, J, c) + w1 * at(I + sx, J, c)) +
           w1 * (w3 * at(I, J + sy, c) + w1 * at(I + sx, J + sy, c));
  };
  if (DIM == 3) {
    const T z0 = face(K), z1 = face(K + sz);
    return w3 * z0 + w1 * z1;
  }
  return face(0);
}

// Sweeps of a level in LDS; a level whose units fit one wavefront is swept by
// it alone without barriers (its LDS accesses are in order).
template <int DIM, bool DVAR, int CMODE, typename T, int NC>
__device__ inline void small_sweeps(T* E, const Slots& S, SmallCells<T, NC>& q,
                                    const SmallConst<T>& s, const SmallRobin<T>& R, int sweeps) {
  if (S.units <= 64) {
    if (threadIdx.x < 64)
      for (int n = 0; n < sweeps; ++n) {
        (void)small_colour<DIM, DVAR, CMODE>(E, 0, S, q, s, R, false);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        (void)small_colour<DIM, DVAR, CMODE>(E, 1, S, q, s, R, false);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    __syncthreads();
    return;
  }
  for (int n = 0; n < sweeps; ++n) {
    (void)small_colour<DIM, DVAR, CMODE>(E, 0, S, q, s, R, false);
    __syncthreads();
    (void)small_colour<DIM, DVAR, CMODE>(E, 1, S, q, s, R, false);
    __syncthreads();
  }
}

// Level l on the way down: its error from 0 (or from `start`), the sweeps and,
// unless it is the smallest, its residual restricted to the next level's
// right-hand side.  unit >= 0: the level's right-hand side is that unit vector.
template <int DIM, bool DVAR, int CMODE, int NC, typename T>
__device__ inline void bottom_down(T* L, const BottomLevel<T>& V, int l, int n, int res_at,
                                   int sweeps, const T* start, int unit) {
  const BoxLevel& G = V.G;
  const Slots S = slots_of(G);
  BoxArraysT<T> A = V.A;
  if (l > 0) A.r = L + V.f;
  T* E = L + V.e;
  const SmallConst<T> s = small_const<DIM, DVAR, CMODE>(G, A);
  SmallCells<T, NC> q;
  small_load<DIM, DVAR, CMODE>(G, A, S, s, q);
  if (unit >= 0) {
#pragma unroll
    for (int v = 0; v < NC; ++v)
#pragma unroll
      for (int c = 0; c < 2; ++c) q.k[c][v].f = q.flags[c][v] >> 8 == unit ? (T)1 : (T)0;
  }
  small_start(E, start, S, q);
  __syncthreads();
  small_sweeps<DIM, DVAR, CMODE>(E, S, q, s, V.R, sweeps);
  if (l + 1 == n) return;
  T* res = L + res_at;
#pragma unroll
  for (int v = 0; v < NC; ++v)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      T one;
      small_residuals<DIM, DVAR, CMODE, 1>(E, c, v, S, q, s, V.R, &one);
      if (q.flags[c][v]) res[q.flags[c][v] >> 8] = one;
    }
  __syncthreads();
  // the mean over the children of every coarse cell (mg_restrict_value)
  const BottomLevel<T> W(l + 1);
  const BoxLevel& Gc = W.G;
  const int nc = Gc.n[0] * Gc.n[1] * (DIM == 3 ? Gc.n[2] : 1);
  T* fc = L + W.f;
  for (int t = threadIdx.x; t < nc; t += blockDim.x) {
    const int I = t % Gc.n[0], J = (t / Gc.n[0]) % Gc.n[1], K = t / (Gc.n[0] * Gc.n[1]);
    T sum = 0;
    for (int c2 = 0; c2 < (DIM == 3 ? 2 : 1); ++c2)
      for (int c1 = 0; c1 < 2; ++c1)
        for (int c0 = 0; c0 < 2; ++c0)
          sum += res[(2 * I + c0) + G.n[0] * ((2 * J + c1) +
                                              G.n[1] * (DIM == 3 ? 2 * K + c2 : 0))];
    fc[t] = sum * (T)(DIM == 3 ? 0.125 : 0.25);
  }
  __syncthreads();
}

// Level l on the way up: the next level's error interpolated and added, then
// the sweeps; `out` (or nullptr) receives the result.
template <int DIM, bool DVAR, int CMODE, int NC, typename T>
__device__ inline void bottom_up(T* L, const BottomLevel<T>& V, int l, int sweeps, int unit,
                                 T* out, int stride) {
  const BottomLevel<T> W(l + 1);
  const BoxLevel& G = V.G;
  const BoxLevel& Gc = W.G;
  const Slots S = slots_of(G), Sc = slots_of(Gc);
  BoxArraysT<T> A = V.A;
  if (l > 0) A.r = L + V.f;
  T* E = L + V.e;
  const T* Ec = L + W.e;
  const SmallConst<T> s = small_const<DIM, DVAR, CMODE>(G, A);
  SmallCells<T, NC> q;
  small_load<DIM, DVAR, CMODE>(G, A, S, s, q);
#pragma unroll
  for (int v = 0; v < NC; ++v)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if (q.flags[c][v]) {
        if (unit >= 0) q.k[c][v].f = q.flags[c][v] >> 8 == unit ? (T)1 : (T)0;
        const int n = q.flags[c][v] >> 8;
        const int i = n % G.n[0], j = (n / G.n[0]) % G.n[1], k = n / (G.n[0] * G.n[1]);
        T& x = E[c * S.stride + S.pad + q.slot[v]];
        q.u[c][v] = x + small_prolong<DIM>(Ec, Gc, Sc, W.R, i, j, DIM == 3 ? k : 0);
        x = q.u[c][v];
      }
  __syncthreads();
  small_sweeps<DIM, DVAR, CMODE>(E, S, q, s, V.R, sweeps);
  if (out)
#pragma unroll
    for (int v = 0; v < NC; ++v)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        if (q.flags[c][v]) out[(long)stride * (q.flags[c][v] >> 8)] = q.u[c][v];
}

// The levels of P (its first member of the argument segment, see kernarg);
// the error of the first from 0 (from_input 0) or from e, and to e.  With
// `columns` (the first level's cells) work-group b solves for the b-th unit
// vector, from 0, into column b of the row-major matrix e.  A level of no more
// units than threads takes the code for one unit a thread.
template <int DIM, bool DVAR, int CMODE, typename T>
__global__ void __launch_bounds__(kBottomThreads)
k_mg_bottom(Bottom<T> P, T* e, int from_input, int columns, const int* stop) {
  __shared__ T L[kBottomLds];
  if (*stop) return;
  const int stride = columns > 0 ? columns : 1;
  T* result = columns > 0 ? e + blockIdx.x : e;
  for (int l = 0; l < P.n; ++l) {
    const BottomLevel<T> V(l);
    const int sweeps = l + 1 == P.n ? P.last : P.pre;
    const int unit = l == 0 && columns > 0 ? (int)blockIdx.x : -1;
    const T* start = l == 0 && from_input ? e : nullptr;
    if (slots_of(V.G).units <= (int)blockDim.x)
      bottom_down<DIM, DVAR, CMODE, 1>(L, V, l, P.n, P.res, sweeps, start, unit);
    else
      bottom_down<DIM, DVAR, CMODE, kBottomSlots>(L, V, l, P.n, P.res, sweeps, start, unit);
  }
  for (int l = P.n - 2; l >= 0; --l) {
    const BottomLevel<T> V(l);
    const int unit = l == 0 && columns > 0 ? (int)blockIdx.x : -1;
    T* out = l == 0 ? result : nullptr;
    if (slots_of(V.G).units <= (int)blockDim.x)
      bottom_up<DIM, DVAR, CMODE, 1>(L, V, l, P.post, unit, out, stride);
    else
      bottom_up<DIM, DVAR, CMODE, kBottomSlots>(L, V, l, P.post, unit, out, stride);
  }
  if (P.n == 1) {
    const BottomLevel<T> V(0);
    const BoxLevel& G = V.G;
    const Slots S = slots_of(G);
    const int par = colour_parity(G);
    const int n = G.n[0] * G.n[1] * (DIM == 3 ? G.n[2] : 1);
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
      const int i = t % G.n[0], j = (t / G.n[0]) % G.n[1], k = t / (G.n[0] * G.n[1]);
      result[(long)stride * t] = L[V.e + pos2(par + i + j + k) * S.stride + S.pad + (i >> 1) +
                                   S.row * j + (DIM == 3 ? S.plane * k : 0)];
    }
  }
}

// e = B f with the row-major n x n matrix B, a wavefront per row; FP64 sums.
template <typename T>
__global__ void __launch_bounds__(kThreads)
k_mg_dense(const T* B, int n, const T* f, T* e, const int* stop) {
  if (*stop) return;
  const int row = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (row >= n) return;
  const T* b = B + (long)row * n;
  double acc = 0.0;
#pragma unroll 4
  for (int j = threadIdx.x & 63; j < n; j += 64) acc += (double)b[j] * (double)f[j];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) e[row] = (T)acc;
}

// LDS offsets of the n levels G; false: they do not fit.
template <typename T>
bool bottom_plan(const BoxLevel* G, int n, Bottom<T>& P) {
  if (n < 1 || n > kBottomLevels) return false;
  if (slots_of(G[0]).units > kBottomSlots * kBottomThreads) return false;
  auto cells = [&](int l) { return G[l].n[0] * G[l].n[1] * (G[l].dim == 3 ? G[l].n[2] : 1); };
  long at = 0;
  for (int l = 0; l < n; ++l) {
    P.G[l] = G[l];
    P.e[l] = (int)at;
    at += 2 * slots_of(G[l]).stride;
    P.f[l] = (int)at;
    if (l > 0) at += cells(l);
  }
  P.res = (int)at;
  if (n > 1) at += cells(0);
  P.n = n;
  return at <= kBottomLds;
}

template <typename T>
void bottom_launch(const BoxLevel* G, const BoxArrays* A, int n, const RobinDev& bc, int pre,
                   int post, int last, T* e, int from_input, int columns, const int* stop,
                   hipStream_t s) {
  Bottom<T> P{};
  if (!bottom_plan(G, n, P)) throw hipErrorInvalidValue;
  P.pre = pre;
  P.post = post;
  P.last = last;
  for (int l = 0; l < n; ++l) {
    P.A[l] = typed<T>(A[l]);
    P.R[l] = small_robin<T>(G[l], bc);
  }
  // a constant C takes the code of cell data, half the variants to compile
  const dim3 grid(columns > 0 ? columns : 1), block(small_threads(G[0], true));
  const bool dvar = P.A[0].D[0] != nullptr, c = P.A[0].cmode != 0;
  auto go = [&](auto dim, auto var, auto cmode) {
    constexpr int DIM = decltype(dim)::value, CMODE = decltype(cmode)::value;
    constexpr bool DVAR = decltype(var)::value;
    hipLaunchKernelGGL((k_mg_bottom<DIM, DVAR, CMODE, T>), grid, block, 0, s, P, e, from_input,
                       columns, stop);
  };
  auto coef = [&](auto dim, auto var) {
    if (c) go(dim, var, std::integral_constant<int, 2>{});
    else go(dim, var, std::integral_constant<int, 0>{});
  };
  auto kind = [&](auto dim) {
    if (dvar) coef(dim, std::true_type{});
    else coef(dim, std::false_type{});
  };
  if (G[0].dim == 3) kind(std::integral_constant<int, 3>{});
  else kind(std::integral_constant<int, 2>{});
  check_launch();
}

}  // namespace

int mg_bottom_first(const BoxLevel* G, int n) {
  Bottom<double> P;
  for (int m = 0; m < n; ++m) {
    const BoxLevel& B = G[m];
    if ((long)B.n[0] * B.n[1] * (B.dim == 3 ? B.n[2] : 1) <= kMGDenseCells &&
        bottom_plan(G + m, n - m, P))
      return m;
  }
  return n;
}

void launch_mg_bottom(const BoxLevel* G, const BoxArrays* A, int n, const RobinDev& bc, int pre,
                      int post, int last, double* e, int from_input, int columns,
                      const int* stop, hipStream_t s) {
  if (A[0].fp32)
    bottom_launch<float>(G, A, n, bc, pre, post, last, as<float>(e), from_input, columns, stop, s);
  else
    bottom_launch<double>(G, A, n, bc, pre, post, last, e, from_input, columns, stop, s);
}

void launch_mg_dense(const double* B, int n, const double* f, double* e, int fp32,
                     const int* stop, hipStream_t s) {
  const dim3 grid((n + kThreads / 64 - 1) / (kThreads / 64)), block(kThreads);
  if (fp32)
    hipLaunchKernelGGL(k_mg_dense<float>, grid, block, 0, s, as<float>(B), n, as<float>(f),
                       as<float>(e), stop);
  else
    hipLaunchKernelGGL(k_mg_dense<double>, grid, block, 0, s, B, n, f, e, stop);
  check_launch();
}

}  // namespace sfac
