// Red-black sweeps of a level in one work-group (box_small.h).
#include "box_small.h"

#include <type_traits>

namespace sfac {
namespace {

// Slots held on each side of a colour array of `slots` slots.
constexpr int small_pad(int slots) { return slots <= 2048 ? slots / 4 : 512; }

// `sweeps` red-black sweeps (fewer if the early-exit test of BoxCheck stops
// them), u from uin to the buffer e0 or e1 by the parity of the sweeps done.
// Every sweep's test needs only whether some |residual| of the last patch is
// above the tolerance, one LDS word; the largest is formed once at the end.
template <int DIM, bool DVAR, int CMODE, typename T, int NC>
__global__ void __launch_bounds__(kSmallThreads(DVAR || CMODE == 2))
k_box_lds_rbgs(BoxLevel G, BoxArraysT<T> A, SmallRobin<T> R, const T* uin, T* e0, T* e1,
               int sweeps, BoxCheck K, int check) {
  constexpr int kSlots = NC * kSmallThreads(DVAR || CMODE == 2);
  __shared__ T E[2 * (kSlots + 2 * small_pad(kSlots))];
  __shared__ int above[3];
  __shared__ double wm[16];
  if (!check && K.stop && *K.stop) return;
  const Slots S = slots_of(G);
  const SmallConst<T> s = small_const<DIM, DVAR, CMODE>(G, A);
  SmallCells<T, NC> q;
  small_load<DIM, DVAR, CMODE>(G, A, S, s, q);
  small_start(E, uin, S, q);
  if (threadIdx.x < 3) above[threadIdx.x] = 0;
  __syncthreads();
  int done = 0;
  bool stop = false;
  double mr = 0.0;
  while (done < sweeps && !stop) {
    mr = (double)small_colour<DIM, DVAR, CMODE>(E, 0, S, q, s, R, check != 0);
    __syncthreads();
    mr = fmax(mr, (double)small_colour<DIM, DVAR, CMODE>(E, 1, S, q, s, R, check != 0));
    if (check) {
      // the word of the next sweep, whose last readers passed the barrier above
      if (threadIdx.x == 0) above[(done + 1) % 3] = 0;
      if (__any(mr > K.tol) && (threadIdx.x & 63) == 0) above[done % 3] = 1;
    }
    __syncthreads();
    if (check) stop = above[done % 3] == 0;
    ++done;
  }
  T* out = (done & 1) ? e1 : e0;
#pragma unroll
  for (int v = 0; v < NC; ++v)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if (q.flags[c][v]) out[q.flags[c][v] >> 8] = q.u[c][v];
  if (check) {
    for (int o = 32; o > 0; o >>= 1) mr = fmax(mr, __shfl_xor(mr, o, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = mr;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < (int)blockDim.x / 64; ++w) mr = fmax(mr, wm[w]);
      *K.sweeps = done;
      if (K.maxres_out) *K.maxres_out = mr;
      if (stop) *K.stop = 1;
    }
  }
}

// Most units per thread and colour compiled in, where k_box_lds_rbgs is faster
// than two sweeps per launch (box_pair.hip).  us per sweep with the early-exit
// test, against that:
//   coefficients: four, 15^3 D 4.4 (5.2), D and C 5.5 (5.3), 16^3 3.1 (5.0),
//     4.3 (5.1), FP32 2.4 (5.1), 64 x 64 1.8 (2.9); eight spill, in 3-D up to
//     211 registers, and take 11 (5.1) on 20^3, but 2-D FP32 2.5 (3.0) on 90 x 90;
//   constant D and C: two, 16^3 2.6 (4.5), 64 x 64 1.5 (2.9); four, 90 x 90
//     3.1 (3.0), FP32 2.1 (2.9).
template <int DIM, typename T>
constexpr int kSmallSlots(bool coefs) {
  return DIM == 2 && sizeof(T) == 4 ? (coefs ? 8 : 4) : (coefs ? 4 : 2);
}
// A launch reads its coefficients once and pays for it over its sweeps: with
// four units and more it takes 5 to 13 us longer to start than a pair, so
// calls of few sweeps (two on 16^3: 53.5 against 48.4, 64 x 64 38.4 (33.3))
// go to pairs.
constexpr int kSmallFewSweeps = 16, kSmallFewSlots = 2;

// Units per thread and colour of k_box_lds_rbgs for a call of that many
// sweeps, 0 if it is not the better one.
int small_slots(const BoxLevel& G, bool coefs, bool fp32, int sweeps) {
  const Slots S = slots_of(G);
  const int threads = kSmallThreads(coefs);
  int nc = 1;
  while (nc * threads < S.units) nc *= 2;
  int most = G.dim == 3 ? kSmallSlots<3, double>(coefs)
                        : (fp32 ? kSmallSlots<2, float>(coefs) : kSmallSlots<2, double>(coefs));
  if (coefs && sweeps < kSmallFewSweeps) most = kSmallFewSlots;
  if (nc > most) return 0;
  return S.count <= nc * threads && S.pad <= small_pad(nc * threads) ? nc : 0;
}

template <int DIM, bool DVAR, int CMODE>
struct LdsRun {
  template <typename T>
  static void run(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc, const T* uin,
                  T* e0, T* e1, int sweeps, const BoxCheck& K, int check, hipStream_t s) {
    constexpr bool coefs = DVAR || CMODE == 2;
    constexpr int most = kSmallSlots<DIM, T>(coefs);
    const int nc = small_slots(G, coefs, sizeof(T) == 4, sweeps);
    const dim3 grid(1), block(small_threads(G, coefs));
    const SmallRobin<T> R = small_robin<T>(G, bc);
    auto go = [&](auto slots) {
      constexpr int NC = decltype(slots)::value;
      hipLaunchKernelGGL((k_box_lds_rbgs<DIM, DVAR, CMODE, T, NC>), grid, block, 0, s, G, A, R,
                         uin, e0, e1, sweeps, K, check);
    };
    if (nc == 1) go(std::integral_constant<int, 1>{});
    else if (nc == 2) go(std::integral_constant<int, 2>{});
    else if (nc == 4 && most >= 4) go(std::integral_constant<int, most >= 4 ? 4 : 2>{});
    else if (nc == 8 && most >= 8) go(std::integral_constant<int, most >= 8 ? 8 : 2>{});
    else throw hipErrorInvalidValue;
    check_launch();
  }
};

}  // namespace

bool box_lds_pays(const BoxLevel& G, const BoxArrays& A, int sweeps) {
  return small_slots(G, A.D[0] != nullptr || A.cmode == 2, A.fp32 != 0, sweeps) > 0;
}

void launch_box_lds_rbgs(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc,
                         const double* uin, double* e0, double* e1, int sweeps,
                         const BoxCheck& K, int check, hipStream_t s) {
  if (A.fp32)
    dispatch3<LdsRun>(G, typed<float>(A), bc, as<float>(uin), as<float>(e0), as<float>(e1),
                      sweeps, K, check, s);
  else
    dispatch3<LdsRun>(G, typed<double>(A), bc, uin, e0, e1, sweeps, K, check, s);
}

}  // namespace sfac
