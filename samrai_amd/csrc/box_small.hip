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

// Units per thread and colour of k_box_lds_rbgs, 0 if the grid-parallel sweep
// is the better one.  Coefficients: what the registers of 512 threads hold,
// 4096 cells in FP64 and 8192 in FP32.  Constant D and C: 4096 cells in 3-D
// (16^3 2.5 us against 8.7; 20^3 spills and takes as long as the grid
// launch's 8.3) and 8192 in 2-D (128 x 64 3.2 us against 4.5).
int small_slots(const BoxLevel& G, bool coefs, bool fp32) {
  const Slots S = slots_of(G);
  const int threads = kSmallThreads(coefs);
  int nc = 1;
  while (nc * threads < S.units) nc *= 2;
  if (nc > (coefs ? (fp32 ? 8 : 4) : (G.dim == 3 ? 2 : 4))) return 0;
  return S.count <= nc * threads && S.pad <= small_pad(nc * threads) ? nc : 0;
}

template <int DIM, bool DVAR, int CMODE>
struct LdsRun {
  template <typename T>
  static void run(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc, const T* uin,
                  T* e0, T* e1, int sweeps, const BoxCheck& K, int check, hipStream_t s) {
    constexpr bool coefs = DVAR || CMODE == 2;
    const int nc = small_slots(G, coefs, sizeof(T) == 4);
    const dim3 grid(1), block(small_threads(G, coefs));
    const SmallRobin<T> R = small_robin<T>(G, bc);
    auto go = [&](auto slots) {
      constexpr int NC = decltype(slots)::value;
      hipLaunchKernelGGL((k_box_lds_rbgs<DIM, DVAR, CMODE, T, NC>), grid, block, 0, s, G, A, R,
                         uin, e0, e1, sweeps, K, check);
    };
    if (nc == 1) go(std::integral_constant<int, 1>{});
    else if (nc == 2) go(std::integral_constant<int, 2>{});
    else if (nc == 4) go(std::integral_constant<int, 4>{});
    else if (nc == 8 && coefs && sizeof(T) == 4)
      go(std::integral_constant<int, coefs && sizeof(T) == 4 ? 8 : 4>{});
    else throw hipErrorInvalidValue;
    check_launch();
  }
};

}  // namespace

bool box_lds_fits(const BoxLevel& G, const BoxArrays& A) {
  return small_slots(G, A.D[0] != nullptr || A.cmode == 2, A.fp32 != 0) > 0;
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
