// Two red-black sweeps of a single-rectangle level per launch (gfx950).
//
// A sweep of a level of 10^4 to 10^5 cells takes 5 to 6 us whatever its tiles
// are: the launch, one round trip to memory and the steps of one tile, with
// the machine mostly idle.  Here a work-group stages its tile grown by four
// cells and takes both sweeps in LDS, red on the tile grown by three, black on
// it grown by two, red by one, black on the tile; what neighbouring tiles
// compute too comes from the same inputs in the same expression order, so the
// values are those of two k_box_rbgs launches bit for bit.  The idle units pay
// for the redundant cells (4.4 cells' coefficients loaded per owned one at
// 8x8x8).  A cell's coefficients are read and its diagonal inverted once for
// both sweeps, and the physical ghosts are formed inside the updates (the cell
// is its face ghost's only interior neighbour).
// us per sweep, FP64, without and with the early-exit test, against single
// sweeps with their best tile: variable D 32^3 4.3, 4.9 (5.6, 7.3), 45 x 58 x 39
// 5.7, 6.3 (6.3, 8.3), 248 x 184 2.4, 3.5 (3.8, 7.9).  At 64^3 pairs took 10.4,
// 11.4 (7.4, 10.3): the redundant cells cost more than the launches.
// All of a colour's reads at once (as in box_small.hip) spilled and was slower,
// 32^3 5.4.
#include "box_small.h"

#include <type_traits>

namespace sfac {
namespace {

template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline T pair_update(T* U, int q, int SY, int SZ, int fl, const Coef<T>& k, T dudr,
                                const SmallConst<T>& s, const SmallRobin<T>& R) {
  const T uc = U[q];
  T n[6] = {U[q - 1], U[q + 1], U[q - SY], U[q + SY], DIM == 3 ? U[q - SZ] : (T)0,
            DIM == 3 ? U[q + SZ] : (T)0};
  if (fl & 63) {
#pragma unroll
    for (int loc = 0; loc < 2 * DIM; ++loc)
      if (fl & (1 << loc)) n[loc] = small_ghost<DIM>(R, loc, uc);
  }
  const T fxl = (DVAR ? k.xl : s.kx) * (uc - n[0]);
  const T fxh = (DVAR ? k.xh : s.kx) * (n[1] - uc);
  const T fyl = (DVAR ? k.yl : s.ky) * (uc - n[2]);
  const T fyh = (DVAR ? k.yh : s.ky) * (n[3] - uc);
  T div = s.dxi * (fxh - fxl) + s.dyi * (fyh - fyl);
  if (DIM == 3) {
    const T fzl = (DVAR ? k.zl : s.kz) * (uc - n[4]);
    const T fzh = (DVAR ? k.zh : s.kz) * (n[5] - uc);
    div = div + s.dzi * (fzh - fzl);
  }
  const T res = CMODE == 0 ? k.f - div : k.f - div - (CMODE == 2 ? k.c : s.cc) * uc;
  const T du = -res * ((DVAR || CMODE == 2) ? dudr : s.dudr);
  U[q] = uc + du;
  return fabs(res);
}

// flags of a cell: 0-5 faces on the physical boundary, 6 updated in the first
// sweep, 7 in the second, 8 owned and in the last patch.
template <int DIM, bool DVAR, int CMODE, int TX, int TY, int TZ, int NT, typename T>
__global__ void __launch_bounds__(NT)
k_box_pair(BoxLevel G, BoxArraysT<T> A, SmallRobin<T> R, PairCheck K, int sweeps, int ntx, int nty,
           int ntiles, int per_xcd) {
  constexpr int H = 4, HZ = DIM == 3 ? H : 0;
  constexpr int LX = TX + 2 * H, LY = TY + 2 * H, LZ = DIM == 3 ? TZ + 2 * H : 1;
  constexpr int SY = LX, SZ = LX * LY, NL = SZ * LZ;
  __shared__ T U[NL];
  __shared__ double wm[2][NT / 64];
  const int b = blockIdx.x;
  const T* ein = A.ein;
  T* eout = A.eout;
  if (K.slots) {
    // the pair before this launch: where it stopped, if it did.  A launch
    // marks its decision with its own number, so that its other work-groups,
    // which may see the mark, take the same one.
    const int flag = *K.stop;
    if (flag != 0 && flag != K.launch + 1) return;
    if (K.launch > 0) {
      const int prev = (K.launch + 2) % 3;
      const double m0 = __longlong_as_double((long long)K.slots[2 * prev]);
      const double m1 = __longlong_as_double((long long)K.slots[2 * prev + 1]);
      const bool after0 = !(m0 > K.tol), after1 = K.prev == 2 && !(m1 > K.tol);
      const bool stop = after0 || after1, last = K.final != 0;
      if ((stop || last) && b == 0 && threadIdx.x == 0) {
        const bool first = after0 || K.prev == 1;
        *K.sweeps = 2 * (K.launch - 1) + (first ? 1 : 2);
        *K.buffer = K.launch & 1;
        if (K.maxres_out) *K.maxres_out = first ? m0 : m1;
        if (stop) *K.stop = K.launch + 1;
      }
      if (after0 && K.prev == 2) {
        // stopped after the first sweep of the pair: that sweep again from
        // the pair's input, over its result
        ein = A.eout;
        eout = const_cast<T*>(A.ein);
        sweeps = 1;
      } else if (stop || last) {
        return;
      }
    }
    if (b == 0 && threadIdx.x == 0) {
      const int next = (K.launch + 1) % 3;
      K.slots[2 * next] = 0ull;
      K.slots[2 * next + 1] = 0ull;
    }
  } else if (K.stop && *K.stop) {
    return;
  }
  const int t = (b & 7) * per_xcd + (b >> 3);  // XCD-aware tile order (k_box_rbgs)
  if (t >= ntiles) return;
  const int tx = t % ntx, ty = (t / ntx) % nty, tz = t / (ntx * nty);
  const int x0 = tx * TX - H, y0 = ty * TY - H, z0 = DIM == 3 ? tz * TZ - H : 0;
  const int n0 = G.n[0], n1 = G.n[1], n2 = DIM == 3 ? G.n[2] : 1;
  const long plane = (long)n0 * n1;

  // the staged tile
  constexpr int NE = (NL + NT - 1) / NT;
  T v[NE];
#pragma unroll
  for (int c = 0; c < NE; ++c) {
    const int q = threadIdx.x + c * NT;
    const int i = x0 + q % LX, j = y0 + (q / LX) % LY, k = DIM == 3 ? z0 + q / SZ : 0;
    const bool in = ein && q < NL && i >= 0 && i < n0 && j >= 0 && j < n1 && k >= 0 && k < n2;
    v[c] = in ? ein[i + (long)n0 * j + plane * k] : (T)0;
  }
  // this thread's red cells (tile grown by three) and black ones (by two)
  const int par = pos2(colour_parity(G) + x0 + y0 + z0);
  constexpr int RX = (TX + 6) / 2, RY = TY + 6, RZ = DIM == 3 ? TZ + 6 : 1;
  constexpr int BX = (TX + 4) / 2, BY = TY + 4, BZ = DIM == 3 ? TZ + 4 : 1;
  constexpr int NRW = RX * RY * RZ, NR = (NRW + NT - 1) / NT;
  constexpr int NBW = BX * BY * BZ, NB = (NBW + NT - 1) / NT;
  const SmallConst<T> s = small_const<DIM, DVAR, CMODE>(G, A);
  auto setup = [&](int lx, int ly, int lz, bool valid, int second, int& q, int& fl, Coef<T>& k,
                   T& dudr) {
    const int i = x0 + lx, j = y0 + ly, kk = DIM == 3 ? z0 + lz : 0;
    q = lx + SY * ly + SZ * lz;
    fl = 0;
    k = Coef<T>{};
    dudr = (T)0;
    if (!valid || i < 0 || i >= n0 || j < 0 || j >= n1 || kk < 0 || kk >= n2) return;
    // distance to the tile
    const int d = max(max(max(H - lx, lx - (TX + H - 1)), max(H - ly, ly - (TY + H - 1))),
                      DIM == 3 ? max(HZ - lz, lz - (TZ + H - 1)) : 0);
    const bool lp = d <= 0 && i >= G.lp_lo[0] && i <= G.lp_hi[0] && j >= G.lp_lo[1] &&
                    j <= G.lp_hi[1] && (DIM == 2 || (kk >= G.lp_lo[2] && kk <= G.lp_hi[2]));
    fl = 64 | (d <= second ? 128 : 0) | (lp ? 256 : 0) | (i == 0 ? 1 : 0) |
         (i == n0 - 1 ? 2 : 0) | (j == 0 ? 4 : 0) | (j == n1 - 1 ? 8 : 0) |
         (DIM == 3 ? (kk == 0 ? 16 : 0) | (kk == n2 - 1 ? 32 : 0) : 0);
    k = load_coef<DIM, DVAR, CMODE>(G, A, i, j, kk);
  };
  int rq[NR], rf[NR], bq[NB], bf[NB];
  Coef<T> rk[NR], bk[NB];
  T rd[NR], bd[NB];
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    const int w = threadIdx.x + u * NT;
    const int ly = 1 + (w / RX) % RY, lz = DIM == 3 ? 1 + w / (RX * RY) : 0;
    const int lx = 1 + pos2(par + 1 + ly + lz) + 2 * (w % RX);
    setup(lx, ly, lz, w < NRW, 1, rq[u], rf[u], rk[u], rd[u]);
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int w = threadIdx.x + u * NT;
    const int ly = 2 + (w / BX) % BY, lz = DIM == 3 ? 2 + w / (BX * BY) : 0;
    const int lx = 2 + pos2(par + 1 + ly + lz) + 2 * (w % BX);
    setup(lx, ly, lz, w < NBW, 0, bq[u], bf[u], bk[u], bd[u]);
  }
#pragma unroll
  for (int c = 0; c < NE; ++c)
    if (threadIdx.x + c * NT < NL) U[threadIdx.x + c * NT] = v[c];
  if (DVAR || CMODE == 2) {
    auto finish = [&](int fl, Coef<T>& k, T& dudr) {
      if (!fl) return;
      dudr = cell_dudr<DIM, DVAR, CMODE>(k, G, A);
      k.xl = s.dxi * k.xl;
      k.xh = s.dxi * k.xh;
      k.yl = s.dyi * k.yl;
      k.yh = s.dyi * k.yh;
      k.zl = s.dzi * k.zl;
      k.zh = s.dzi * k.zh;
    };
#pragma unroll
    for (int u = 0; u < NR; ++u) finish(rf[u], rk[u], rd[u]);
#pragma unroll
    for (int u = 0; u < NB; ++u) finish(bf[u], bk[u], bd[u]);
  }
  __syncthreads();
  double mr[2] = {0.0, 0.0};
#pragma unroll
  for (int sw = 0; sw < 2; ++sw) {
    if (sw < sweeps) {
      // with one sweep only the tile's own red and black cells matter, and the
      // wider region of the first sweep holds them
      const int need = sw == 0 ? 64 : 128;
#pragma unroll
      for (int u = 0; u < NR; ++u)
        if (rf[u] & need) {
          const T r = pair_update<DIM, DVAR, CMODE>(U, rq[u], SY, SZ, rf[u], rk[u], rd[u], s, R);
          if (rf[u] & 256) mr[sw] = fmax(mr[sw], (double)r);
        }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < NB; ++u)
        if (bf[u] & need) {
          const T r = pair_update<DIM, DVAR, CMODE>(U, bq[u], SY, SZ, bf[u], bk[u], bd[u], s, R);
          if (bf[u] & 256) mr[sw] = fmax(mr[sw], (double)r);
        }
      __syncthreads();
    }
  }
  for (int w = threadIdx.x; w < TX * TY * (DIM == 3 ? TZ : 1); w += NT) {
    const int ox = w % TX, oy = (w / TX) % TY, oz = w / (TX * TY);
    const int i = x0 + H + ox, j = y0 + H + oy, k = DIM == 3 ? z0 + H + oz : 0;
    if (i < n0 && j < n1 && k < n2)
      eout[i + (long)n0 * j + plane * k] = U[(ox + H) + SY * (oy + H) + SZ * (oz + HZ)];
  }
  if (K.slots) {
    const bool meets = x0 + H <= G.lp_hi[0] && x0 + H + TX > G.lp_lo[0] && y0 + H <= G.lp_hi[1] &&
                       y0 + H + TY > G.lp_lo[1] &&
                       (DIM == 2 || (z0 + H <= G.lp_hi[2] && z0 + H + TZ > G.lp_lo[2]));
    if (meets) {  // uniform over the work-group
#pragma unroll
      for (int sw = 0; sw < 2; ++sw) {
        double m = mr[sw];
        for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
        if ((threadIdx.x & 63) == 0) wm[sw][threadIdx.x >> 6] = m;
      }
      __syncthreads();
      if (threadIdx.x < 2) {
        double m = wm[threadIdx.x][0];
        for (int w = 1; w < NT / 64; ++w) m = fmax(m, wm[threadIdx.x][w]);
        raise_max(K.slots + 2 * (K.launch % 3) + threadIdx.x, m);
      }
    }
  }
}

template <int DIM, bool DVAR, int CMODE, int TX, int TY, int TZ, int NT, typename T>
void pair_tile(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc, const PairCheck& K,
               int sweeps, hipStream_t s) {
  const int ntx = (G.n[0] + TX - 1) / TX, nty = (G.n[1] + TY - 1) / TY;
  const int ntz = DIM == 3 ? (G.n[2] + TZ - 1) / TZ : 1;
  const int ntiles = ntx * nty * ntz, per_xcd = (ntiles + 7) / 8;
  hipLaunchKernelGGL((k_box_pair<DIM, DVAR, CMODE, TX, TY, TZ, NT, T>), dim3(8 * per_xcd),
                     dim3(NT), 0, s, G, A, small_robin<T>(G, bc), K, sweeps, ntx, nty, ntiles,
                     per_xcd);
  check_launch();
}

template <int DIM, bool DVAR, int CMODE>
struct PairRun {
  template <typename T>
  static void run(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc,
                  const PairCheck& K, int sweeps, hipStream_t s) {
    if constexpr (DIM == 2)
      pair_tile<2, DVAR, CMODE, 16, 16, 1, 256>(G, A, bc, K, sweeps, s);
    else if ((long)G.n[0] * G.n[1] * G.n[2] <= kPairSmallTile)
      pair_tile<3, DVAR, CMODE, 8, 8, 4, 512>(G, A, bc, K, sweeps, s);
    else
      pair_tile<3, DVAR, CMODE, 8, 8, 8, 512>(G, A, bc, K, sweeps, s);
  }
};

}  // namespace

bool box_pair_pays(const BoxLevel& G) {
  const long n = (long)G.n[0] * G.n[1] * (G.dim == 3 ? G.n[2] : 1);
  return n <= (G.dim == 3 ? kPairCells3 : kPairCells2);
}

void launch_box_pair(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc,
                     const PairCheck& K, int sweeps, hipStream_t s) {
  if (A.fp32) dispatch3<PairRun>(G, typed<float>(A), bc, K, sweeps, s);
  else dispatch3<PairRun>(G, typed<double>(A), bc, K, sweeps, s);
}

}  // namespace sfac
