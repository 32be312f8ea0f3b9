// Colour-fused red-black sweeps over a single-rectangle level (gfx950).
//
// Per work-group: one TX x TY x TZ tile of owned cells.  LDS holds the tile
// grown by two cells on every side (clipped to the level, plus the physical
// ghost layer).  Per launch:
//   1. early-exit test of the previous sweep (every work-group reads the
//      same max-residual word, so all of them take the same decision);
//   2. load u; compute the face ghosts of the physical boundary in LDS;
//   3. red update on the tile grown by one (halo reds are recomputed from the
//      same inputs as their owning tile, so they are bit-identical);
//   4. refresh the face ghosts from the updated reds;
//   5. black update on the owned tile; write the owned tile back.
// The per-cell arithmetic is rbgswithfluxmax{vardc,condc}{varsf,consf}3d /
// 2d (solv_cellpoissonfacops3d.f:136-481, 2d :95-364) in its expression
// order, and the ghosts are settype1cells (solv_cartesianrobinbchelper3d.f),
// as in the level-batched kernels.  Edge and corner ghosts are not read by
// the 7-point (5-point) stencil, so they are not formed here; the caller's
// final ghost fill sets them in the patches.
//
// Every kernel is templated on the storage type T: double is the reference
// arithmetic; float is the mixed-precision coarse solve (FP32 storage and
// arithmetic inside the FP64 FAC iteration), with the same expression order.
#include "box_device.h"

namespace sfac {
namespace {

__device__ inline bool same_bits(double a, double b) {
  return __double_as_longlong(a) == __double_as_longlong(b);
}
__device__ inline bool same_bits(float a, float b) { return __float_as_int(a) == __float_as_int(b); }

// Work-group max of v (kThreads threads); result valid in thread 0.
__device__ inline double block_max(double v, double* wm) {
  for (int s = 32; s > 0; s >>= 1) v = fmax(v, __shfl_xor(v, s, 64));
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < kThreads / 64; ++w) v = fmax(v, wm[w]);
  return v;
}

// Value of the lane that CTRL (a data-parallel primitive's control) names.
template <int CTRL>
__device__ inline double lane_value(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Largest |residual| of the sweep that raised slot s, the same in every lane: a
// lane reads one word of the slot (one load for all; read in turn they cost
// 0.4 us), then the maximum over eight lanes.
__device__ inline double slot_max(const unsigned long long* slots, int s) {
  static_assert(kCheckWords == 8, "three steps");
  double m = __longlong_as_double(
      (long long)slots[s * kCheckSlot + threadIdx.x % kCheckWords * kCheckLine]);
  m = fmax(m, lane_value<0xb1>(m));   // neighbours in a pair (quad_perm 1, 0, 3, 2)
  m = fmax(m, lane_value<0x4e>(m));   // the other pair of four (quad_perm 2, 3, 0, 1)
  m = fmax(m, lane_value<0x141>(m));  // the other four of eight (row_half_mirror)
  const long long b = __double_as_longlong(m);
  return __longlong_as_double(((long long)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                              (unsigned int)__builtin_amdgcn_readfirstlane((int)b));
}

// Early-exit test of the previous sweep (see BoxCheck).  Every wave reads
// the stop flag and the previous sweep's max-residual words itself (no
// barrier): all read the same words and take the same decision (a stop that
// work-group 0 records during this sweep follows from the same test), and
// work-group 0 records it.  true: skip this sweep.
__device__ inline bool stop_sweep(const BoxCheck& K, int b) {
  if (!K.stop) return false;
  bool stop;
  if (K.slots && K.sweep > 0) {
    // all are read unconditionally, so that their loads are in flight
    // together (one memory round trip before the decision)
    const int flag = *K.stop;
    const double m = slot_max(K.slots, (K.sweep + 2) % 3);
    const bool now = !(m > K.tol);
    stop = (flag != 0) | now;
    if (flag == 0 && now && b == 0 && threadIdx.x == 0) {
      *K.stop = 1;
      *K.sweeps = K.sweep;
      if (K.maxres_out) *K.maxres_out = m;
    }
  } else {
    stop = *K.stop != 0;
  }
  // the slot the next sweep raises (its last reader was the previous sweep)
  if (!stop && K.slots && b == 0 && threadIdx.x < kCheckWords)
    K.slots[(K.sweep + 1) % 3 * kCheckSlot + threadIdx.x * kCheckLine] = 0ull;
  return stop;
}

template <int DIM, bool DVAR, int CMODE, int TX, int TY, int TZ, typename T>
__global__ void __launch_bounds__(kThreads)
k_box_rbgs(BoxLevel G, BoxArraysT<T> A, RobinDev bc, int homogeneous, BoxCheck K, int ntx,
           int nty, int ntiles, int per_xcd) {
  constexpr int LX = TX + 4, LY = TY + 4, LZ = DIM == 3 ? TZ + 4 : 1;
  constexpr int SY = LX, SZ = LX * LY;
  constexpr int ZH = DIM == 3 ? 2 : 0;  // LDS halo along z
  __shared__ T U[LX * LY * LZ];
  __shared__ double wm[kThreads / 64];
  // XCD-aware tile order: work-groups are dealt round-robin to the 8 XCDs,
  // so consecutive tiles (one slab of the level) share an XCD's L2.
  const int b = blockIdx.x;

  // 1. early exit (first, so that its loads overlap the tile set-up)
  if (stop_sweep(K, b)) return;

  const int t = (b & 7) * per_xcd + (b >> 3);
  if (t >= ntiles) return;
  const int tx = t % ntx, ty = (t / ntx) % nty, tz = t / (ntx * nty);
  const int x0 = tx * TX, y0 = ty * TY, z0 = DIM == 3 ? tz * TZ : 0;
  const int n0 = G.n[0], n1 = G.n[1], n2 = DIM == 3 ? G.n[2] : 1;

  // colour parity: red <=> (ilev + jlev + klev + shift) even; in LDS
  // coordinates the sum is base + lx + ly + lz
  const int base = G.lo[0] + G.lo[1] + (DIM == 3 ? G.lo[2] : 0) + x0 + y0 + z0 - 4 - ZH + G.shift;
  const int pb = pos2(base);
  // red cells: half-rows of the tile grown by one; black: of the owned tile
  constexpr int HX = (TX + 2) / 2, RY = TY + 2, RZ = DIM == 3 ? TZ + 2 : 1;
  constexpr int NRW = HX * RY * RZ, NR = (NRW + kThreads - 1) / kThreads;
  constexpr int HB = TX / 2, BZ = DIM == 3 ? TZ : 1;
  constexpr int NBW = HB * TY * BZ, NB = (NBW + kThreads - 1) / kThreads;
  auto red_cell = [&](int w, int& lx, int& ly, int& lz) {
    const int m = w % HX;
    ly = 1 + (w / HX) % RY;
    lz = DIM == 3 ? 1 + w / (HX * RY) : 0;
    lx = 1 + pos2(pb + 1 + ly + lz) + 2 * m;
  };
  auto black_cell = [&](int w, int& lx, int& ly, int& lz) {
    const int m = w % HB;
    ly = 2 + (w / HB) % TY;
    lz = DIM == 3 ? 2 + w / (HB * TY) : 0;
    lx = 3 - pos2(pb + ly + lz) + 2 * m;
  };
  auto inside = [&](int i, int j, int k) {
    return i >= 0 && i < n0 && j >= 0 && j < n1 && (DIM == 2 || (k >= 0 && k < n2));
  };

  // 2. issue every global load of the sweep up front: the grown tile of u
  // and the coefficients of each cell this thread updates
  // u: each thread loads whole z-columns of the grown tile (one index
  // decomposition per column, then a fixed stride per plane)
  constexpr int NCOL = (LX * LY + kThreads - 1) / kThreads;
  const long plane = (long)n0 * n1;
  T v[NCOL][LZ];
#pragma unroll
  for (int c = 0; c < NCOL; ++c) {
    const int col = threadIdx.x + c * kThreads;
    const int lx = col % LX, ly = col / LX;
    const int i = x0 - 2 + lx, j = y0 - 2 + ly;
    // ein == nullptr: u = 0 before the sweep (nothing to load)
    const bool xy = A.ein && col < LX * LY && i >= 0 && i < n0 && j >= 0 && j < n1;
    const T* src = A.ein + ((long)i + (long)n0 * j);
#pragma unroll
    for (int lz = 0; lz < LZ; ++lz) {
      const int k = z0 - ZH + lz;
      v[c][lz] = (xy && (DIM == 2 || (k >= 0 && k < n2))) ? src[plane * k] : (T)0;
    }
  }
  // the cells this thread updates: LDS index, flags (1 update, 2 counts
  // for the early-exit maximum) and coefficients
  const bool lp_tile = K.slots != nullptr;
  auto in_lp = [&](int i, int j, int k) {
    return i >= G.lp_lo[0] && i <= G.lp_hi[0] && j >= G.lp_lo[1] && j <= G.lp_hi[1] &&
           (DIM == 2 || (k >= G.lp_lo[2] && k <= G.lp_hi[2]));
  };
  Coef<T> cr[NR], cb[NB];
  int rq[NR], rf[NR], bq[NB], bf[NB];
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    const int w = threadIdx.x + u * kThreads;
    int lx, ly, lz;
    red_cell(w, lx, ly, lz);
    const int i = x0 - 2 + lx, j = y0 - 2 + ly, k = z0 - ZH + lz;
    const bool act = w < NRW && inside(i, j, k);
    const bool own = lx >= 2 && lx < TX + 2 && ly >= 2 && ly < TY + 2 &&
                     (DIM == 2 || (lz >= 2 && lz < TZ + 2));
    rq[u] = lx + SY * ly + SZ * lz;
    rf[u] = (act ? 1 : 0) | ((act && lp_tile && own && in_lp(i, j, k)) ? 2 : 0);
    cr[u] = act ? load_coef<DIM, DVAR, CMODE>(G, A, i, j, k) : Coef<T>{};
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int w = threadIdx.x + u * kThreads;
    int lx, ly, lz;
    black_cell(w, lx, ly, lz);
    const int i = x0 - 2 + lx, j = y0 - 2 + ly, k = z0 - ZH + lz;
    const bool act = w < NBW && inside(i, j, k);
    bq[u] = lx + SY * ly + SZ * lz;
    bf[u] = (act ? 1 : 0) | ((act && lp_tile && in_lp(i, j, k)) ? 2 : 0);
    cb[u] = act ? load_coef<DIM, DVAR, CMODE>(G, A, i, j, k) : Coef<T>{};
  }
#pragma unroll
  for (int c = 0; c < NCOL; ++c) {
    const int col = threadIdx.x + c * kThreads;
    if (col < LX * LY)
#pragma unroll
      for (int lz = 0; lz < LZ; ++lz) U[col + SZ * lz] = v[c][lz];
  }
  __syncthreads();

  // face ghosts of the physical boundary that fall inside the LDS tile
  auto ghosts = [&]() {
    for (int a = 0; a < DIM; ++a)
      for (int side = 0; side < 2; ++side) {
        const int org[3] = {x0 - 2, y0 - 2, z0 - ZH};
        const int gidx = side ? G.n[a] : -1;     // ghost index along a
        const int l = gidx - org[a];
        const int lext[3] = {LX, LY, LZ};
        if (l < 0 || l >= lext[a]) continue;
        const int t1 = a == 0 ? 1 : 0, t2 = a == 2 ? 1 : 2;
        const int e1 = lext[t1], e2 = DIM == 3 ? lext[t2] : 1;
        for (int w = threadIdx.x; w < e1 * e2; w += kThreads) {
          int lc[3];
          lc[a] = l;
          lc[t1] = w % e1;
          lc[t2] = w / e1;
          const int g1 = org[t1] + lc[t1], g2 = org[t2] + lc[t2];
          if (g1 < 0 || g1 >= G.n[t1]) continue;
          if (DIM == 3 && (g2 < 0 || g2 >= G.n[t2])) continue;
          const int q = lc[0] + SY * lc[1] + SZ * lc[2];
          const int stride = a == 0 ? 1 : (a == 1 ? SY : SZ);
          const T uin = U[side ? q - stride : q + stride];
          U[q] = robin_ghost<DIM>(G, bc, homogeneous, 2 * a + side, uin);
        }
      }
  };
  ghosts();
  __syncthreads();

  double mr = 0.0;
  // constant D and C: one reciprocal diagonal for the whole level
  const T dudr_c = (!DVAR && CMODE != 2) ? cell_dudr<DIM, DVAR, CMODE>(Coef<T>{}, G, A) : (T)0;

  // 3. red cells of the tile grown by one
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    if (rf[u] & 1) {
      const T dudr = (!DVAR && CMODE != 2) ? dudr_c : cell_dudr<DIM, DVAR, CMODE>(cr[u], G, A);
      const T ra = cell_update<DIM, DVAR, CMODE>(U, rq[u], SY, SZ, SZ, cr[u], G, A, dudr);
      if (rf[u] & 2) mr = fmax(mr, (double)ra);
    }
  }
  __syncthreads();
  ghosts();
  __syncthreads();

  // 5. black cells of the owned tile
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    if (bf[u] & 1) {
      const T dudr = (!DVAR && CMODE != 2) ? dudr_c : cell_dudr<DIM, DVAR, CMODE>(cb[u], G, A);
      const T ra = cell_update<DIM, DVAR, CMODE>(U, bq[u], SY, SZ, SZ, cb[u], G, A, dudr);
      if (bf[u] & 2) mr = fmax(mr, (double)ra);
    }
  }
  __syncthreads();
  constexpr int NOC = (TX * TY + kThreads - 1) / kThreads;
#pragma unroll
  for (int c = 0; c < NOC; ++c) {
    const int col = threadIdx.x + c * kThreads;
    const int ox = col % TX, oy = col / TX;
    const int i = x0 + ox, j = y0 + oy;
    if (col >= TX * TY || i >= n0 || j >= n1) continue;
    T* dst = A.eout + ((long)i + (long)n0 * j);
    const T* src = U + (ox + 2) + SY * (oy + 2) + SZ * ZH;
#pragma unroll
    for (int oz = 0; oz < (DIM == 3 ? TZ : 1); ++oz)
      if (DIM == 2 || z0 + oz < n2) dst[plane * (z0 + oz)] = src[SZ * oz];
  }
  if (lp_tile) {
    const int ti[3] = {tx - K.tlo[0], ty - K.tlo[1], DIM == 3 ? tz - K.tlo[2] : 0};
    const bool meets = ti[0] >= 0 && ti[0] < K.tn[0] && ti[1] >= 0 && ti[1] < K.tn[1] &&
                       ti[2] >= 0 && ti[2] < K.tn[2];
    if (meets) {  // uniform over the work-group
      mr = block_max(mr, wm);
      if (threadIdx.x == 0)
        atomicMax(K.slots + K.sweep % 3 * kCheckSlot + b % kCheckWords * kCheckLine,
                  (unsigned long long)__double_as_longlong(mr));
    }
  }
}

__global__ void __launch_bounds__(kThreads) k_box_final_check(BoxCheck K, int nsweeps) {
  if (*K.stop) return;  // stopped early: already recorded
  const double m = slot_max(K.slots, (nsweeps - 1) % 3);
  if (threadIdx.x == 0) {
    *K.sweeps = nsweeps;
    if (K.maxres_out) *K.maxres_out = m;
    if (!(m > K.tol)) *K.stop = 1;
  }
}

template <typename T, typename PT = double>
__global__ void __launch_bounds__(kThreads)
k_box_cells(const BoxItem* items, const Chunk* chunks, LevelGeom L, PT* const* x, int g,
            T* box0, T* box1, const int* count, int count_host, BoxLevel G, int to_box) {
  T* box = ((count ? *count : count_host) & 1) ? box1 : box0;
  const Chunk ch = chunks[xcd_chunk()];
  if (ch.item < 0) return;
  const BoxItem it = items[ch.item];
  const Box pb = L.box[it.p];
  const View v = make_view(pb.lo, pb.hi, g, L.dim);
  PT* xp = x[it.p];
  for (int t = threadIdx.x; t < kCellsPerChunk; t += kThreads) {
    int c[3];
    if (!decode_box(it, (long)ch.start + t, c)) break;
    const long o = (long)(c[0] - G.lo[0]) +
                   (long)G.n[0] * ((c[1] - G.lo[1]) + (long)G.n[1] * (L.dim == 3 ? c[2] - G.lo[2] : 0));
    if (to_box) box[o] = (T)ld(xp[v.at(c[0], c[1], c[2])]);
    else st(xp[v.at(c[0], c[1], c[2])], box[o]);
  }
}

// grid (npatch, slices): faces of axis a of patch blockIdx.x
template <typename T>
__global__ void __launch_bounds__(kThreads)
k_box_side(LevelGeom L, const double* const* x, int g, int a, T* box, BoxLevel G, int* mismatch,
           int verify) {
  const int p = blockIdx.x;
  const Box pb = L.box[p];
  int e[3] = {1, 1, 1};
  for (int d = 0; d < L.dim; ++d) e[d] = pb.hi[d] - pb.lo[d] + 1 + (d == a ? 1 : 0);
  int bn[3] = {G.n[0], G.n[1], L.dim == 3 ? G.n[2] : 1};
  bn[a] += 1;
  const View v = make_view(pb.lo, pb.hi, g, L.dim, a);
  const double* xp = x[p];
  const long nf = (long)e[0] * e[1] * e[2];
  for (long t = (long)blockIdx.y * kThreads + threadIdx.x; t < nf;
       t += (long)gridDim.y * kThreads) {
    const int i = pb.lo[0] + (int)(t % e[0]);
    const int j = pb.lo[1] + (int)((t / e[0]) % e[1]);
    const int k = L.dim == 3 ? pb.lo[2] + (int)(t / ((long)e[0] * e[1])) : 0;
    const long o = (long)(i - G.lo[0]) +
                   (long)bn[0] * ((j - G.lo[1]) + (long)bn[1] * (L.dim == 3 ? k - G.lo[2] : 0));
    const T val = (T)xp[v.at(i, j, k)];
    if (!verify) box[o] = val;
    else if (!same_bits(box[o], val))
      *mismatch = 1;
  }
}

template <int DIM, bool DVAR, int CMODE, int TX, int TY, int TZ, typename T>
void launch_tile(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc, int homogeneous,
                 const BoxCheck& K, hipStream_t s) {
  const int ntx = (G.n[0] + TX - 1) / TX, nty = (G.n[1] + TY - 1) / TY;
  const int ntz = DIM == 3 ? (G.n[2] + TZ - 1) / TZ : 1;
  const int ntiles = ntx * nty * ntz;
  const int per_xcd = (ntiles + 7) / 8;
  hipLaunchKernelGGL((k_box_rbgs<DIM, DVAR, CMODE, TX, TY, TZ, T>), dim3(8 * per_xcd),
                     dim3(kThreads), 0, s, G, A, bc, homogeneous, K, ntx, nty, ntiles, per_xcd);
  check_launch();
}

constexpr int kVariants = 13;
constexpr BoxTile kTiles3[kVariants] = {{32, 8, 8}, {16, 8, 8},  {32, 16, 4},
                                        {64, 4, 4}, {32, 8, 4},  {16, 16, 4},
                                        {16, 16, 8}, {32, 16, 8}, {24, 8, 8},
                                        {16, 4, 4}, {16, 8, 4}, {8, 8, 4}, {8, 4, 4}};
constexpr BoxTile kTiles2[kVariants] = {{64, 16, 1}, {32, 16, 1}, {32, 32, 1},
                                        {128, 8, 1}, {64, 8, 1},  {16, 16, 1},
                                        {64, 16, 1}, {64, 16, 1}, {64, 16, 1},
                                        {16, 8, 1}, {32, 8, 1}, {64, 4, 1}, {8, 8, 1}};

template <int DIM, bool DVAR, int CMODE, typename T>
void launch_variant(int variant, const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc,
                    int homogeneous, const BoxCheck& K, hipStream_t s) {
  if (DIM == 3) {
    switch (variant) {
      case 1: launch_tile<3, DVAR, CMODE, 16, 8, 8>(G, A, bc, homogeneous, K, s); break;
      case 2: launch_tile<3, DVAR, CMODE, 32, 16, 4>(G, A, bc, homogeneous, K, s); break;
      case 3: launch_tile<3, DVAR, CMODE, 64, 4, 4>(G, A, bc, homogeneous, K, s); break;
      case 4: launch_tile<3, DVAR, CMODE, 32, 8, 4>(G, A, bc, homogeneous, K, s); break;
      case 5: launch_tile<3, DVAR, CMODE, 16, 16, 4>(G, A, bc, homogeneous, K, s); break;
      case 6: launch_tile<3, DVAR, CMODE, 16, 16, 8>(G, A, bc, homogeneous, K, s); break;
      case 7: launch_tile<3, DVAR, CMODE, 32, 16, 8>(G, A, bc, homogeneous, K, s); break;
      case 8: launch_tile<3, DVAR, CMODE, 24, 8, 8>(G, A, bc, homogeneous, K, s); break;
      case 9: launch_tile<3, DVAR, CMODE, 16, 4, 4>(G, A, bc, homogeneous, K, s); break;
      case 10: launch_tile<3, DVAR, CMODE, 16, 8, 4>(G, A, bc, homogeneous, K, s); break;
      case 11: launch_tile<3, DVAR, CMODE, 8, 8, 4>(G, A, bc, homogeneous, K, s); break;
      case 12: launch_tile<3, DVAR, CMODE, 8, 4, 4>(G, A, bc, homogeneous, K, s); break;
      default: launch_tile<3, DVAR, CMODE, 32, 8, 8>(G, A, bc, homogeneous, K, s); break;
    }
  } else {
    switch (variant) {
      case 1: launch_tile<2, DVAR, CMODE, 32, 16, 1>(G, A, bc, homogeneous, K, s); break;
      case 2: launch_tile<2, DVAR, CMODE, 32, 32, 1>(G, A, bc, homogeneous, K, s); break;
      case 3: launch_tile<2, DVAR, CMODE, 128, 8, 1>(G, A, bc, homogeneous, K, s); break;
      case 4: launch_tile<2, DVAR, CMODE, 64, 8, 1>(G, A, bc, homogeneous, K, s); break;
      case 5: launch_tile<2, DVAR, CMODE, 16, 16, 1>(G, A, bc, homogeneous, K, s); break;
      case 9: launch_tile<2, DVAR, CMODE, 16, 8, 1>(G, A, bc, homogeneous, K, s); break;
      case 10: launch_tile<2, DVAR, CMODE, 32, 8, 1>(G, A, bc, homogeneous, K, s); break;
      case 11: launch_tile<2, DVAR, CMODE, 64, 4, 1>(G, A, bc, homogeneous, K, s); break;
      case 12: launch_tile<2, DVAR, CMODE, 8, 8, 1>(G, A, bc, homogeneous, K, s); break;
      default: launch_tile<2, DVAR, CMODE, 64, 16, 1>(G, A, bc, homogeneous, K, s); break;
    }
  }
}

template <int DIM, typename T>
void launch_dim(int variant, const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc,
                int homogeneous, const BoxCheck& K, hipStream_t s) {
  const bool dvar = A.D[0] != nullptr;
  if (dvar) {
    if (A.cmode == 2) launch_variant<DIM, true, 2>(variant, G, A, bc, homogeneous, K, s);
    else if (A.cmode == 1) launch_variant<DIM, true, 1>(variant, G, A, bc, homogeneous, K, s);
    else launch_variant<DIM, true, 0>(variant, G, A, bc, homogeneous, K, s);
  } else {
    if (A.cmode == 2) launch_variant<DIM, false, 2>(variant, G, A, bc, homogeneous, K, s);
    else if (A.cmode == 1) launch_variant<DIM, false, 1>(variant, G, A, bc, homogeneous, K, s);
    else launch_variant<DIM, false, 0>(variant, G, A, bc, homogeneous, K, s);
  }
}

// ------------------------------------------------------------------------
// Geometric multigrid on a single-rectangle level (the coarsest level's
// solver when coarse_solver_choice is "mg"/"hypre").  Level m+1 halves every
// extent of level m; cell-centred full-weighting restriction of the residual
// (mean of the 2^dim children), separable linear prolongation (weights 3/4
// and 1/4 per axis, homogeneous Robin ghosts beyond the domain), red-black
// Gauss-Seidel smoothing by k_box_rbgs, and a one-work-group LDS solve on
// the smallest grid.  All kernels return at once when *stop is set.

// u at box index (i, j, k) with homogeneous Robin ghosts one cell beyond the
// domain along any axis (applied axis by axis).
template <int DIM, typename T>
__device__ inline T mg_at(const BoxLevel& G, const RobinDev& bc, const T* u, int i, int j,
                          int k) {
  int c[3] = {i, j, k}, lo[3] = {0, 0, 0};
  for (int a = 0; a < DIM; ++a) {
    lo[a] = c[a] < 0 ? 0 : (c[a] >= G.n[a] ? G.n[a] - 1 : c[a]);
  }
  T v = u[(long)lo[0] + (long)G.n[0] * (lo[1] + (long)G.n[1] * (DIM == 3 ? lo[2] : 0))];
  for (int a = 0; a < DIM; ++a) {
    if (c[a] < 0) v = robin_ghost<DIM>(G, bc, 1, 2 * a, v);
    else if (c[a] >= G.n[a]) v = robin_ghost<DIM>(G, bc, 1, 2 * a + 1, v);
  }
  return v;
}

// Residual f - (div D grad u + C u) of one cell, in the smoother's
// expression order (global-memory neighbours, Robin ghosts at the domain).
template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline T mg_residual_q(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc,
                                  const T* u, int i, int j, int k, const Coef<T>& q) {
  const int n0 = G.n[0], n1 = G.n[1];
  const long c = (long)i + (long)n0 * (j + (long)n1 * k);
  const T dxi = (T)(1.0 / G.dx[0]), dyi = (T)(1.0 / G.dx[1]);
  const T dzi = DIM == 3 ? (T)(1.0 / G.dx[2]) : (T)0;
  const T dc = (T)A.dconst;
  const T uc = u[c];
  T Dxl, Dxh, Dyl, Dyh, Dzl = 0, Dzh = 0;
  if (DVAR) {
    Dxl = q.xl; Dxh = q.xh; Dyl = q.yl; Dyh = q.yh;
    if (DIM == 3) { Dzl = q.zl; Dzh = q.zh; }
  } else {
    Dxl = Dxh = Dyl = Dyh = Dzl = Dzh = dc;
  }
  const T uxl = i > 0 ? u[c - 1] : robin_ghost<DIM>(G, bc, 1, 0, uc);
  const T uxh = i < n0 - 1 ? u[c + 1] : robin_ghost<DIM>(G, bc, 1, 1, uc);
  const T uyl = j > 0 ? u[c - n0] : robin_ghost<DIM>(G, bc, 1, 2, uc);
  const T uyh = j < n1 - 1 ? u[c + n0] : robin_ghost<DIM>(G, bc, 1, 3, uc);
  const T fxl = dxi * Dxl * (uc - uxl);
  const T fxh = dxi * Dxh * (uxh - uc);
  const T fyl = dyi * Dyl * (uc - uyl);
  const T fyh = dyi * Dyh * (uyh - uc);
  T fzl = 0, fzh = 0;
  if (DIM == 3) {
    const long s2 = (long)n0 * n1;
    const T uzl = k > 0 ? u[c - s2] : robin_ghost<DIM>(G, bc, 1, 4, uc);
    const T uzh = k < G.n[2] - 1 ? u[c + s2] : robin_ghost<DIM>(G, bc, 1, 5, uc);
    fzl = dzi * Dzl * (uc - uzl);
    fzh = dzi * Dzh * (uzh - uc);
  }
  T scal;
  if (CMODE == 2) scal = q.c;
  else scal = CMODE == 1 ? (T)A.cconst : (T)0;
  if (DIM == 3)
    return q.f - (dxi * (fxh - fxl) + dyi * (fyh - fyl) + dzi * (fzh - fzl)) - scal * uc;
  return q.f - (dxi * (fxh - fxl) + dyi * (fyh - fyl)) - scal * uc;
}
template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline T mg_residual(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc,
                                const T* u, int i, int j, int k) {
  return mg_residual_q<DIM, DVAR, CMODE>(G, A, bc, u, i, j, k,
                                         load_coef<DIM, DVAR, CMODE>(G, A, i, j, k));
}

// Mean over the 2^dim children of coarse cell (I, J, K) of the fine
// residual (children summed in i, j, k order).  In 3-D four children's loads
// in flight and a third wave per SIMD are better than eight, but not with FP64
// face coefficients (kRestrictAll): us a call over 64^3 to 256^3 levels, four and
// eight, D per face FP64 79, 74, FP32 48, 54, constant D 41, 42.
template <int DIM, bool DVAR, typename T>
constexpr bool kRestrictAll = DIM == 2 || (DVAR && sizeof(T) == 8);
template <int DIM, bool DVAR, int CMODE, typename T>
__device__ inline T mg_restrict_value(const BoxLevel& Gf, const BoxArraysT<T>& A,
                                      const RobinDev& bc, const T* u, int I, int J, int K) {
  T sum = 0;
#pragma unroll (kRestrictAll<DIM, DVAR, T> ? 2 : 1)
  for (int c2 = 0; c2 < (DIM == 3 ? 2 : 1); ++c2)
    for (int c1 = 0; c1 < 2; ++c1)
      for (int c0 = 0; c0 < 2; ++c0)
        sum += mg_residual<DIM, DVAR, CMODE>(Gf, A, bc, u, 2 * I + c0, 2 * J + c1,
                                             DIM == 3 ? 2 * K + c2 : 0);
  return sum * (T)(DIM == 3 ? 0.125 : 0.25);
}

// Cell (i, j, k) of linear index t of a box n0 x n1 x ... (a level has at most
// 2^30 cells: setupBoxPath).  In 32 bits: a 64-bit division is a routine of over
// 100 instructions, as long as the rest of these kernels' work on a cell.
__device__ inline void mg_cell(unsigned t, int n0, int n1, int& i, int& j, int& k) {
  const unsigned row = t / (unsigned)n0;
  i = (int)(t - row * (unsigned)n0);
  k = (int)(row / (unsigned)n1);
  j = (int)(row - (unsigned)k * (unsigned)n1);
}

// fc = mean over the 2^dim children of the fine residual (one thread per
// coarse cell).
template <int DIM, bool DVAR, int CMODE, typename T>
__global__ void __launch_bounds__(kThreads)
k_mg_restrict_residual(BoxLevel Gf, BoxArraysT<T> A, RobinDev bc, const T* u, BoxLevel Gc, T* fc,
                       const int* stop) {
  if (*stop) return;
  const long nc = (long)Gc.n[0] * Gc.n[1] * (DIM == 3 ? Gc.n[2] : 1);
  for (long t = (long)blockIdx.x * kThreads + threadIdx.x; t < nc;
       t += (long)gridDim.x * kThreads) {
    int I, J, K;
    if (DIM == 3 && kRestrictAll<DIM, DVAR, T>) {
      // 64-bit divisions: with mg_cell all of the eight children's loads go
      // ahead of their uses, in so many registers that one wave per SIMD is
      // left (91 us a call)
      I = (int)(t % Gc.n[0]);
      J = (int)((t / Gc.n[0]) % Gc.n[1]);
      K = (int)(t / ((long)Gc.n[0] * Gc.n[1]));
    } else {
      mg_cell((unsigned)t, Gc.n[0], Gc.n[1], I, J, K);
    }
    fc[t] = mg_restrict_value<DIM, DVAR, CMODE>(Gf, A, bc, u, I, J, K);
  }
}

// ef += separable linear interpolation of ec: weights 3/4 (the parent) and 1/4
// (its neighbour towards the child) per axis, homogeneous Robin ghosts beyond
// the domain.  One thread per pair of fine cells under a parent in x: the two
// share the parents' column, 12 coarse values for both instead of 8 each, and
// their part of ef is one access; cells whose neighbours all lie inside read
// them without the ghosts' tests.  FP64, 128^3 and 64^3 together 38 us with one
// thread per fine cell, 27 us with this.
template <int DIM, typename T>
__global__ void __launch_bounds__(kThreads)
k_mg_prolong_add(BoxLevel Gc, RobinDev bc, const T* ec, BoxLevel Gf, T* ef, const int* stop) {
  if (*stop) return;
  const long np = (long)Gc.n[0] * Gf.n[1] * (DIM == 3 ? Gf.n[2] : 1);
  const T w3 = (T)0.75, w1 = (T)0.25;
  for (long t = (long)blockIdx.x * kThreads + threadIdx.x; t < np;
       t += (long)gridDim.x * kThreads) {
    int I, j, k;
    mg_cell((unsigned)t, Gc.n[0], Gf.n[1], I, j, k);
    const int J = j >> 1, K = k >> 1;
    const int Js = J + ((j & 1) ? 1 : -1), Ks = K + ((k & 1) ? 1 : -1);
    const T e0 = ef[2 * t], e1 = ef[2 * t + 1];
    // rows (J, K), (Js, K), (J, Ks), (Js, Ks) at I - 1, I, I + 1
    constexpr int NR = DIM == 3 ? 4 : 2;
    T v[NR][3];
    if (I > 0 && I + 1 < Gc.n[0] && Js >= 0 && Js < Gc.n[1] &&
        (DIM == 2 || (Ks >= 0 && Ks < Gc.n[2]))) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const T* x = ec + I + (long)Gc.n[0] * ((r & 1 ? Js : J) +
                                               (long)Gc.n[1] * (DIM == 3 ? (r & 2 ? Ks : K) : 0));
        v[r][0] = x[-1];
        v[r][1] = x[0];
        v[r][2] = x[1];
      }
    } else {
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int a = 0; a < 3; ++a)
          v[r][a] = mg_at<DIM>(Gc, bc, ec, I + a - 1, r & 1 ? Js : J,
                               DIM == 3 ? (r & 2 ? Ks : K) : 0);
    }
    T y[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      T row[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) row[r] = w3 * v[r][1] + w1 * v[r][2 * c];
      const T z0 = w3 * row[0] + w1 * row[1];
      y[c] = DIM == 3 ? w3 * z0 + w1 * (w3 * row[NR - 2] + w1 * row[NR - 1]) : z0;
    }
    ef[2 * t] = e0 + y[0];
    ef[2 * t + 1] = e1 + y[1];
  }
}

// Coefficients of level m+1 from level m: a coarse face takes the mean of
// the 2^(dim-1) fine faces it covers; C the mean of the 2^dim children.
template <int DIM, typename T>
__global__ void __launch_bounds__(kThreads)
k_mg_coarsen_coef(BoxLevel Gf, BoxArraysT<T> Af, BoxLevel Gc, T* Dc0, T* Dc1, T* Dc2, T* Cc) {
  const int nc[3] = {Gc.n[0], Gc.n[1], DIM == 3 ? Gc.n[2] : 1};
  const int nf[3] = {Gf.n[0], Gf.n[1], DIM == 3 ? Gf.n[2] : 1};
  T* Dc[3] = {Dc0, Dc1, Dc2};
  for (int a = 0; a < DIM; ++a) {
    if (!Dc[a]) continue;
    int e[3] = {nc[0], nc[1], nc[2]};
    e[a] += 1;
    int ef[3] = {nf[0], nf[1], nf[2]};
    ef[a] += 1;
    const long n = (long)e[0] * e[1] * e[2];
    const int t1 = a == 0 ? 1 : 0, t2 = a == 2 ? 1 : 2;
    for (long t = (long)blockIdx.x * kThreads + threadIdx.x; t < n;
         t += (long)gridDim.x * kThreads) {
      int c[3] = {(int)(t % e[0]), (int)((t / e[0]) % e[1]), (int)(t / ((long)e[0] * e[1]))};
      T sum = 0;
      for (int q2 = 0; q2 < (DIM == 3 ? 2 : 1); ++q2)
        for (int q1 = 0; q1 < 2; ++q1) {
          int f[3];
          f[a] = 2 * c[a];
          f[t1] = 2 * c[t1] + q1;
          f[t2] = DIM == 3 ? 2 * c[t2] + q2 : 0;
          sum += Af.D[a][(long)f[0] + (long)ef[0] * (f[1] + (long)ef[1] * f[2])];
        }
      Dc[a][t] = sum * (T)(DIM == 3 ? 0.25 : 0.5);
    }
  }
  if (Cc) {
    const long n = (long)nc[0] * nc[1] * nc[2];
    for (long t = (long)blockIdx.x * kThreads + threadIdx.x; t < n;
         t += (long)gridDim.x * kThreads) {
      const int I = (int)(t % nc[0]), J = (int)((t / nc[0]) % nc[1]);
      const int K = (int)(t / ((long)nc[0] * nc[1]));
      T sum = 0;
      for (int c2 = 0; c2 < (DIM == 3 ? 2 : 1); ++c2)
        for (int c1 = 0; c1 < 2; ++c1)
          for (int c0 = 0; c0 < 2; ++c0)
            sum += Af.C[(long)(2 * I + c0) +
                        (long)nf[0] * ((2 * J + c1) + (long)nf[1] * (DIM == 3 ? 2 * K + c2 : 0))];
      Cc[t] = sum * (T)(DIM == 3 ? 0.125 : 0.25);
    }
  }
}

constexpr int kMGSmallEdge = 4;

// Partial sums of the squared residual (x == nullptr) or of x^2 over a
// level, one per work-group of a fixed grid.
template <int DIM, bool DVAR, int CMODE, typename T>
__global__ void __launch_bounds__(kThreads)
k_mg_sumsq(BoxLevel G, BoxArraysT<T> A, RobinDev bc, const T* u, const T* x, double* partial,
           const int* stop) {
  __shared__ double sm[kThreads / 64];
  if (*stop) return;
  const long n = (long)G.n[0] * G.n[1] * (DIM == 3 ? G.n[2] : 1);
  double acc = 0.0;
  for (long t = (long)blockIdx.x * kThreads + threadIdx.x; t < n;
       t += (long)gridDim.x * kThreads) {
    double v;
    if (x) {
      v = (double)x[t];
    } else {
      int i, j, k;
      mg_cell((unsigned)t, G.n[0], G.n[1], i, j, k);
      v = (double)mg_residual<DIM, DVAR, CMODE>(G, A, bc, u, i, j, k);
    }
    acc += v * v;
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = 0.0;
    for (int w = 0; w < kThreads / 64; ++w) sum += sm[w];
    partial[blockIdx.x] = sum;
  }
}

// Convergence test after iteration `it` (it < 0: before the first): stop
// when ||r|| <= tol ||b|| (or b = 0), as hypre's relative-residual test.
// Relative-residual test after iteration it (it < 0: the b = 0 test only).
__device__ inline void mg_check(const double* rr, const double* bb, double tol, int it, int* stop,
                                int* iters, double* relres) {
  const double b = sqrt(*bb);
  if (it < 0) {
    if (!(b > 0.0)) {
      *stop = 1;
      *iters = 0;
      *relres = 0.0;
    }
    return;
  }
  const double rel = sqrt(*rr) / b;
  *iters = it + 1;
  *relres = rel;
  if (!(rel > tol)) *stop = 1;
}

// *out = sum of the n partials (in k_sum's order: a strided sum per thread,
// then the wavefront and work-group reductions), then the relative-residual
// test on it, in one launch; nothing once the solve has stopped.
constexpr int kMGSumThreads = 1024;
__global__ void __launch_bounds__(kMGSumThreads)
k_mg_sum_check(const double* partial, int n, double* out, const double* bb, double tol, int it,
               int* stop, int* iters, double* relres) {
  if (*stop) return;
  double acc = 0.0;
#pragma unroll 4
  for (int t = threadIdx.x; t < n; t += kMGSumThreads) acc += partial[t];
  __shared__ double sm[kMGSumThreads / 64];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = 0.0;
    for (int w = 0; w < kMGSumThreads / 64; ++w) v += sm[w];
    out[0] = v;
    mg_check(out, bb, tol, it, stop, iters, relres);
  }
}

}  // namespace

int box_tile_variants(int) { return kVariants; }

BoxTile box_tile(int dim, int variant) {
  if (variant < 0 || variant >= kVariants) variant = 0;
  return dim == 3 ? kTiles3[variant] : kTiles2[variant];
}

void launch_box_rbgs(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc, int homogeneous,
                     const BoxCheck& K, int variant, hipStream_t s) {
  if (A.fp32) {
    const BoxArraysT<float> At = typed<float>(A);
    if (G.dim == 3) launch_dim<3>(variant, G, At, bc, homogeneous, K, s);
    else launch_dim<2>(variant, G, At, bc, homogeneous, K, s);
  } else {
    const BoxArraysT<double> At = typed<double>(A);
    if (G.dim == 3) launch_dim<3>(variant, G, At, bc, homogeneous, K, s);
    else launch_dim<2>(variant, G, At, bc, homogeneous, K, s);
  }
}

void launch_box_final_check(const BoxCheck& K, int nsweeps, hipStream_t s) {
  hipLaunchKernelGGL(k_box_final_check, dim3(1), dim3(kThreads), 0, s, K, nsweeps);
  check_launch();
}

void launch_box_cells(const GhostLaunch& cells, const LevelGeom& L, double* const* x, int g,
                      double* box0, double* box1, const int* count, int count_host,
                      const BoxLevel& G, int to_box, hipStream_t s, int fp32, int patch_elem) {
  if (cells.nchunks == 0) return;
  if (patch_elem != 8) {
    // the mixed-precision error vector: FP32 / BF16 patch data, box in the
    // coarse solve's precision
    const dim3 g_(xcd_grid(cells.nchunks)), b_(kThreads);
    if (patch_elem == 4) {
      auto xp = reinterpret_cast<float* const*>(x);
      if (fp32)
        hipLaunchKernelGGL((k_box_cells<float, float>), g_, b_, 0, s, cells.items, cells.chunks,
                           L, xp, g, reinterpret_cast<float*>(box0),
                           reinterpret_cast<float*>(box1), count, count_host, G, to_box);
      else
        hipLaunchKernelGGL((k_box_cells<double, float>), g_, b_, 0, s, cells.items,
                           cells.chunks, L, xp, g, box0, box1, count, count_host, G, to_box);
    } else {
      auto xp = reinterpret_cast<bf16* const*>(x);
      if (fp32)
        hipLaunchKernelGGL((k_box_cells<float, bf16>), g_, b_, 0, s, cells.items, cells.chunks,
                           L, xp, g, reinterpret_cast<float*>(box0),
                           reinterpret_cast<float*>(box1), count, count_host, G, to_box);
      else
        hipLaunchKernelGGL((k_box_cells<double, bf16>), g_, b_, 0, s, cells.items, cells.chunks,
                           L, xp, g, box0, box1, count, count_host, G, to_box);
    }
    check_launch();
    return;
  }
  if (fp32)
    hipLaunchKernelGGL(k_box_cells<float>, dim3(xcd_grid(cells.nchunks)), dim3(kThreads), 0, s,
                       cells.items, cells.chunks, L, x, g, reinterpret_cast<float*>(box0),
                       reinterpret_cast<float*>(box1), count, count_host, G, to_box);
  else
    hipLaunchKernelGGL(k_box_cells<double>, dim3(xcd_grid(cells.nchunks)), dim3(kThreads), 0, s,
                       cells.items, cells.chunks, L, x, g, box0, box1, count, count_host, G,
                       to_box);
  check_launch();
}

void launch_box_side(const LevelGeom& L, const double* const* x, int g, int a, double* box,
                     const BoxLevel& G, int* mismatch, hipStream_t s, int verify, int fp32) {
  if (L.npatch == 0) return;
  dim3 grid(L.npatch, 64);
  for (int pass = 0; pass < (verify ? 2 : 1); ++pass) {
    if (fp32)
      hipLaunchKernelGGL(k_box_side<float>, grid, dim3(kThreads), 0, s, L, x, g, a,
                         reinterpret_cast<float*>(box), G, mismatch, pass);
    else
      hipLaunchKernelGGL(k_box_side<double>, grid, dim3(kThreads), 0, s, L, x, g, a, box, G,
                         mismatch, pass);
    check_launch();
  }
}


// ------------------------------------------------------------ multigrid

namespace {
constexpr int kMGGrid = 1024;  // work-groups of the grid-stride MG kernels

inline int mg_blocks(long n) {
  long b = (n + kThreads - 1) / kThreads;
  return (int)(b < kMGGrid ? (b > 0 ? b : 1) : kMGGrid);
}

template <int DIM, bool DVAR, int CMODE>
struct RestrictRun {
  template <typename T>
  static void run(const BoxLevel& Gf, const BoxArraysT<T>& A, const RobinDev& bc, const T* u,
                  const BoxLevel& Gc, T* fc, const int* stop, hipStream_t s) {
    const long nc = (long)Gc.n[0] * Gc.n[1] * (DIM == 3 ? Gc.n[2] : 1);
    hipLaunchKernelGGL((k_mg_restrict_residual<DIM, DVAR, CMODE, T>), dim3(mg_blocks(nc)),
                       dim3(kThreads), 0, s, Gf, A, bc, u, Gc, fc, stop);
    check_launch();
  }
};

template <int DIM, bool DVAR, int CMODE>
struct SumsqRun {
  template <typename T>
  static void run(const BoxLevel& G, const BoxArraysT<T>& A, const RobinDev& bc, const T* u,
                  const T* x, double* partial, const int* stop, hipStream_t s) {
    hipLaunchKernelGGL((k_mg_sumsq<DIM, DVAR, CMODE, T>), dim3(kMGGrid), dim3(kThreads), 0, s, G,
                       A, bc, u, x, partial, stop);
    check_launch();
  }
};

}  // namespace

int mg_small_edge() { return kMGSmallEdge; }
int mg_partials() { return kMGGrid; }

void launch_mg_restrict_residual(const BoxLevel& Gf, const BoxArrays& A, const RobinDev& bc,
                                 const double* u, const BoxLevel& Gc, double* fc,
                                 const int* stop, hipStream_t s) {
  if (A.fp32)
    dispatch3<RestrictRun>(Gf, typed<float>(A), bc, as<float>(u), Gc, as<float>(fc), stop, s);
  else
    dispatch3<RestrictRun>(Gf, typed<double>(A), bc, u, Gc, fc, stop, s);
}

template <typename T>
static void mg_prolong(const BoxLevel& Gc, const RobinDev& bc, const T* ec, const BoxLevel& Gf,
                       T* ef, const int* stop, hipStream_t s) {
  // fine extents are twice the coarse ones
  const long np = (long)Gc.n[0] * Gf.n[1] * (Gf.dim == 3 ? Gf.n[2] : 1);
  if (Gf.dim == 3)
    hipLaunchKernelGGL((k_mg_prolong_add<3, T>), dim3(mg_blocks(np)), dim3(kThreads), 0, s, Gc,
                       bc, ec, Gf, ef, stop);
  else
    hipLaunchKernelGGL((k_mg_prolong_add<2, T>), dim3(mg_blocks(np)), dim3(kThreads), 0, s, Gc,
                       bc, ec, Gf, ef, stop);
  check_launch();
}

void launch_mg_prolong_add(const BoxLevel& Gc, const RobinDev& bc, const double* ec,
                           const BoxLevel& Gf, double* ef, const int* stop, hipStream_t s,
                           int fp32) {
  if (fp32) mg_prolong<float>(Gc, bc, as<float>(ec), Gf, as<float>(ef), stop, s);
  else mg_prolong<double>(Gc, bc, ec, Gf, ef, stop, s);
}

template <typename T>
static void mg_coarsen(const BoxLevel& Gf, const BoxArraysT<T>& Af, const BoxLevel& Gc,
                       T* const* Dc, T* Cc, hipStream_t s) {
  const long nf = (long)Gf.n[0] * Gf.n[1] * (Gf.dim == 3 ? Gf.n[2] : 1);
  if (Gf.dim == 3)
    hipLaunchKernelGGL((k_mg_coarsen_coef<3, T>), dim3(mg_blocks(nf)), dim3(kThreads), 0, s, Gf,
                       Af, Gc, Dc[0], Dc[1], Dc[2], Cc);
  else
    hipLaunchKernelGGL((k_mg_coarsen_coef<2, T>), dim3(mg_blocks(nf)), dim3(kThreads), 0, s, Gf,
                       Af, Gc, Dc[0], Dc[1], (T*)nullptr, Cc);
  check_launch();
}

void launch_mg_coarsen_coef(const BoxLevel& Gf, const BoxArrays& Af, const BoxLevel& Gc,
                            double* const* Dc, double* Cc, hipStream_t s) {
  if (Af.fp32) {
    float* D32[3] = {as<float>(Dc[0]), as<float>(Dc[1]), as<float>(Dc[2])};
    mg_coarsen<float>(Gf, typed<float>(Af), Gc, D32, as<float>(Cc), s);
  } else {
    mg_coarsen<double>(Gf, typed<double>(Af), Gc, Dc, Cc, s);
  }
}

void launch_mg_sumsq(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc, const double* u,
                     const double* x, double* partial, const int* stop, hipStream_t s) {
  if (A.fp32)
    dispatch3<SumsqRun>(G, typed<float>(A), bc, as<float>(u), as<float>(x), partial, stop, s);
  else
    dispatch3<SumsqRun>(G, typed<double>(A), bc, u, x, partial, stop, s);
}

void launch_mg_sum_check(const double* partial, int n, double* out, const double* bb, double tol,
                         int it, int* stop, int* iters, double* relres, hipStream_t s) {
  hipLaunchKernelGGL(k_mg_sum_check, dim3(1), dim3(kMGSumThreads), 0, s, partial, n, out, bb, tol,
                     it, stop, iters, relres);
  check_launch();
}

}  // namespace sfac
