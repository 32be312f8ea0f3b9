// Learned block smoother: a 3-layer 3x3x3 convolution network over 16^3
// blocks of a level, trained on the GPU by the library's own forward and
// backward kernels.
//
// It has no counterpart in the reference (CellPoissonFACOps only offers the
// red-black Gauss-Seidel smoother, solv/CellPoissonFACOps.C:1338-1514); it
// maps the residual of a block (plus log D) to an error correction, and the
// red-black smoother stays the fallback, with the FP64 residual as the convergence test.
//
// Network: 2 input channels (r h^2 / s, log D) -> 16 -> 16 -> 1, ReLU after
// the hidden layers, "same" zero padding at the block faces.  Weights are
// kept in FP32 (Adam state too) and fed to the matrix cores in BF16; every
// convolution accumulates in FP32.  Channel counts are padded to 16 so that
// every layer is the same implicit GEMM: per output row of 16 cells and per
// pair of taps, one v_mfma_f32_16x16x32_bf16 with M = 16 cells, N = 16
// output channels, K = 2 taps x 16 input channels (the weight gradient has
// K = 32 cells).
//
// Activations are channels-last BF16: act[block][z][y][x][16] (32 B per
// cell).  Convolution weights are stored per tap: wf[t][co][ci] (forward)
// and wb[t][ci][co] with the tap flipped (backward data), t = 9(dz+1) +
// 3(dy+1) + (dx+1).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "samrai_learned.h"

namespace samrai_amd {
void set_last_error(const std::string& msg);
}

namespace {

constexpr int NB = 16;                 // block side
constexpr int NCELL = NB * NB * NB;    // cells per block
constexpr int CH = 16;                 // padded channel count
constexpr int NTAP = 27;
constexpr int WSZ = NTAP * CH * CH;    // conv weights per layer
constexpr int PSZ = WSZ + CH;          // + bias
constexpr int GSZ = (NTAP + 1) * CH * CH;  // gradient slab: 27 taps + bias row
constexpr int NLAYER = 3;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int NPAIR = (NTAP + 1) / 2;  // tap pairs per K = 32 MFMA
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t f2bf(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
  // the conversion instruction rounds to nearest even too
  return __builtin_bit_cast(uint16_t, (__bf16)f);
#else
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (inputs are finite)
  return (uint16_t)(u >> 16);
#endif
}
__host__ __device__ inline float bf2f(uint16_t h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

enum { MODE_HIDDEN = 0, MODE_FINAL = 1, MODE_BWD = 2 };

// One work-group per z-plane of a block (16 rows of 16 cells), four waves
// of four rows each.  The plane's input neighbourhood (planes z-1..z+1,
// rows -1..16, cells -1..16; zeros outside the block) is staged once in LDS
// with 16-byte loads, and each wave keeps its 27 weight taps in registers.
// Lane l: cell x = l & 15 of the A operand, channel group g = l >> 4.
// A[i][k]  (lane l: i = l & 15, k = 4g..4g+3)  = input at (x + dx, y + dy, z + dz), channel k
// B[k][n]  (lane l: n = l & 15, k = 4g..4g+3)  = w[t][n][k]
// D[i][n]  (lane l: i = 4g + j, n = l & 15)
// MODE_HIDDEN: out = relu(D + bias) as BF16 activations.
// MODE_FINAL : pred[cell] = D[cell][0] + bias[0] (FP32).
// MODE_BWD   : out = D * (mask[cell][n] > 0) as BF16 (gradient of the
//              previous layer's pre-activation; mask = its ReLU output).
constexpr int CONV_ROWS = 4;
constexpr int HB = NB + 2;  // halo-padded side

template <int MODE>
__global__ __launch_bounds__(256) void k_conv(const uint16_t* __restrict__ x,
                                              const uint16_t* __restrict__ w,
                                              const float* __restrict__ bias,
                                              const uint16_t* __restrict__ mask,
                                              uint16_t* __restrict__ out,
                                              float* __restrict__ pred, int nplanes) {
  __shared__ uint4 tile[3 * HB * HB * 2];  // 31104 B: [pz][py][px][2 halves of 8 channels]
  const int plane = blockIdx.x;
  if (plane >= nplanes) return;  // whole work-group
  const int b = plane / NB;
  const int z = plane % NB;
  const uint16_t* xb = x + (size_t)b * NCELL * CH;
  for (int s = threadIdx.x; s < 3 * HB * HB * 2; s += 256) {
    const int half = s & 1;
    const int c = s >> 1;
    const int px = c % HB, py = (c / HB) % HB, pz = c / (HB * HB);
    const int xx = px - 1, yy = py - 1, zz = z + pz - 1;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if ((unsigned)xx < (unsigned)NB && (unsigned)yy < (unsigned)NB && (unsigned)zz < (unsigned)NB)
      v = *reinterpret_cast<const uint4*>(xb + ((size_t)((zz * NB + yy) * NB + xx)) * CH +
                                          8 * half);
    tile[s] = v;
  }
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int cx = lane & 15;
  const int g = lane >> 4;
  // K = 32 per MFMA: two taps of 16 channels.  Lane group g holds channels
  // 8 (g & 1) .. +7 of tap 2q + (g >> 1); the 28th tap is zero weights.
  const int half = g & 1;
  const int tsel = g >> 1;
  bf16x8 wr[NPAIR];
#pragma unroll
  for (int q = 0; q < NPAIR; ++q) {
    const int t = 2 * q + tsel;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (t < NTAP) v = *reinterpret_cast<const uint4*>(w + (t * CH + cx) * CH + 8 * half);
    wr[q] = __builtin_bit_cast(bf16x8, v);
  }
  const float bv = MODE == MODE_HIDDEN ? bias[cx] : (MODE == MODE_FINAL ? bias[0] : 0.f);
  __syncthreads();
  const uint16_t* lds = reinterpret_cast<const uint16_t*>(tile);
  for (int r = 0; r < CONV_ROWS; ++r) {
    const int y = wave * CONV_ROWS + r;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NPAIR; ++q) {
      const int t = min(2 * q + tsel, NTAP - 1);  // the zero-weight 28th tap reads tap 27's cells
      const int dz = t / 9 - 1, dy = (t / 3) % 3 - 1, dx = t % 3 - 1;
      const uint4 v = *reinterpret_cast<const uint4*>(
          lds + (((dz + 1) * HB + (y + dy + 1)) * HB + (cx + dx + 1)) * CH + 8 * half);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v), wr[q], acc, 0,
                                                    0, 0);
    }
    const size_t cell0 = (size_t)(plane * NB + y) * NB;  // first cell of the row
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t cell = cell0 + 4 * g + j;
      float v = acc[j];
      if (MODE == MODE_HIDDEN) {
        v += bv;
        v = v > 0.f ? v : 0.f;
        out[cell * CH + cx] = f2bf(v);
      } else if (MODE == MODE_FINAL) {
        if (cx == 0) pred[cell] = v + bv;
      } else {
        const bool on = bf2f(mask[cell * CH + cx]) > 0.f;
        out[cell * CH + cx] = f2bf(on ? v : 0.f);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The three layers in one kernel.
//
// Layer by layer the network moves every hidden activation (32 B a cell)
// through HBM twice and does 14 K = 32 products of 16 cells per layer although
// the first layer has 2 input channels and the last 1 output channel.  Here a
// work-group takes a z-slab of a block (the whole block when there are enough
// of them) and marches through its planes, four of each hidden layer in LDS:
// step i forms plane i + 2 of the first layer, plane i of the second, the tap
// products of plane i - 2 of the third and the prediction of plane i - 3, all
// from planes of earlier steps, so that one barrier a step is enough (it
// waits for LDS only, the stores drain behind it).  The hidden activations are
// written once, for a backward pass, and not read back here.  What bounds it
// are the LDS reads and, of a block, the latency of its 64 KB of input, which is
// loaded while the block before it is worked on:
//   layer 1: K holds 16 taps x 2 channels, so 2 products a row;
//   layer 2: a fragment (row y', taps dx = -1 and 0 of one dz, or dx = 1 of two)
//     serves the three output rows y' - 1 .. y' + 1, 5 fragments a row and 15
//     products (20 fragment reads for the two rows a wave forms, not 28);
//   layer 3: N holds the 9 (dy, dx) taps, K two dz, 2 products a row; the
//     prediction is then 9 adds per cell.
// A correction of 4096 blocks (features, three layers, correction) 1.66 ms as
// five kernels, 0.63 ms so: 0.43 PFLOP/s of real channels, 3.3 TB/s (0.58 ms
// without the hidden activations' stores).
constexpr int FWD_THREADS = 512;
constexpr int FP = HB * HB;          // cells of a halo-padded plane
constexpr int FWD_F = HB * FP;       // words: features, two BF16 a cell, all planes
constexpr int FWD_H = FP * 2;        // uint4 per plane of 16 channels
constexpr int FWD_G = FP * 9;        // floats per plane of tap products
constexpr int FWD_LDS = FWD_F * 4 + 8 * FWD_H * 16 + 2 * FWD_G * 4;  // 129600 B

struct Forward {
  const uint16_t* x0;    // features (FROM_R false)
  const double* r;       // residual and log D (nullptr: logd_const), FROM_R
  const double* logd;
  double logd_const, h2;
  uint16_t* x0_out;      // features, scales (FROM_R)
  double* scale;
  const uint16_t* w[NLAYER];
  const float* bias[NLAYER];
  uint16_t* act[2];      // hidden activations
  float* pred;
  double* e;             // omega * scale * prediction (FROM_R)
  double omega;
  int nblocks;
};

// Barrier that orders LDS accesses only.
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// FROM_R: one work-group per block at a time forms its scale and features from
// the residual and writes the correction; else a work-group takes 16 / slabs
// planes of a block.
// Work-group b takes slabs b, b + gridDim.x, ... of all.
template <bool FROM_R>
__global__ __launch_bounds__(FWD_THREADS) void k_forward(Forward P, int slabs) {
  __shared__ __align__(16) unsigned char lds[FWD_LDS];
  uint32_t* F = reinterpret_cast<uint32_t*>(lds);
  uint4* H1 = reinterpret_cast<uint4*>(lds + FWD_F * 4);
  uint4* H2 = H1 + 4 * FWD_H;
  float* G = reinterpret_cast<float*>(H2 + 4 * FWD_H);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int cx = lane & 15, g = lane >> 4, half = g & 1, tsel = g >> 1;
  const int nwork = P.nblocks * slabs;
  if ((int)blockIdx.x >= nwork) return;
  constexpr int NV = FROM_R ? NCELL / FWD_THREADS : 1;
  double rv[NV], lv[NV];
  auto fetch = [&](int b) {  // a block's residual and log D
    if (FROM_R)
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const size_t c = (size_t)b * NCELL + threadIdx.x + k * FWD_THREADS;
        rv[k] = P.r[c];
        lv[k] = P.logd ? P.logd[c] : P.logd_const;
      }
  };
  fetch(blockIdx.x);
  for (int q = threadIdx.x; q < FWD_LDS / 16; q += FWD_THREADS)
    reinterpret_cast<uint4*>(lds)[q] = make_uint4(0u, 0u, 0u, 0u);

  // weights: layer 1 [m], layer 2 [5 kinds][dy], layer 3 [dz pair]
  bf16x8 w1[2], w2[5][3], w3[2];
  // layer 1's inputs: taps 16 m + 4 g .. + 3 (two channels each) of the
  // lane's cell, as offsets in F; the taps past the 27th have zero weights
  int off1[2][4];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    uint32_t u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int t = 16 * m + 4 * g + k, tt = min(t, NTAP - 1);
      u[k] = t < NTAP ? *reinterpret_cast<const uint32_t*>(P.w[0] + (t * CH + cx) * CH) : 0u;
      off1[m][k] = ((tt / 9) * HB + (tt / 3) % 3 + 2 * wave) * HB + cx + tt % 3;
    }
    w1[m] = __builtin_bit_cast(bf16x8, make_uint4(u[0], u[1], u[2], u[3]));
  }
#pragma unroll
  for (int f = 0; f < 5; ++f)
#pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
      // f < 3: dz = f, dx = tsel; f = 3: dz = tsel, dx = 2; f = 4: dz = 2, dx = 2
      const int dz = f < 3 ? f : (f == 3 ? tsel : 2), dx = f < 3 ? tsel : 2;
      const int t = dz * 9 + dy * 3 + dx;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (f < 4 || tsel == 0)
        v = *reinterpret_cast<const uint4*>(P.w[1] + (t * CH + cx) * CH + 8 * half);
      w2[f][dy] = __builtin_bit_cast(bf16x8, v);
    }
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int dz = m == 0 ? tsel : 2;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (cx < 9 && (m == 0 || tsel == 0))
      v = *reinterpret_cast<const uint4*>(P.w[2] + ((dz * 9 + cx) * CH) * CH + 8 * half);
    w3[m] = __builtin_bit_cast(bf16x8, v);
  }
  const float b1 = P.bias[0][cx], b2 = P.bias[1][cx], b3 = P.bias[2][0];
  const int nz = NB / slabs;
  const int y0 = 2 * wave;  // this wave's rows
  uint16_t* h1 = reinterpret_cast<uint16_t*>(H1);
  uint16_t* h2 = reinterpret_cast<uint16_t*>(H2);
  lds_barrier();

  for (int work = blockIdx.x; work < nwork; work += gridDim.x) {
    const int b = work / slabs, z0 = (work % slabs) * nz, zend = z0 + nz;
    // features of the block into F (interior; the halo stays 0)
    double scale = 0.0;
    if (FROM_R) {
      double* red = reinterpret_cast<double*>(G);  // free here
      double s2 = 0.0;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        rv[k] *= P.h2;
        s2 += rv[k] * rv[k];
      }
      for (int o = 32; o > 0; o >>= 1) s2 += __shfl_xor(s2, o, 64);
      if (lane == 0) red[wave] = s2;
      lds_barrier();
      s2 = 0.0;
#pragma unroll
      for (int k = 0; k < FWD_THREADS / 64; ++k) s2 += red[k];
      lds_barrier();
      if (threadIdx.x < FWD_THREADS / 64) red[threadIdx.x] = 0.0;  // G's halo is read as zeros
      // a block whose residual is zero (or not finite) gets scale 0 (k_features)
      const double sq = sqrt(s2 / NCELL);
      const bool live = sq > 0.0;
      scale = live ? sq : 0.0;
      if (threadIdx.x == 0) P.scale[b] = scale;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const int c = threadIdx.x + k * FWD_THREADS;
        const uint32_t lo = live ? f2bf((float)(rv[k] / sq)) : (uint16_t)0;
        const uint32_t hi = f2bf((float)lv[k]);
        F[((c >> 8) + 1) * FP + (((c >> 4) & 15) + 1) * HB + (c & 15) + 1] = lo | (hi << 16);
        uint4* dst = reinterpret_cast<uint4*>(P.x0_out + ((size_t)b * NCELL + c) * CH);
        dst[0] = make_uint4(lo | (hi << 16), 0u, 0u, 0u);
        dst[1] = make_uint4(0u, 0u, 0u, 0u);
      }
      if (work + (int)gridDim.x < nwork) fetch(work + gridDim.x);
    } else {
      const int p0 = max(z0 - 3, 0), p1 = min(z0 + nz + 3, NB);
      for (int c = p0 * 256 + threadIdx.x; c < p1 * 256; c += FWD_THREADS)
        F[((c >> 8) + 1) * FP + (((c >> 4) & 15) + 1) * HB + (c & 15) + 1] =
            *reinterpret_cast<const uint32_t*>(P.x0 + ((size_t)b * NCELL + c) * CH);
    }
    lds_barrier();

    for (int i = z0 - 4; i < zend + 3; ++i) {
      // layer 1, plane i + 2
      if (i + 2 >= z0 - 2 && i + 2 < zend + 2) {
        const int z = i + 2;
        uint16_t* dst = h1 + (z & 3) * FWD_H * 8;
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        const bool in = (unsigned)z < (unsigned)NB;  // planes beyond the block are 0
        if (in) {
          const uint32_t* src = F + z * FP;
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const uint4 v = make_uint4(src[off1[m][0] + q * HB], src[off1[m][1] + q * HB],
                                         src[off1[m][2] + q * HB], src[off1[m][3] + q * HB]);
              acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v),
                                                               w1[m], acc[q], 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float v = acc[q][j] + b1;
            dst[((y0 + q + 1) * HB + 4 * g + j + 1) * CH + cx] = f2bf(in && v > 0.f ? v : 0.f);
          }
      }
      // layer 3, tap products of plane i - 2
      if (i - 2 >= z0 && i - 2 < zend) {
        float* dst = G + (i & 1) * FWD_G;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const int dz = m == 0 ? tsel : 2;
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, H2[((i - 3 + dz) & 3) * FWD_H +
                                              ((y0 + q + 1) * HB + cx + 1) * 2 + half]),
                w3[m], acc, 0, 0, 0);
          }
          if (cx < 9)
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[((y0 + q + 1) * HB + 4 * g + j + 1) * 9 + cx] = acc[j];
        }
      }
      // layer 2, plane i
      if (i >= z0 - 1 && i < zend + 1) {
        uint16_t* dst = h2 + (i & 3) * FWD_H * 8;
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        const bool in = (unsigned)i < (unsigned)NB;
        if (in) {
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {  // input row y0 - 1 + rr, at padded y0 + rr
            bf16x8 a[5];
#pragma unroll
            for (int f = 0; f < 5; ++f) {
              const int dz = f < 3 ? f : (f == 3 ? tsel : 2), dx = f < 3 ? tsel : 2;
              a[f] = __builtin_bit_cast(
                  bf16x8, H1[((i + dz - 1) & 3) * FWD_H + ((y0 + rr) * HB + cx + dx) * 2 + half]);
            }
#pragma unroll
            for (int f = 0; f < 5; ++f)
#pragma unroll
              for (int q = 0; q < 2; ++q) {
                const int dy = rr - q;  // offset + 1 of output row y0 + q
                if (dy >= 0 && dy < 3)
                  acc[q] =
                      __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[f], w2[f][dy], acc[q], 0, 0, 0);
              }
          }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float v = acc[q][j] + b2;
            dst[((y0 + q + 1) * HB + 4 * g + j + 1) * CH + cx] = f2bf(in && v > 0.f ? v : 0.f);
          }
      }
      // prediction of plane i - 3
      if (i - 3 >= z0 && threadIdx.x < 256) {
        const float* src = G + ((i - 1) & 1) * FWD_G;
        const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
        float p = b3;
#pragma unroll
        for (int t = 0; t < 9; ++t) p += src[((y + t / 3) * HB + x + t % 3) * 9 + t];
        const size_t c = (size_t)b * NCELL + (i - 3) * 256 + threadIdx.x;
        P.pred[c] = p;
        if (FROM_R) P.e[c] = P.omega * scale * (double)p;
      }
      // hidden planes to memory: the first layer's plane i + 1, the second's i - 1
      const int c = threadIdx.x >> 1, hf = threadIdx.x & 1;
      const int at = (((c >> 4) + 1) * HB + (c & 15) + 1) * 2 + hf;
      const int za = i + 1, zb = i - 1;
      if (za >= z0 && za < zend)
        reinterpret_cast<uint4*>(P.act[0])[((size_t)b * NCELL + za * 256 + c) * 2 + hf] =
            H1[(za & 3) * FWD_H + at];
      if (zb >= z0 && zb < zend)
        reinterpret_cast<uint4*>(P.act[1])[((size_t)b * NCELL + zb * 256 + c) * 2 + hf] =
            H2[(zb & 3) * FWD_H + at];
      lds_barrier();
    }
  }
}

// Weight gradient: dW[t][co][ci] = sum_cells G[cell][co] X[cell + off(t)][ci],
// db[co] = sum_cells G[cell][co]: 28 products per 32 cells (27 taps and a ones
// column), K = 32 cells = two rows of 16.  Both operands need a channel's cells
// consecutive while memory holds a cell's channels so, and read from memory
// they are 2-byte loads, which bound the first version (69 us for 64 blocks).
// Here a work-group stages the planes of its z-slab once, transposed in LDS
// ([channel][row][cell], rows of 24 elements whose first 8 are zeros: 16-byte
// reads of eight cells, the neighbouring row's zeros at both ends), a ring of
// four planes of X and two of G so that the next planes load and store while
// the current ones are multiplied; a (dz, dy) row is read once and its dx = -1
// and 1 neighbours are formed by 32-bit funnel shifts.  The channel strides
// (220 and 132 words) spread 16 channels over all LDS banks.  A training
// step of 64 blocks (three of these, the rest of the network and Adam) 0.37 ms
// with the first version, 0.12 ms with this one and the fused forward pass.
// A[m][k] (lane l: m = co = l & 15, k = cells 8g..8g+7) = G[cell_k][co]
// B[k][n] (lane l: n = ci = l & 15, k = cells 8g..8g+7) = X[cell_k + off(t)][ci]
// D[m][n] (lane l: m = 4g + j, n = l & 15) -> partial[t][m][n]
constexpr int WG_ROW = 24;                  // elements of a staged row of X
constexpr int WG_XC = 440;                  // per channel: 18 rows and padding
constexpr int WG_XP = CH * WG_XC;           // per plane
constexpr int WG_GC = 264;                  // per channel of G: 256 cells and padding
constexpr int WG_GP = CH * WG_GC;
constexpr int WG_LDS = 4 * WG_XP + 2 * WG_GP;  // 73,216 B: two work-groups a CU

__global__ __launch_bounds__(256) void k_wgrad(const uint16_t* __restrict__ x,
                                               const uint16_t* __restrict__ gz,
                                               float* __restrict__ partial, int nblocks,
                                               int slabs) {
  __shared__ __align__(16) uint16_t lds[WG_LDS];
  uint16_t* X = lds;
  uint16_t* Gs = lds + 4 * WG_XP;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int cx = lane & 15, g = lane >> 4;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;  // staged cell
  const int nz = NB / slabs, nwork = nblocks * slabs;
  for (int q = threadIdx.x; q < WG_LDS / 8; q += 256)
    reinterpret_cast<uint4*>(lds)[q] = make_uint4(0u, 0u, 0u, 0u);
  f32x4 acc[NTAP + 1];
#pragma unroll
  for (int t = 0; t <= NTAP; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
  {
    const uint32_t v = cx == 0 ? 0x3f803f80u : 0u;
    ones = __builtin_bit_cast(bf16x8, make_uint4(v, v, v, v));
  }
  struct Cell {
    uint4 lo, hi;
  };
  // the caller's arrays are aligned to their elements only; global memory takes
  // a 16-byte load at any address, so this is one instruction either way
  struct __attribute__((packed, aligned(2))) Channels {
    uint32_t w[8];
  };
  auto load = [&](const uint16_t* p, int b, int z) {  // plane z's cell of this thread
    Cell c{make_uint4(0u, 0u, 0u, 0u), make_uint4(0u, 0u, 0u, 0u)};
    if ((unsigned)z < (unsigned)NB) {
      const Channels q = *reinterpret_cast<const Channels*>(
          p + ((size_t)b * NCELL + z * 256 + threadIdx.x) * CH);
      c.lo = make_uint4(q.w[0], q.w[1], q.w[2], q.w[3]);
      c.hi = make_uint4(q.w[4], q.w[5], q.w[6], q.w[7]);
    }
    return c;
  };
  auto store = [&](uint16_t* dst, int stride, const Cell& c) {  // a channel per `stride`
    const uint32_t w[8] = {c.lo.x, c.lo.y, c.lo.z, c.lo.w, c.hi.x, c.hi.y, c.hi.z, c.hi.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      dst[(2 * k) * stride] = (uint16_t)(w[k] & 0xffffu);
      dst[(2 * k + 1) * stride] = (uint16_t)(w[k] >> 16);
    }
  };
  auto xcell = [&](int z) { return X + ((z + 4) & 3) * WG_XP + (ty + 1) * WG_ROW + 8 + tx; };
  auto gcell = [&](int z) { return Gs + (z & 1) * WG_GP + threadIdx.x; };
  lds_barrier();
  for (int work = blockIdx.x; work < nwork; work += gridDim.x) {
    const int b = work / slabs, z0 = (work % slabs) * nz;
    {
      const Cell a0 = load(x, b, z0 - 1), a1 = load(x, b, z0), a2 = load(x, b, z0 + 1);
      const Cell g0 = load(gz, b, z0);
      store(xcell(z0 - 1), WG_XC, a0);
      store(xcell(z0), WG_XC, a1);
      store(xcell(z0 + 1), WG_XC, a2);
      store(gcell(z0), WG_GC, g0);
    }
    lds_barrier();
    for (int z = z0; z < z0 + nz; ++z) {
      const bool more = z + 1 < z0 + nz;
      Cell xn{}, gn{};
      if (more) {
        xn = load(x, b, z + 2);
        gn = load(gz, b, z + 1);
      }
#pragma unroll
      for (int rp = 0; rp < 2; ++rp) {
        const int y = 2 * (wave + 4 * rp) + (g >> 1), xo = 8 * (g & 1);
        const bf16x8 a = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const uint4*>(Gs + (z & 1) * WG_GP + cx * WG_GC + 16 * y + xo));
#pragma unroll
        for (int q = 0; q < 9; ++q) {
          const int dz = q / 3 - 1, dy = q % 3 - 1;
          const uint16_t* row =
              X + ((z + dz + 4) & 3) * WG_XP + cx * WG_XC + (y + dy + 1) * WG_ROW + 8 + xo;
          const uint4 v = *reinterpret_cast<const uint4*>(row);
          const uint32_t lo = row[-1], hi = row[8];
          // eight cells from x - 1 and from x + 1
          const uint32_t s0 = __builtin_amdgcn_alignbit(v.x, lo << 16, 16);
          const uint32_t s1 = __builtin_amdgcn_alignbit(v.y, v.x, 16);
          const uint32_t s2 = __builtin_amdgcn_alignbit(v.z, v.y, 16);
          const uint32_t s3 = __builtin_amdgcn_alignbit(v.w, v.z, 16);
          const uint32_t s4 = __builtin_amdgcn_alignbit(hi, v.w, 16);
          acc[3 * q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, __builtin_bit_cast(bf16x8, make_uint4(s0, s1, s2, s3)), acc[3 * q], 0, 0, 0);
          acc[3 * q + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, __builtin_bit_cast(bf16x8, v), acc[3 * q + 1], 0, 0, 0);
          acc[3 * q + 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, __builtin_bit_cast(bf16x8, make_uint4(s1, s2, s3, s4)), acc[3 * q + 2], 0, 0, 0);
        }
        acc[NTAP] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, acc[NTAP], 0, 0, 0);
      }
      if (more) {  // planes z + 2 and z + 1: slots the current step does not read
        store(xcell(z + 2), WG_XC, xn);
        store(gcell(z + 1), WG_GC, gn);
      }
      lds_barrier();
    }
  }
  // the four wavefronts' sums, in a fixed order, into one slab
  float* red = reinterpret_cast<float*>(lds);  // two slabs of GSZ floats
  auto put = [&](float* p) {
#pragma unroll
    for (int t = 0; t <= NTAP; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) p[(t * CH + 4 * g + j) * CH + cx] = acc[t][j];
  };
  auto add = [&](const float* p) {
#pragma unroll
    for (int t = 0; t <= NTAP; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[t][j] += p[(t * CH + 4 * g + j) * CH + cx];
  };
  static_assert(2 * GSZ * 4 <= WG_LDS * 2, "two slabs fit the staging buffer");
  if (wave >= 2) put(red + (wave - 2) * GSZ);
  __syncthreads();
  if (wave < 2) add(red + wave * GSZ);
  __syncthreads();
  if (wave == 1) put(red);
  __syncthreads();
  if (wave == 0) {
    add(red);
    put(partial + (size_t)blockIdx.x * GSZ);
  }
}

// Sum of the work-groups' slabs: 16 threads per output each summing every
// 16th slab in order, then the 16 partial sums in a fixed order
// (deterministic).  blockIdx.y: a layer, `layer_stride` slabs apart.
struct GradOut {
  float* grad[NLAYER];
};
__global__ __launch_bounds__(256) void k_wgrad_reduce(const float* __restrict__ partial,
                                                      int nslabs, size_t layer_stride,
                                                      GradOut out) {
  __shared__ float red[16][17];
  const int o = threadIdx.x & 15;
  const int part = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + o;
  const float* p = partial + blockIdx.y * layer_stride;
  float s = 0.f;
  if (i < GSZ)
    for (int w = part; w < nslabs; w += 16) s += p[(size_t)w * GSZ + i];
  red[part][o] = s;
  __syncthreads();
  if (part == 0 && i < GSZ) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[k][o];
    out.grad[blockIdx.y][i] = t;
  }
}

// Features of one block per work-group (1024 threads, four cells each, read
// once: a training batch has fewer blocks than there are compute units, and its
// time is this chain's): s = RMS over the block of r h^2;
// X[cell] = (r h^2 / s, log D, 0...).
constexpr int kFeatThreads = 1024;
__global__ __launch_bounds__(kFeatThreads) void k_features(const double* __restrict__ r,
                                                           const double* __restrict__ logd,
                                                           double logd_const, double h2,
                                                           uint16_t* __restrict__ x,
                                                           double* __restrict__ scale) {
  constexpr int NV = NCELL / kFeatThreads;
  __shared__ double red[kFeatThreads / 64];
  const int b = blockIdx.x;
  const size_t c0 = (size_t)b * NCELL + threadIdx.x;
  double v[NV], l[NV], s2 = 0.0;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    v[k] = r[c0 + k * kFeatThreads] * h2;
    l[k] = logd ? logd[c0 + k * kFeatThreads] : logd_const;
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) s2 += v[k] * v[k];
  for (int o = 32; o > 0; o >>= 1) s2 += __shfl_xor(s2, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s2;
  __syncthreads();
  s2 = 0.0;
#pragma unroll
  for (int k = 0; k < kFeatThreads / 64; ++k) s2 += red[k];
  // a block whose residual is zero (or not finite) gets scale 0: zero
  // features, a zero correction and no loss term
  const double s = sqrt(s2 / NCELL);
  const bool live = s > 0.0;
  if (threadIdx.x == 0) scale[b] = live ? s : 0.0;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const uint32_t lo = live ? f2bf((float)(v[k] / s)) : (uint16_t)0;
    const uint32_t hi = f2bf((float)l[k]);
    uint4* dst = reinterpret_cast<uint4*>(x + (c0 + k * kFeatThreads) * CH);
    dst[0] = make_uint4(lo | (hi << 16), 0u, 0u, 0u);
    dst[1] = make_uint4(0u, 0u, 0u, 0u);
  }
}

// Loss 1/N sum (pred - e/s)^2 and its gradient, written as channel 0 of a
// 16-channel BF16 tensor (the final layer's output gradient).
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ pred,
                                              const double* __restrict__ target,
                                              const double* __restrict__ scale, int ncells,
                                              float inv_n, uint16_t* __restrict__ gout,
                                              float* __restrict__ loss_partial) {
  __shared__ float red[256];
  const int c = blockIdx.x * 256 + threadIdx.x;
  float d2 = 0.f;
  if (c < ncells) {
    const double sc = scale[c / NCELL];
    const float d = sc > 0.0 ? pred[c] - (float)(target[c] / sc) : 0.f;
    d2 = d * d;
    uint4* dst = reinterpret_cast<uint4*>(gout + (size_t)c * CH);
    dst[0] = make_uint4((uint32_t)f2bf(2.f * d * inv_n), 0u, 0u, 0u);
    dst[1] = make_uint4(0u, 0u, 0u, 0u);
  }
  red[threadIdx.x] = d2;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss_partial[blockIdx.x] = red[0];
}

__global__ void k_sum_f32(const float* __restrict__ a, int n, float scale_by,
                          float* __restrict__ out) {
  __shared__ float red[256];
  float s = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) s += a[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0] * scale_by;
}

// Adam on the FP32 master parameters of layer blockIdx.y (27*16*16 weights
// then 16 biases), then the BF16 copies in forward and (flipped, transposed)
// backward layouts.  Weights outside the layer's real channel counts stay 0.
struct AdamLayer {
  float *p, *m, *v;
  const float* grad;
  uint16_t *wf, *wb;
  float* bias;
  int cin, cout;
};
struct AdamLayers {
  AdamLayer l[NLAYER];
};
__global__ void k_adam(AdamLayers all, float lr, float beta1, float beta2, float eps, float bc1,
                       float bc2) {
  const AdamLayer L = all.l[blockIdx.y];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= PSZ) return;
  float gi;
  bool live;
  int t = 0, co, ci = 0;
  if (i < WSZ) {
    t = i / (CH * CH);
    co = (i / CH) % CH;
    ci = i % CH;
    live = ci < L.cin && co < L.cout;
    gi = L.grad[i];
  } else {
    co = i - WSZ;
    live = co < L.cout;
    gi = L.grad[(NTAP * CH + co) * CH + 0];
  }
  float pi = L.p[i];
  if (live) {
    const float mi = beta1 * L.m[i] + (1.f - beta1) * gi;
    const float vi = beta2 * L.v[i] + (1.f - beta2) * gi * gi;
    L.m[i] = mi;
    L.v[i] = vi;
    pi -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  } else {
    pi = 0.f;
  }
  L.p[i] = pi;
  if (i < WSZ) {
    const uint16_t h = f2bf(pi);
    L.wf[(t * CH + co) * CH + ci] = h;
    L.wb[((NTAP - 1 - t) * CH + ci) * CH + co] = h;
  } else {
    L.bias[co] = pi;
  }
}

// Copy of the master parameters into the BF16 layouts (after set/init).
__global__ void k_sync_weights(const float* __restrict__ p, uint16_t* __restrict__ wf,
                               uint16_t* __restrict__ wb, float* __restrict__ bias) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= PSZ) return;
  if (i < WSZ) {
    const int t = i / (CH * CH), co = (i / CH) % CH, ci = i % CH;
    const uint16_t h = f2bf(p[i]);
    wf[(t * CH + co) * CH + ci] = h;
    wb[((NTAP - 1 - t) * CH + ci) * CH + co] = h;
  } else {
    bias[i - WSZ] = p[i];
  }
}

__global__ void k_correction(const float* __restrict__ pred, const double* __restrict__ scale,
                             double omega, int ncells, double* __restrict__ e) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < ncells) e[c] = omega * scale[c / NCELL] * (double)pred[c];
}

// ---------------------------------------------------------------------------
// Block problems: div(D grad e) = r on each 16^3 block with homogeneous
// Dirichlet data on the block faces (ghost = -interior, the homogeneous
// Robin ghost of the FAC error equation), D on faces:
//   dxf[b][z][y][0..16], dyf[b][z][0..16][x], dzf[b][0..16][y][x].
// Cell p: sum_f D_f (e_nbr - e_p) / h^2 = r_p, with e_nbr = -e_p across a
// block face.  Red-black SOR, one work-group per block, e in LDS (FP64).
__device__ inline void block_coeffs(const double* dxf, const double* dyf, const double* dzf,
                                    int x, int y, int z, double c[6]) {
  c[0] = dxf[(z * NB + y) * (NB + 1) + x];
  c[1] = dxf[(z * NB + y) * (NB + 1) + x + 1];
  c[2] = dyf[(z * (NB + 1) + y) * NB + x];
  c[3] = dyf[(z * (NB + 1) + y + 1) * NB + x];
  c[4] = dzf[(z * NB + y) * NB + x];
  c[5] = dzf[((z + 1) * NB + y) * NB + x];
}

__device__ inline double block_nbr_sum(const double* es, int x, int y, int z, const double c[6],
                                       double ep, double* diag) {
  // returns sum_f D_f e_nbr with e_nbr = -e_p across block faces; diag = sum_f D_f
  const int p = (z * NB + y) * NB + x;
  double s = 0.0;
  s += c[0] * (x > 0 ? es[p - 1] : -ep);
  s += c[1] * (x < NB - 1 ? es[p + 1] : -ep);
  s += c[2] * (y > 0 ? es[p - NB] : -ep);
  s += c[3] * (y < NB - 1 ? es[p + NB] : -ep);
  s += c[4] * (z > 0 ? es[p - NB * NB] : -ep);
  s += c[5] * (z < NB - 1 ? es[p + NB * NB] : -ep);
  *diag = c[0] + c[1] + c[2] + c[3] + c[4] + c[5];
  return s;
}

// Value of the lane one to the left (SHIFT < 0) or right of this one within
// its row of 16 lanes, 0 beyond the row's ends.
template <int SHIFT>
__device__ inline double row_shift(double v) {
  constexpr int ctrl = SHIFT < 0 ? 0x111 : 0x101;  // row_shr:1 / row_shl:1
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Red-black SOR of a block by one work-group of 512 threads.  The sweeps run
// hundreds of times over the same block, so what bounds them is the traffic
// of a sweep, not the block's one load: every thread keeps half a z-column
// (8 cells of one (x, y)) with its iterate, right-hand side and six folded
// weights in registers, and only the iterate's copy for the y neighbours is
// in LDS.  Of a cell's six neighbours the two along z are the thread's own
// registers, the two along x come from the neighbouring lanes (a row of 16
// lanes is a row of the block), the two along y from LDS.  With
// w_f = omega D_f / diag and b = omega h^2 r / diag an update is seven fused
// multiply-adds, e' = (1 - omega) e + sum_f w_f e_f - b, diag counting a
// boundary face twice (its ghost is -e) and its w_f being 0.
// 1000 blocks, 400 sweeps: 15.9 ms with the coefficients re-read from L2 and
// the diagonal divided out in every update, 1.02 ms so.
constexpr int kSorThreads = 512;
__global__ __launch_bounds__(kSorThreads) void k_block_sor(
    const double* __restrict__ r, const double* __restrict__ dxf, const double* __restrict__ dyf,
    const double* __restrict__ dzf, double h2, int sweeps, double omega, int from_input,
    double* __restrict__ e) {
  __shared__ double es[NCELL];
  const int b = blockIdx.x;
  const double* rb = r + (size_t)b * NCELL;
  const double* bx = dxf + (size_t)b * NB * NB * (NB + 1);
  const double* by = dyf + (size_t)b * NB * NB * (NB + 1);
  const double* bz = dzf + (size_t)b * NB * NB * (NB + 1);
  double* eb = e + (size_t)b * NCELL;
  const int x = threadIdx.x & 15, y = (threadIdx.x >> 4) & 15;
  const int z0 = (int)(threadIdx.x >> 8) * 8;
  const int q = (x + y) & 1;  // z0 is even
  // slot k of colour c: the cell at z0 + 2k + (q ^ c); its z neighbours are
  // slot k of the other colour (w[4], above it iff q ^ c = 0) and slot
  // k - 1 or k + 1 of it or, past the half column, the cell zn (w[5])
  double u[2][4], rhs[2][4], w[2][4][6];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int qc = q ^ c;
      const int z = z0 + 2 * k + qc;
      const int p = (z * NB + y) * NB + x;
      double f[6];
      block_coeffs(bx, by, bz, x, y, z, f);
      const bool out[6] = {x == 0, x == NB - 1, y == 0, y == NB - 1, z == 0, z == NB - 1};
      double diag = f[0] + f[1] + f[2] + f[3] + f[4] + f[5];
#pragma unroll
      for (int s = 0; s < 6; ++s)
        if (out[s]) diag += f[s];
      const double inv = omega / diag;
#pragma unroll
      for (int s = 0; s < 6; ++s) f[s] = out[s] ? 0.0 : f[s] * inv;
#pragma unroll
      for (int s = 0; s < 4; ++s) w[c][k][s] = f[s];
      w[c][k][4] = qc ? f[4] : f[5];
      w[c][k][5] = qc ? f[5] : f[4];
      rhs[c][k] = h2 * rb[p] * inv;
      u[c][k] = from_input ? eb[p] : 0.0;
      es[p] = u[c][k];
    }
  __syncthreads();
  const double keep = 1.0 - omega;
  const int cell = y * NB + x;
  const int yl = y > 0 ? -NB : 0, yh = y < NB - 1 ? NB : 0;  // a boundary face has w = 0
  for (int s = 0; s < sweeps; ++s) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int qc = q ^ c;
      const int zn = qc ? (z0 + 8 < NB ? z0 + 8 : NB - 1) : (z0 > 0 ? z0 - 1 : 0);
      const double end = es[zn * NB * NB + cell];
      double nl[4], nh[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int p = (z0 + 2 * k + qc) * NB * NB + cell;
        nl[k] = es[p + yl];
        nh[k] = es[p + yh];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double* o = u[c ^ 1];
        const double below = k > 0 ? o[k > 0 ? k - 1 : 0] : end;
        const double above = k < 3 ? o[k < 3 ? k + 1 : 3] : end;
        double v = fma(keep, u[c][k], -rhs[c][k]);
        v = fma(w[c][k][4], o[k], v);
        v = fma(w[c][k][5], qc ? above : below, v);
        v = fma(w[c][k][0], row_shift<-1>(o[k]), v);
        v = fma(w[c][k][1], row_shift<1>(o[k]), v);
        v = fma(w[c][k][2], nl[k], v);
        v = fma(w[c][k][3], nh[k], v);
        u[c][k] = v;
        es[(z0 + 2 * k + qc) * NB * NB + cell] = v;
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      eb[((z0 + 2 * k + (q ^ c)) * NB + y) * NB + x] = u[c][k];
}

// rout = r - div(D grad e) on each block (same operator as k_block_sor).
__global__ __launch_bounds__(256) void k_block_residual(const double* __restrict__ r,
                                                        const double* __restrict__ dxf,
                                                        const double* __restrict__ dyf,
                                                        const double* __restrict__ dzf,
                                                        double inv_h2,
                                                        const double* __restrict__ e,
                                                        double* __restrict__ rout) {
  const int b = blockIdx.x;
  const double* bx = dxf + (size_t)b * NB * NB * (NB + 1);
  const double* by = dyf + (size_t)b * NB * NB * (NB + 1);
  const double* bz = dzf + (size_t)b * NB * NB * (NB + 1);
  const double* eb = e + (size_t)b * NCELL;
  for (int p = threadIdx.x; p < NCELL; p += 256) {
    const int x = p % NB, y = (p / NB) % NB, z = p / (NB * NB);
    double c[6], diag;
    block_coeffs(bx, by, bz, x, y, z, c);
    const double ep = eb[p];
    const double nb = block_nbr_sum(eb, x, y, z, c, ep, &diag);
    rout[(size_t)b * NCELL + p] = r[(size_t)b * NCELL + p] - (nb - diag * ep) * inv_h2;
  }
}

// Level <-> blocks (every patch of the level is one 16^3 block).  Patch
// arrays are ArrayData layout (x fastest over the ghost box); cell data with
// ghost 0 and side data with ghost 0 have the block layouts directly.
// The level's patches are covered by 16^3 windows (one network block each):
// record w = {p, ox, oy, oz, nx, ny, nz, 0}: window cell (x, y, z) is cell
// (ox + x, oy + y, oz + z) of patch p's interior (nx, ny, nz cells); window
// cells beyond the patch read 0 and get no correction.  A 16^3 patch is one
// window at the origin.
struct WinCell {
  int p, px, py, pz, nx, ny, nz;
  bool inside;
};
__device__ inline WinCell win_cell(const int* __restrict__ win, long i) {
  const int w = (int)(i / NCELL), c = (int)(i % NCELL);
  const int* r = win + 8 * w;
  WinCell q;
  q.p = r[0];
  q.px = r[1] + c % NB;
  q.py = r[2] + (c / NB) % NB;
  q.pz = r[3] + c / (NB * NB);
  q.nx = r[4];
  q.ny = r[5];
  q.nz = r[6];
  q.inside = q.px < q.nx && q.py < q.ny && q.pz < q.nz;
  return q;
}

__global__ void k_gather_blocks(double* const* __restrict__ tab, const int* __restrict__ win,
                                int nblocks, double* __restrict__ out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)nblocks * NCELL) return;
  const WinCell q = win_cell(win, i);
  out[i] = q.inside ? tab[q.p][(q.pz * q.ny + q.py) * q.nx + q.px] : 0.0;
}

__global__ void k_logd_blocks(double* const* __restrict__ tx, double* const* __restrict__ ty,
                              double* const* __restrict__ tz, const int* __restrict__ win,
                              int nblocks, double* __restrict__ logd) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)nblocks * NCELL) return;
  const WinCell q = win_cell(win, i);
  if (!q.inside) {
    logd[i] = 0.0;
    return;
  }
  const int x = q.px, y = q.py, z = q.pz, nx = q.nx, ny = q.ny;
  const double* X = tx[q.p];
  const double* Y = ty[q.p];
  const double* Z = tz[q.p];
  const double s = log(X[(z * ny + y) * (nx + 1) + x]) + log(X[(z * ny + y) * (nx + 1) + x + 1]) +
                   log(Y[(z * (ny + 1) + y) * nx + x]) + log(Y[(z * (ny + 1) + y + 1) * nx + x]) +
                   log(Z[(z * ny + y) * nx + x]) + log(Z[((z + 1) * ny + y) * nx + x]);
  logd[i] = s / 6.0;
}

__global__ void k_add_blocks(double* const* __restrict__ tab, int ghost,
                             const int* __restrict__ win, int nblocks,
                             const double* __restrict__ e) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)nblocks * NCELL) return;
  const WinCell q = win_cell(win, i);
  if (!q.inside) return;
  const int sx = q.nx + 2 * ghost, sy = q.ny + 2 * ghost;
  tab[q.p][((q.pz + ghost) * sy + (q.py + ghost)) * sx + (q.px + ghost)] += e[i];
}

// ---------------------------------------------------------------------------
struct Net {
  int max_blocks = 0;
  float* p[NLAYER] = {};     // master parameters
  float* m[NLAYER] = {};
  float* v[NLAYER] = {};
  uint16_t* wf[NLAYER] = {};
  uint16_t* wb[NLAYER] = {};
  float* bias[NLAYER] = {};
  float* grad[NLAYER] = {};
  uint16_t* act[NLAYER] = {};  // act[0] = features, act[1..2] = hidden outputs
  uint16_t* gbuf[2] = {};      // gradients of pre-activations (ping-pong)
  float* pred = nullptr;
  double* scale = nullptr;
  float* partial = nullptr;
  float* loss_partial = nullptr;
  float* loss = nullptr;
  double* blk[3] = {};         // level gathers: residual, log D, correction
  int step = 0;
  int attached = 0;            // solvers using the network (learned_attach)
  int cin[NLAYER] = {2, CH, CH};
  int cout[NLAYER] = {CH, CH, 1};
};

struct HipFail {
  hipError_t e;
};
inline void ck(hipError_t e) {
  if (e != hipSuccess) throw HipFail{e};
}
struct ArgFail {
  std::string msg;
};
inline void need(bool ok, const char* msg) {
  if (!ok) throw ArgFail{msg};
}

template <class F>
int guarded(F&& f) {
  try {
    f();
    ck(hipGetLastError());
    return 0;
  } catch (const HipFail& e) {
    samrai_amd::set_last_error(std::string("HIP error: ") + hipGetErrorString(e.e));
  } catch (const ArgFail& e) {
    samrai_amd::set_last_error(e.msg);
  } catch (...) {
    samrai_amd::set_last_error("unknown error in learned smoother");
  }
  return -1;
}

template <class T>
T* dalloc(size_t n) {
  void* ptr = nullptr;
  ck(hipMalloc(&ptr, n * sizeof(T)));
  return static_cast<T*>(ptr);
}

// Work-groups (slabs of partial sums) of the weight gradient, and z-slabs per
// block: quarters of a block while whole ones would leave compute units idle,
// at most two work-groups per compute unit, which then take several.
constexpr int kWgradGroups = 512;
constexpr int wgrad_slabs(int nblocks) { return nblocks < 128 ? 4 : 1; }
constexpr int wgrad_groups(int nblocks) {
  return std::min(nblocks * wgrad_slabs(nblocks), kWgradGroups);
}

// Gradient slabs, one per work-group, of the allocation-free weight gradient
// (sfac_conv3x3x3_wgrad_bf16_noalloc): one array per GPU, held until the
// process ends.  Host code never passes `scratch` itself to a kernel (on the
// host it names a stand-in, not device memory): it passes the address that
// hipGetSymbolAddress returns for the current device.
constexpr int NOALLOC_MAX_BLOCKS = SFAC_WGRAD_NOALLOC_MAX_BLOCKS;
constexpr int NOALLOC_SLABS = 4 * NOALLOC_MAX_BLOCKS;
constexpr size_t NOALLOC_FLOATS = (size_t)NOALLOC_SLABS * GSZ;  // 1.75 MiB
constexpr bool noalloc_slabs_fit() {
  for (int n = 1; n <= NOALLOC_MAX_BLOCKS; ++n)
    if (wgrad_groups(n) > NOALLOC_SLABS) return false;
  return true;
}
static_assert(noalloc_slabs_fit(), "a slab for every work-group");
__device__ __align__(256) float scratch[NOALLOC_FLOATS];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up on the first
// call for that device.
float* scratch_on_current_device() {
  int dev = 0;
  ck(hipGetDevice(&dev));
  need(dev >= 0 && dev < kMaxDevices, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    ck(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    need(ptr != nullptr, "hipGetSymbolAddress returned a null scratch address");
    g_scratch_ptr[dev] = static_cast<float*>(ptr);
  }
  return g_scratch_ptr[dev];
}

void launch_conv(int mode, const uint16_t* x, const uint16_t* w, const float* bias,
                 const uint16_t* mask, uint16_t* out, float* pred, int nblocks, hipStream_t s) {
  static_assert(4 * CONV_ROWS == NB, "a work-group's four waves cover one z-plane");
  const int nplanes = nblocks * NB;
  const dim3 grid(nplanes), block(256);
  if (mode == MODE_HIDDEN)
    hipLaunchKernelGGL(k_conv<MODE_HIDDEN>, grid, block, 0, s, x, w, bias, mask, out, pred,
                       nplanes);
  else if (mode == MODE_FINAL)
    hipLaunchKernelGGL(k_conv<MODE_FINAL>, grid, block, 0, s, x, w, bias, mask, out, pred,
                       nplanes);
  else
    hipLaunchKernelGGL(k_conv<MODE_BWD>, grid, block, 0, s, x, w, bias, mask, out, pred,
                       nplanes);
}

void launch_wgrad_partial(const uint16_t* x, const uint16_t* gz, float* partial, int nblocks,
                          hipStream_t s) {
  hipLaunchKernelGGL(k_wgrad, dim3(wgrad_groups(nblocks)), dim3(256), 0, s, x, gz, partial, nblocks,
                     wgrad_slabs(nblocks));
}

void launch_wgrad(const uint16_t* x, const uint16_t* gz, float* partial, float* grad, int nblocks,
                  hipStream_t s) {
  launch_wgrad_partial(x, gz, partial, nblocks, s);
  GradOut out{{grad, nullptr, nullptr}};
  hipLaunchKernelGGL(k_wgrad_reduce, dim3((GSZ + 15) / 16), dim3(256), 0, s, partial,
                     wgrad_groups(nblocks), (size_t)0, out);
}

// Work-groups of k_forward: one per compute unit (its LDS allows no more).
constexpr int kForwardGroups = 256;

Forward forward_args(Net* n, int nblocks) {
  Forward P{};
  P.x0 = n->act[0];
  P.x0_out = n->act[0];
  P.scale = n->scale;
  for (int l = 0; l < NLAYER; ++l) {
    P.w[l] = n->wf[l];
    P.bias[l] = n->bias[l];
  }
  P.act[0] = n->act[1];
  P.act[1] = n->act[2];
  P.pred = n->pred;
  P.nblocks = nblocks;
  return P;
}

// Prediction and hidden activations from the features in act[0].  Work-groups
// per block: whole blocks once they fill the compute units, else quarters
// (which form five more planes of each layer than they need alone).
void forward(Net* n, int nblocks, hipStream_t s) {
  const int slabs = nblocks >= 256 ? 1 : 4;
  hipLaunchKernelGGL(k_forward<false>, dim3(std::min(nblocks * slabs, kForwardGroups)),
                     dim3(FWD_THREADS), 0, s, forward_args(n, nblocks), slabs);
}

// Scale, features, prediction and correction e of every block from r and
// log D, with the buffers features + forward leave.
void correction(Net* n, const double* r, const double* logd, double logd_const, double h2,
                double omega, double* e, int nblocks, hipStream_t s) {
  Forward P = forward_args(n, nblocks);
  P.r = r;
  P.logd = logd;
  P.logd_const = logd_const;
  P.h2 = h2;
  P.omega = omega;
  P.e = e;
  hipLaunchKernelGGL(k_forward<true>, dim3(std::min(nblocks, kForwardGroups)),
                     dim3(FWD_THREADS), 0, s, P, 1);
}

// Loss and gradients of every layer (after forward on the same features).
void backward(Net* n, const double* target, int nblocks, hipStream_t s) {
  const int ncells = nblocks * NCELL;
  const int nlb = (ncells + 255) / 256;
  hipLaunchKernelGGL(k_loss, dim3(nlb), dim3(256), 0, s, n->pred, target, n->scale, ncells,
                     1.f / (float)ncells, n->gbuf[0], n->loss_partial);
  hipLaunchKernelGGL(k_sum_f32, dim3(1), dim3(256), 0, s, n->loss_partial, nlb,
                     1.f / (float)ncells, n->loss);
  // layer 3: gradient gbuf[0] (channel 0 only); the layers' partial sums side
  // by side, summed in one launch
  const size_t stride = (size_t)wgrad_groups(nblocks) * GSZ;
  launch_wgrad_partial(n->act[2], n->gbuf[0], n->partial + 2 * stride, nblocks, s);
  launch_conv(MODE_BWD, n->gbuf[0], n->wb[2], nullptr, n->act[2], n->gbuf[1], nullptr, nblocks, s);
  // layer 2
  launch_wgrad_partial(n->act[1], n->gbuf[1], n->partial + stride, nblocks, s);
  launch_conv(MODE_BWD, n->gbuf[1], n->wb[1], nullptr, n->act[1], n->gbuf[0], nullptr, nblocks, s);
  // layer 1 (its input gradient is not needed)
  launch_wgrad_partial(n->act[0], n->gbuf[0], n->partial, nblocks, s);
  GradOut out{{n->grad[0], n->grad[1], n->grad[2]}};
  hipLaunchKernelGGL(k_wgrad_reduce, dim3((GSZ + 15) / 16, NLAYER), dim3(256), 0, s, n->partial,
                     wgrad_groups(nblocks), stride, out);
}

void adam(Net* n, float lr, hipStream_t s) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  n->step += 1;
  const float bc1 = 1.f - std::pow(b1, (float)n->step);
  const float bc2 = 1.f - std::pow(b2, (float)n->step);
  AdamLayers a;
  for (int l = 0; l < NLAYER; ++l)
    a.l[l] = AdamLayer{n->p[l],  n->m[l],  n->v[l],    n->grad[l], n->wf[l],
                       n->wb[l], n->bias[l], n->cin[l], n->cout[l]};
  hipLaunchKernelGGL(k_adam, dim3((PSZ + 255) / 256, NLAYER), dim3(256), 0, s, a, lr, b1, b2, eps,
                     bc1, bc2);
}

void sync_weights(Net* n, hipStream_t s) {
  for (int l = 0; l < NLAYER; ++l)
    hipLaunchKernelGGL(k_sync_weights, dim3((PSZ + 255) / 256), dim3(256), 0, s, n->p[l],
                       n->wf[l], n->wb[l], n->bias[l]);
}

// He-style uniform initialisation from a fixed 64-bit LCG (host), biases 0,
// channels outside each layer's real counts 0.
void init_params(Net* n, unsigned long long seed, hipStream_t s) {
  uint64_t st = seed * 6364136223846793005ull + 1442695040888963407ull;
  auto uni = [&]() {
    st = st * 6364136223846793005ull + 1442695040888963407ull;
    return ((st >> 11) * (1.0 / 9007199254740992.0)) * 2.0 - 1.0;
  };
  std::vector<float> h(PSZ);
  for (int l = 0; l < NLAYER; ++l) {
    const double a = std::sqrt(6.0 / (NTAP * n->cin[l]));
    for (int i = 0; i < PSZ; ++i) {
      float val = 0.f;
      if (i < WSZ) {
        const int co = (i / CH) % CH, ci = i % CH;
        if (ci < n->cin[l] && co < n->cout[l]) val = (float)(a * uni());
      }
      h[i] = val;
    }
    ck(hipMemcpyAsync(n->p[l], h.data(), PSZ * sizeof(float), hipMemcpyHostToDevice, s));
    ck(hipMemsetAsync(n->m[l], 0, PSZ * sizeof(float), s));
    ck(hipMemsetAsync(n->v[l], 0, PSZ * sizeof(float), s));
  }
  ck(hipStreamSynchronize(s));
  sync_weights(n, s);
  n->step = 0;
}

void free_net(Net* n) {
  for (int l = 0; l < NLAYER; ++l) {
    (void)hipFree(n->p[l]);
    (void)hipFree(n->m[l]);
    (void)hipFree(n->v[l]);
    (void)hipFree(n->wf[l]);
    (void)hipFree(n->wb[l]);
    (void)hipFree(n->bias[l]);
    (void)hipFree(n->grad[l]);
    (void)hipFree(n->act[l]);
  }
  (void)hipFree(n->gbuf[0]);
  (void)hipFree(n->gbuf[1]);
  (void)hipFree(n->pred);
  (void)hipFree(n->scale);
  (void)hipFree(n->partial);
  (void)hipFree(n->loss_partial);
  (void)hipFree(n->loss);
  for (int k = 0; k < 3; ++k) (void)hipFree(n->blk[k]);
  delete n;
}

Net* net_of(void* h, int nblocks) {
  need(h != nullptr, "null learned smoother");
  Net* n = static_cast<Net*>(h);
  need(nblocks >= 0 && nblocks <= n->max_blocks, "block count outside [0, max_blocks]");
  return n;
}

}  // namespace

namespace samrai_amd {
// A solver attaching (delta 1) or detaching (-1) the network: a network
// with a solver attached cannot be destroyed (the solver's captured cycle
// graphs hold its buffers).
int learned_attach(void* net, int delta) {
  return guarded([&] {
    need(net != nullptr, "null learned smoother");
    Net* n = static_cast<Net*>(net);
    need(n->attached + delta >= 0, "learned smoother: detach without attach");
    n->attached += delta;
  });
}

// Blocks the network holds buffers for.
int learned_max_blocks(void* net) {
  return net ? static_cast<Net*>(net)->max_blocks : 0;
}

// The learned correction of one level over the 16^3 windows `windows`
// (device, 8 ints each, see win_cell) covering its patches:
// u += omega * s * net(r h^2 / s, log D) on every window cell inside its
// patch, r cell data with ghost 0, D side data with ghost 0 (dtab null:
// log D = logd_const everywhere), u cell data with ghost `ughost`.
// Called by sfac_ops_learned_correct (capi.cpp) after its checks.
int learned_correct_level(void* net, double* const* utab, int ughost, double* const* rtab,
                          double* const* const* dtab, double logd_const, const int* windows,
                          int nblocks, double h, double omega, hipStream_t s) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    need(utab && rtab, "null patch tables");
    need(windows || nblocks == 0, "null window table");
    need(h > 0.0, "h must be positive");
    if (nblocks == 0) return;
    const int ncells = nblocks * NCELL;
    const dim3 grid((ncells + 255) / 256), block(256);
    hipLaunchKernelGGL(k_gather_blocks, grid, block, 0, s, rtab, windows, nblocks, n->blk[0]);
    const double* logd = nullptr;
    if (dtab) {
      hipLaunchKernelGGL(k_logd_blocks, grid, block, 0, s, dtab[0], dtab[1], dtab[2], windows,
                         nblocks, n->blk[1]);
      logd = n->blk[1];
    }
    correction(n, n->blk[0], logd, logd_const, h * h, omega, n->blk[2], nblocks, s);
    hipLaunchKernelGGL(k_add_blocks, grid, block, 0, s, utab, ughost, windows, nblocks,
                       n->blk[2]);
  });
}
}  // namespace samrai_amd

namespace {
__global__ void k_zero_f32(float* __restrict__ p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    p[i] = 0.f;
}
}  // namespace

extern "C" {

int sfac_conv3x3x3_bf16(const uint16_t* x, const uint16_t* w, const float* bias,
                        const uint16_t* mask, uint16_t* out, float* pred, int nblocks, int mode,
                        hipStream_t stream) {
  return guarded([&] {
    need(nblocks >= 0, "negative block count");
    need(mode >= 0 && mode <= 2, "mode must be 0 (hidden), 1 (final) or 2 (backward data)");
    need(x && w, "null input or weights");
    need(mode != MODE_HIDDEN || (bias && out), "hidden mode needs bias and out");
    need(mode != MODE_FINAL || (bias && pred), "final mode needs bias and pred");
    need(mode != MODE_BWD || (mask && out), "backward mode needs mask and out");
    if (nblocks == 0) return;
    launch_conv(mode, x, w, bias, mask, out, pred, nblocks, stream);
  });
}

int sfac_conv3x3x3_wgrad_bf16(const uint16_t* x, const uint16_t* gz, float* grad, float* partial,
                              int nblocks, hipStream_t stream) {
  return guarded([&] {
    need(nblocks >= 0, "negative block count");
    need(x && gz && grad && partial, "null pointer");
    if (nblocks == 0) {
      // a fill kernel, not a memset node (callers may capture this call)
      hipLaunchKernelGGL(k_zero_f32, dim3((GSZ + 255) / 256), dim3(256), 0, stream, grad, GSZ);
      return;
    }
    launch_wgrad(x, gz, partial, grad, nblocks, stream);
  });
}

int sfac_conv3x3x3_wgrad_bf16_noalloc(const uint16_t* x, const uint16_t* gz, float* grad,
                                      int nblocks, hipStream_t stream) {
  return guarded([&] {
    need(nblocks >= 0, "negative block count");
    need(nblocks <= NOALLOC_MAX_BLOCKS,
         "sfac_conv3x3x3_wgrad_bf16_noalloc: nblocks exceeds the static scratch maximum "
         "(SFAC_WGRAD_NOALLOC_MAX_BLOCKS = 16)");
    need(x && gz && grad, "null pointer");
    if (nblocks == 0) {
      hipLaunchKernelGGL(k_zero_f32, dim3((GSZ + 255) / 256), dim3(256), 0, stream, grad, GSZ);
      return;
    }
    // every work-group of k_wgrad writes its whole slab, so nothing needs clearing
    launch_wgrad(x, gz, scratch_on_current_device(), grad, nblocks, stream);
  });
}

size_t sfac_conv3x3x3_wgrad_partial_size(int nblocks) {
  // no less than any smaller block count needs
  return nblocks <= 0 ? 0 : (size_t)std::min(4l * nblocks, (long)kWgradGroups) * GSZ;
}

int sfac_block_sor(const double* r, const double* dxf, const double* dyf, const double* dzf,
                   double h, int sweeps, double omega, int from_input, double* e, int nblocks,
                   hipStream_t stream) {
  return guarded([&] {
    need(nblocks >= 0 && sweeps >= 0, "negative block count or sweep count");
    need(r && dxf && dyf && dzf && e, "null pointer");
    need(h > 0.0, "h must be positive");
    if (nblocks == 0) return;
    hipLaunchKernelGGL(k_block_sor, dim3(nblocks), dim3(kSorThreads), 0, stream, r, dxf, dyf, dzf, h * h,
                       sweeps, omega, from_input, e);
  });
}

int sfac_block_residual(const double* r, const double* dxf, const double* dyf, const double* dzf,
                        double h, const double* e, double* rout, int nblocks,
                        hipStream_t stream) {
  return guarded([&] {
    need(nblocks >= 0, "negative block count");
    need(r && dxf && dyf && dzf && e && rout, "null pointer");
    need(h > 0.0, "h must be positive");
    if (nblocks == 0) return;
    hipLaunchKernelGGL(k_block_residual, dim3(nblocks), dim3(256), 0, stream, r, dxf, dyf, dzf,
                       1.0 / (h * h), e, rout);
  });
}

int sfac_learned_create(int max_blocks, unsigned long long seed, void** out) {
  return guarded([&] {
    need(out != nullptr, "null output handle");
    need(max_blocks > 0, "max_blocks must be positive");
    Net* n = new Net;
    n->max_blocks = max_blocks;
    try {
      const size_t ncells = (size_t)max_blocks * NCELL;
      for (int l = 0; l < NLAYER; ++l) {
        n->p[l] = dalloc<float>(PSZ);
        n->m[l] = dalloc<float>(PSZ);
        n->v[l] = dalloc<float>(PSZ);
        n->wf[l] = dalloc<uint16_t>(WSZ);
        n->wb[l] = dalloc<uint16_t>(WSZ);
        n->bias[l] = dalloc<float>(CH);
        n->grad[l] = dalloc<float>(GSZ);
        n->act[l] = dalloc<uint16_t>(ncells * CH);
      }
      n->gbuf[0] = dalloc<uint16_t>(ncells * CH);
      n->gbuf[1] = dalloc<uint16_t>(ncells * CH);
      n->pred = dalloc<float>(ncells);
      n->scale = dalloc<double>(max_blocks);
      // (a smaller batch may take more work-groups than the largest one)
      n->partial = dalloc<float>((size_t)std::min(4l * max_blocks, (long)kWgradGroups) * NLAYER *
                                 GSZ);
      n->loss_partial = dalloc<float>((ncells + 255) / 256);
      n->loss = dalloc<float>(1);
      for (int k = 0; k < 3; ++k) n->blk[k] = dalloc<double>(ncells);
      init_params(n, seed, 0);
      ck(hipStreamSynchronize(0));
    } catch (...) {
      free_net(n);
      throw;
    }
    *out = n;
  });
}

int sfac_learned_destroy(void* net) {
  return guarded([&] {
    if (net) {
      need(static_cast<Net*>(net)->attached == 0,
           "learned smoother: the network is attached to a solver (detach it with "
           "sfac_solver_set_learned_smoother(s, NULL, ...) before destroying it)");
      ck(hipDeviceSynchronize());
      free_net(static_cast<Net*>(net));
    }
  });
}

int sfac_learned_features(void* net, const double* r, const double* logd, double h, int nblocks,
                          hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    need(r != nullptr, "null residual");
    need(h > 0.0, "h must be positive");
    if (nblocks == 0) return;
    hipLaunchKernelGGL(k_features, dim3(nblocks), dim3(kFeatThreads), 0, stream, r, logd, 0.0, h * h,
                       n->act[0], n->scale);
  });
}

int sfac_learned_forward(void* net, int nblocks, hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    if (nblocks == 0) return;
    forward(n, nblocks, stream);
  });
}

int sfac_learned_correction(void* net, double omega, double* e, int nblocks, hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    need(e != nullptr, "null correction");
    if (nblocks == 0) return;
    const int ncells = nblocks * NCELL;
    hipLaunchKernelGGL(k_correction, dim3((ncells + 255) / 256), dim3(256), 0, stream, n->pred,
                       n->scale, omega, ncells, e);
  });
}

int sfac_learned_apply(void* net, const double* r, const double* logd, double h, double omega,
                       double* e, int nblocks, hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    need(r && e, "null residual or correction");
    need(h > 0.0, "h must be positive");
    if (nblocks == 0) return;
    correction(n, r, logd, 0.0, h * h, omega, e, nblocks, stream);
  });
}

int sfac_learned_backward(void* net, const double* target, int nblocks, hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    need(target != nullptr, "null target");
    need(nblocks > 0, "backward needs at least one block");
    backward(n, target, nblocks, stream);
  });
}

int sfac_learned_adam(void* net, float lr, hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, 0);
    adam(n, lr, stream);
  });
}

int sfac_learned_train_step(void* net, const double* r, const double* logd, const double* target,
                            double h, int nblocks, float lr, hipStream_t stream) {
  return guarded([&] {
    Net* n = net_of(net, nblocks);
    need(r && target, "null residual or target");
    need(h > 0.0 && nblocks > 0, "bad h or block count");
    hipLaunchKernelGGL(k_features, dim3(nblocks), dim3(kFeatThreads), 0, stream, r, logd, 0.0, h * h,
                       n->act[0], n->scale);
    forward(n, nblocks, stream);
    backward(n, target, nblocks, stream);
    adam(n, lr, stream);
  });
}

int sfac_learned_get_params(void* net, float* host, int which) {
  return guarded([&] {
    Net* n = net_of(net, 0);
    need(host != nullptr, "null host buffer");
    need(which >= 0 && which <= 1, "which: 0 = parameters, 1 = gradients");
    for (int l = 0; l < NLAYER; ++l) {
      if (which == 0)
        ck(hipMemcpy(host + (size_t)l * PSZ, n->p[l], PSZ * sizeof(float), hipMemcpyDeviceToHost));
      else
        ck(hipMemcpy(host + (size_t)l * GSZ, n->grad[l], GSZ * sizeof(float),
                     hipMemcpyDeviceToHost));
    }
  });
}

int sfac_learned_set_params(void* net, const float* host) {
  return guarded([&] {
    Net* n = net_of(net, 0);
    need(host != nullptr, "null host buffer");
    for (int l = 0; l < NLAYER; ++l) {
      ck(hipMemcpy(n->p[l], host + (size_t)l * PSZ, PSZ * sizeof(float), hipMemcpyHostToDevice));
      ck(hipMemset(n->m[l], 0, PSZ * sizeof(float)));
      ck(hipMemset(n->v[l], 0, PSZ * sizeof(float)));
    }
    sync_weights(n, 0);
    ck(hipStreamSynchronize(0));
    n->step = 0;
  });
}

int sfac_learned_loss(void* net, float* loss) {
  return guarded([&] {
    Net* n = net_of(net, 0);
    need(loss != nullptr, "null loss");
    ck(hipMemcpy(loss, n->loss, sizeof(float), hipMemcpyDeviceToHost));
  });
}

int sfac_learned_buffers(void* net, void** features, float** pred, double** scale) {
  return guarded([&] {
    Net* n = net_of(net, 0);
    if (features) *features = n->act[0];
    if (pred) *pred = n->pred;
    if (scale) *scale = n->scale;
  });
}

}  // extern "C"
