// Colour-fused red-black sweeps on a level that is one rectangle of cells.
//
// The coarsest level of a FAC solve usually tiles the physical domain
// exactly (level 0 of every benchmark hierarchy).  Its same-level ghost
// copies are exact copies and its only other ghosts are physical Robin
// ghosts, so the patches can be gathered once per smoothing call into
// contiguous arrays and every sweep becomes ONE launch: each work-group
// loads a tile plus a two-cell halo into LDS, updates the red cells of the
// tile grown by one (the halo reds are recomputed redundantly, from the same
// inputs and in the same expression order, so they equal the neighbour
// tile's values bit for bit), refreshes the physical ghosts in LDS, then
// updates the black cells of the tile and writes the tile back.  The result
// is identical to the patch-by-patch red pass / ghost fill / black pass /
// ghost fill sequence of CellPoissonFACOps::smoothErrorByRedBlack
// (solv/CellPoissonFACOps.C:1338-1514).
#pragma once

#include "level_kernels.h"

namespace sfac {

struct BoxLevel {
  int dim;
  int n[3];         // cells per axis
  int lo[3];        // level index of cell (0,0,0)
  double dx[3];
  int shift;        // colour shift: red <=> (i + j + k + shift) even (level indices)
  int lp_lo[3];     // last patch box, relative to lo (early-exit test)
  int lp_hi[3];
};

// Arrays of the level.  fp32 = 0: FP64 storage and arithmetic (the
// reference's).  fp32 = 1: the arrays hold float values (the pointers are
// reinterpreted; buffers are allocated at the FP64 size either way) and the
// sweeps, transfers and multigrid compute in FP32; the early-exit maxima and
// norm partial sums stay FP64.
struct BoxArrays {
  const double* ein;    // u before the sweep: n0*n1*n2, no ghosts (nullptr: u = 0)
  double* eout;         // u after the sweep (a second buffer: work-groups read
                        // their halos from ein while others write eout)
  const double* r;      // same shape
  const double* D[3];   // side data per axis, +1 along the axis (variable D)
  const double* C;      // cell data (C mode 2)
  double dconst;
  int cmode;
  double cconst;
  int fp32;
};

// The same arrays typed by their storage precision (device side).
template <typename T>
struct BoxArraysT {
  const T* ein;
  T* eout;
  const T* r;
  const T* D[3];
  const T* C;
  double dconst;
  int cmode;
  double cconst;
};

// Early-exit test of the sweep before this launch.  slots: three slots
// (nullptr without a tolerance); sweep s raises slot s % 3 to the max
// |residual| over the last patch (an atomic max of the bit patterns, which
// order like the values for non-negative doubles), reads slot (s + 2) % 3
// (the previous sweep's) and clears slot (s + 1) % 3 for the next sweep.
// A slot has eight words, on lines of their own, a work-group raising the one
// that its index picks: hundreds of work-groups raising one word wait for each
// other, and looking at the word first costs a round trip.  us per sweep, FP64,
// with one word, one looked at first, eight: 128^3 in one patch 34.4, 29.5,
// 19.1; D per face 37.5, 41.3, 31.0; 64^3 9.9, 8.5, 8.6; 128^3 with a last patch
// of 64^3 18.1, 20.1, 18.4; D per face 29.0, 31.0, 29.6.
constexpr int kCheckWords = 8, kCheckLine = 16;
constexpr int kCheckSlot = kCheckWords * kCheckLine, kCheckSize = 3 * kCheckSlot;
struct BoxCheck {
  unsigned long long* slots;
  int tlo[3], tn[3];    // tile range of the last patch
  int sweep;            // index of this sweep
  double tol;
  int* stop;
  int* sweeps;
  double* maxres_out;
};

// Tile shape of a fused sweep.
struct BoxTile {
  int tx, ty, tz;
};
// Tile shapes compiled in (index = variant), per dimension.
constexpr int kBoxTile16x8x4 = 10;  // 3-D
int box_tile_variants(int dim);
BoxTile box_tile(int dim, int variant);

void launch_box_rbgs(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc, int homogeneous,
                     const BoxCheck& K, int variant, hipStream_t s);
// After the last sweep: maxres / sweep count of the last sweep when the
// loop did not stop early.
void launch_box_final_check(const BoxCheck& K, int nsweeps, hipStream_t s);

// Copy cell data between the patches of a level (interior cells) and a
// contiguous box array: to_box 1 gathers, 0 scatters.  The box array is
// box[0] or box[1] by the parity of *count (count == nullptr: of count_host),
// which lets the scatter follow a sweep count known only on the device.
// fp32: the box arrays hold float (converted from / to the FP64 patch data).
// patch_elem: bytes per patch-data value (8 FP64; 4 FP32 and 2 BF16 for the
// mixed-precision error vector, whose table is then typed double* only
// nominally).
void launch_box_cells(const GhostLaunch& cells, const LevelGeom& L, double* const* x, int g,
                      double* box0, double* box1, const int* count, int count_host,
                      const BoxLevel& G, int to_box, hipStream_t s, int fp32 = 0,
                      int patch_elem = 8);
// Gather side data of axis a into the box face array; with verify, faces
// shared by two patches are then compared and *mismatch set to 1 if the
// patches hold different values there.
void launch_box_side(const LevelGeom& L, const double* const* x, int g, int a, double* box,
                     const BoxLevel& G, int* mismatch, hipStream_t s, int verify,
                     int fp32 = 0);

// ---- levels that fit one work-group's LDS (box_small.hip) ----
// Does one work-group hold the level (cells, coefficients of A's kind), and is
// it the faster way to take that many sweeps?
bool box_lds_pays(const BoxLevel& G, const BoxArrays& A, int sweeps);
// `sweeps` red-black sweeps in one launch, homogeneous Robin ghosts: u from
// uin (nullptr: 0) to e0 or e1 by the parity of the sweeps done.  With check,
// K's early-exit test runs after every sweep (tol, stop, sweeps, maxres_out
// as launch_box_rbgs and launch_box_final_check leave them); without,
// nothing is done once *K.stop is set.
void launch_box_lds_rbgs(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc,
                         const double* uin, double* e0, double* e1, int sweeps,
                         const BoxCheck& K, int check, hipStream_t s);

// ---- two sweeps per launch on levels too large for that (box_pair.hip) ----
// Early-exit data of launch number `launch` of a smoothing call.  slots: six
// words (nullptr without a tolerance), two per launch of three; a launch
// raises its two to the max |residual| of its sweeps over the last patch,
// reads those of the launch before it (which took `prev` sweeps) and clears
// those of the next.  When that launch met the tolerance it records stop,
// sweeps, maxres_out and buffer (0: the result is in the buffer launch 0 read,
// 1: in the other), after repeating a first sweep that already met it; final:
// the launch after the last sweeps, which records in any case and sweeps no
// further.
struct PairCheck {
  unsigned long long* slots;
  int launch, prev, final;
  double tol;
  int* stop;
  int* sweeps;
  int* buffer;
  double* maxres_out;
};
// Levels (cells) on which a launch of two sweeps is faster than two launches,
// us per sweep with variable D: 3-D 48^3 5.7 (singly 6.3), 64^3 10.4 (7.4);
// 2-D up to the largest measured, 500^2 3.5 (6.0).  On small 3-D levels 8x8x4
// tiles give the machine more work-groups than 8x8x8 ones: 32^3 has 128 with
// the one, 64 with the other; from 45 x 58 x 39 on there are enough of both and
// 8x8x4 only adds redundant cells (9.8 against 5.7).
constexpr long kPairCells3 = 150000, kPairCells2 = 300000, kPairSmallTile = 40000;
bool box_pair_pays(const BoxLevel& G);
// One or two sweeps from A.ein (nullptr: 0) to A.eout; without slots nothing
// is done once *K.stop is set.
void launch_box_pair(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc,
                     const PairCheck& K, int sweeps, hipStream_t s);

// The lower part of a multigrid V-cycle in one launch, over the n levels G
// (each half the one before) with arrays A (r of the first is its right-hand
// side): pre-sweeps, residual restriction, ..., `last` sweeps from 0 on the
// smallest, prolongation, post-sweeps; the first level's error from 0
// (from_input 0) or from e, to e.  columns (the first level's cells): the map
// from right-hand side to error instead, as a row-major matrix in e.
// mg_bottom_first: the first of n levels with at most kMGDenseCells cells
// from which on they fit a work-group (n: none).
constexpr int kMGDenseCells = 1024;
int mg_bottom_first(const BoxLevel* G, int n);
void launch_mg_bottom(const BoxLevel* G, const BoxArrays* A, int n, const RobinDev& bc, int pre,
                      int post, int last, double* e, int from_input, int columns,
                      const int* stop, hipStream_t s);
// e = B f for that matrix of n rows.
void launch_mg_dense(const double* B, int n, const double* f, double* e, int fp32,
                     const int* stop, hipStream_t s);

// ---- geometric multigrid on a single-rectangle level ----
// Edge of the smallest multigrid grid (halving stops there), and the number
// of partial sums launch_mg_sumsq writes.
int mg_small_edge();
int mg_partials();
// Arrays u, x, fc, ec, ef, Dc, Cc have the precision of A.fp32 (fp32).
// fc = mean over the 2^dim children of f - (div D grad u + C u) on Gf.
void launch_mg_restrict_residual(const BoxLevel& Gf, const BoxArrays& A, const RobinDev& bc,
                                 const double* u, const BoxLevel& Gc, double* fc,
                                 const int* stop, hipStream_t s);
// ef += separable linear interpolation of ec (homogeneous Robin beyond the domain).
void launch_mg_prolong_add(const BoxLevel& Gc, const RobinDev& bc, const double* ec,
                           const BoxLevel& Gf, double* ef, const int* stop, hipStream_t s,
                           int fp32 = 0);
// Coarse D faces (mean of the fine faces they cover) and C (mean of children).
void launch_mg_coarsen_coef(const BoxLevel& Gf, const BoxArrays& Af, const BoxLevel& Gc,
                            double* const* Dc, double* Cc, hipStream_t s);
// mg_partials() partial sums of x^2 (x != nullptr) or of the squared residual of u.
void launch_mg_sumsq(const BoxLevel& G, const BoxArrays& A, const RobinDev& bc, const double* u,
                     const double* x, double* partial, const int* stop, hipStream_t s);
// *out = the sum of n partials (launch_sum's order), then the
// relative-residual test of iteration it on rr = out (it < 0: the b = 0 test
// only), in one launch (nothing once *stop is set).
void launch_mg_sum_check(const double* partial, int n, double* out, const double* bb, double tol,
                         int it, int* stop, int* iters, double* relres, hipStream_t s);

}  // namespace sfac
