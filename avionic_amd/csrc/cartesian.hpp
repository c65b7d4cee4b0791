// Coil-fused masked Cartesian operator pair (K, K^H) on compact k-space.
//
// K  (image -> k-space): z[t,c] = M_t . F^{-1}_ortho(b1_c . u_t)
// K^H (k-space -> image): u_t   = sum_c conj(b1_c) . F_ortho(M_t . z[t,c])
// (CUDA/src/cartesian_operator.cpp:65-160; matlab/backward_opt.m,
// forward_opt.m).
//
// k-space is stored compactly: only the phase-encode rows that carry a nonzero
// mask value are kept, as [t][c][k][x] with k over the sampled rows of frame t.
// A 2D transform is split into a column pass (along y, LDS tile of XB
// columns, coils looped inside the workgroup so the image is read once) and a
// row pass (along x, only sampled rows).  The dual update of z, its prox and
// the adjoint's row transform are fused into the forward row pass.
#pragma once

#include <algorithm>
#include <vector>

#include "common.hpp"

namespace avionic {

// Two-stage passes: butterflies of the radix-rb stage that one lane runs at
// most (16 values in registers).
__host__ __device__ constexpr int two_most(int rb) { return rb <= 4 ? 4 : (rb <= 8 ? 2 : 1); }

struct CartGeom {
  int W, H, C, T;
  int centered;
  int XB, lxb, nxb;  // columns per column-pass tile (two-stage: 2^lxb), tiles
  int RB;            // rows per row-pass block
  int lja, ljb;      // two-stage: log2 of the lanes per row in the radix-ra / -rb stages
  int ckind, rkind;  // kernels that run it (ColKind, RowKind)
  long nrows;          // sampled rows over all frames (row_off[T])
  long nrows_c;        // C * nrows
  const int *row_off;  // [T+1]
  const int *rows;     // [nrows] ky of each sampled row, frame-major
  const float *mrows;  // [nrows][W] mask values of the sampled rows
  const int4 *rowinfo; // [nrows_c] (t, c, r = row_off[t] + k, ky) per compact row
  const int *rowmap;   // [T][H] compact row index k of (t, ky), -1 if not sampled
  float scale;         // 1 / sqrt(H W)
  FftPlan pw, ph;
};

// Kernels of the column passes: runtime plan, two-stage (cart_two.hpp), wide
// runtime plan, two-stage with the constants of length 256.
enum ColKind { kColRt = 0, kColTwo = 1, kColWide = 2, kCol256 = 3 };
constexpr int kColKinds = 4;
// Kernels of the row pass: two-stage, runtime plan, wide runtime plan, and the
// two-stage one of the engine without a bound on its registers (length 256).
enum RowKind { kRowTwo = 0, kRowRt = 1, kRowWide = 2, kRow256 = 3 };
constexpr int kRowKinds = 4;

// Row-pass modes.
enum RowMode {  // Norm2, Residual: one partial sum per row block
  kRowApplyK = 0,     // out = K(u) rows (compact or dense)
  kRowDualUpdate = 1, // z = (z + s K u - s d)/(1 + s/l); zhat = F_row(M z)
  kRowNorm2 = 2,      // partial sums of |K u|^2
  kRowAdjDense = 3,   // zhat = F_row(M z_dense)
  kRowResidual = 4,   // partial sums of |K u - d|^2
  kRowAdjCompact = 5, // zhat = F_row(M z_compact)
};

class FftPlanCache;

// Host-side owner of the mask compaction and FFT plans of one geometry.
struct CartPlan {
  CartGeom g{};
  std::vector<int> h_row_off, h_rows;
  void *d_tables = nullptr;  // row_off, rows, rowinfo, rowmap, twiddles, mrows
  double mask_norm2 = 0.0;  // ||mask||^2 (AdaptLambda)
  bool has_mask = false;

  CartPlan() = default;
  CartPlan(const CartPlan &) = delete;
  CartPlan &operator=(const CartPlan &) = delete;
  ~CartPlan();
  // mask: device pointer [T][H][W] or nullptr.
  void init(int W, int H, int C, int T, const float *mask, int centered, hipStream_t s);
  long kspace_elems() const { return g.nrows_c * (long)g.W; }
  int row_blocks() const { return (int)((g.nrows_c + g.RB - 1) / g.RB); }
};

// Column tiles of a geometry's two-stage passes.  Wide tiles keep every lane
// busy in both stages; narrow ones give more blocks.  The results do not depend
// on the choice.
void set_col_tiles(CartGeom &g, bool wide);
// Rows per block of a two-stage row pass: wide fills the lanes of both stages,
// narrow gives more blocks (and other partial sums).  One operator's calls take
// the narrow form below two wide blocks per CU, where the length of the chain
// counts (TV 128x128x12x8: 8.5 -> 6.5 us); the engine always the wide one (64
// such requests together: 113 -> 100 us).
void set_row_tiles(CartGeom &g, bool wide);
constexpr int kRowWideBlocks = 512;
// Blocks of a column pass on wide tiles, and the count from which wide tiles
// are taken: two blocks per CU.
long wide_col_blocks(const CartGeom &g);
constexpr long kColWideBlocks = 512;

// Coil groups of a forward column pass of `tiles` blocks (each block takes one
// group's coils; the results do not depend on it): enough for four blocks per
// CU.  Measured on MI355X (K, 1 group / this many): 180x240x20x12 (300 tiles)
// 58 -> 47 us, 192x192x20x10 45 -> 35, 160x160x12x8 28.5 -> 20, 128x128x12x8
// 25 -> 15; more groups than that re-read the image for nothing.
inline int col_coil_groups(long tiles, int C) {
  return (int)std::min<long>(C, std::max<long>(1, 1024 / std::max<long>(1, tiles)));
}

// Radices of a length-L transform and its twiddles (tw[m] = exp(-2 pi i m / L))
// on the host; make_fft_plan also uploads them.
void fft_plan_host(int L, FftPlan &p, std::vector<float2> &tw);
void make_fft_plan(int L, FftPlan &p, void **d_tw);

// ---- launchers (all asynchronous on `s`) ----
// Column pass of K: kcol = F^{-1}_y(b1 . (u - usub)) on the sampled rows.
void launch_col_forward(const CartGeom &g, const float2 *u, const float2 *usub, const float2 *b1,
                        float2 *kcol, hipStream_t s);
// Row pass (mode-dependent arguments may be null).
void launch_row_pass(int mode, const CartGeom &g, const float2 *kcol, float2 *z, const float2 *d,
                     float2 *zhat, float2 *out, const float2 *zin, const DevScalars *sc,
                     double *partial, hipStream_t s);
// Column pass of K^H with the coil sum: out = scale * sum_c conj(b1_c) F_y(zhat).
void launch_col_adjoint(const CartGeom &g, const float2 *zhat, const float2 *b1, float2 *out,
                        hipStream_t s);
// Gather dense [t][c][H][W] k-space rows into compact storage (times mask).
void launch_compact_gather(const CartGeom &g, const float2 *dense, float2 *compact, hipStream_t s);
// fft_io's kind (PlanKind) for B transforms of a plan per block of 256 lanes.
int plan_kind(const FftPlan &p, int B);
// Standalone batched 2D FFT (in place).
void launch_fft2(float2 *data, const FftPlan &pw, const FftPlan &ph, int H, int W, int batch,
                 int sign, int centered, float scale, hipStream_t s);
// In-place transform along the slowest axis of `batch` arrays [L][plane].
void launch_fft_axis0(float2 *data, const FftPlan &p, int L, int plane, int batch, int sign,
                      float scale, hipStream_t s);

}  // namespace avionic
