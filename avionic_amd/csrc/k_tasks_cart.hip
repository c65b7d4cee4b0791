// Task-list column and row passes of the Cartesian operator (tasks.hpp).
//
// One kernel per kind of plan (ColKind, RowKind); a launch covers its kind's
// span of blocks and is made only when such a task is resident.  DELTA =
// false: K of the extragradient image (dual update); DELTA = true: K of
// ext - x (step rule, adapting tasks only).  The forward column pass of a
// small launch set splits each task's coils into `groups` blocks per tile.
#include "cart_two.hpp"
#include "tasks_device.hpp"

namespace avionic {

template <bool DELTA, int KIND>
__global__ __launch_bounds__(NTC) void kt_col_forward(const Task *__restrict__ tasks, int n,
                                                      int blk0, int groups) {
  __shared__ float2 tile[KIND & 1 ? kColTwoElems : kColTileElems];
  __shared__ float2 twl[col_table_len(KIND)];
  __shared__ int rml[col_table_len(KIND)];
  const int blk = blk0 + (int)blockIdx.x;
  const Task &T = tasks[find_task<kCol>(tasks, n, blk)];
  if (T.cg.ckind != KIND) return;
  if (!task_active(T.sc)) return;
  if (DELTA && !task_adapt(T.sc)) return;
  const int lb = blk - T.b_col, xbi = lb % T.cg.nxb, t = lb / T.cg.nxb;
  const int cpg = (T.cg.C + groups - 1) / groups, c0 = (int)blockIdx.y * cpg;
  const int c1 = min(T.cg.C, c0 + cpg);
  const float2 *usub = DELTA ? T.x : nullptr;
  if constexpr (KIND == 1)
    col_forward_two<DELTA, TwoRt>(T.cg, xbi, t, c0, c1, T.ext, usub, T.b1, T.kcol, tile, twl, rml);
  else if constexpr (KIND == 3)
    col_forward_two<DELTA, Two256>(T.cg, xbi, t, c0, c1, T.ext, usub, T.b1, T.kcol, tile, twl, rml);
  else
    col_forward_fused<DELTA, KIND == 2>(T.cg, xbi, t, c0, c1, T.ext, usub, T.b1, T.kcol, tile,
                                        twl, rml);
}

// A lane holds the values of its butterflies with z and d beside them: 175 VGPRs,
// two waves per SIMD.  kRowTwo is held to three waves (168 VGPRs, a little of the
// largest radices spilled); at 16 x 16 the spill costs more than the wave, so
// length 256 has its own kernel of the same source (and bits).  Measured on
// MI355X, without the bound / with it: 64 TV 128x128x12x8 123 -> 119 us (the
// compile-time pass for 128 before: 114), 64 TV 96x96x8x6 50 -> 44, 32 TV
// 160x128x12x8 77 -> 68, 16 TGV2 192x160x16x8 69 -> 62, 16 TV 240x128x12x8
// 55 -> 51; 8 ICTGV2 256x256x30x16 168 -> 176.
template <int MODE, int RK>
__global__ __launch_bounds__(NT, RK == kRowTwo ? 3 : 1) void kt_row(const Task *__restrict__ tasks,
                                                                    int n, int blk0) {
  constexpr bool TWO = RK == kRowTwo || RK == kRow256;
  __shared__ float2 tile[TWO ? kRowTwoElems : RTILE];
  __shared__ float2 tile2[(MODE == kRowDualUpdate && !TWO) ? RTILE : 1];
  __shared__ float2 twl[row_table_len(RK)];
  __shared__ double red[MODE == kRowNorm2 ? NT : 1];
  __shared__ int mrl[TWO ? 1 : kRowMaxRows];
  const int blk = blk0 + (int)blockIdx.x;
  const Task &T = tasks[find_task<kRow>(tasks, n, blk)];
  if (T.cg.rkind != RK) return;
  if (!task_active(T.sc)) return;
  if (MODE == kRowNorm2 && !task_adapt(T.sc)) return;
  const int lb = blk - T.b_row;
  double a = 0.0;
  if constexpr (TWO)
    a = row_two<MODE>(T.cg, lb, T.kcol, T.z, T.d, T.zhat, nullptr, nullptr, T.sc, tile, twl);
  else if constexpr (MODE == kRowDualUpdate)
    row_dual_fused<RK == kRowWide>(T.cg, lb, T.kcol, T.z, T.d, T.zhat, T.sc, tile, tile2, twl, mrl);
  else
    a = row_mode_fused<MODE, RK == kRowWide>(T.cg, lb, T.kcol, nullptr, nullptr, nullptr, nullptr,
                                             tile, twl, mrl);
  if (MODE == kRowNorm2) {
    a = block_sum(a, red);
    if (threadIdx.x == 0) T.part_k[lb] = a;
  }
}

// Held to 4 waves per SIMD (the limit the LDS tile sets anyway): the two-stage
// forms spill a little at 128 VGPRs, which with more blocks than the CUs hold
// costs less than a wave (8 x ICTGV2 256x256x30x16 351 -> 340 us, 4 x TGV2
// 160x144x20x12 65 -> 49 us; one reconstruction 57.5 -> 60.8 us).
template <int KIND>
__global__ __launch_bounds__(NTC) __attribute__((amdgpu_waves_per_eu(4)))
void kt_col_adjoint(const Task *__restrict__ tasks, int n, int blk0) {
  __shared__ float2 tile[KIND & 1 ? kColTwoElems : kColTileElems];
  __shared__ float2 twl[col_table_len(KIND)];
  __shared__ int rml[col_table_len(KIND)];
  const int blk = blk0 + (int)blockIdx.x;
  const Task &T = tasks[find_task<kCol>(tasks, n, blk)];
  if (T.cg.ckind != KIND) return;
  if (!task_active(T.sc)) return;
  const int lb = blk - T.b_col, xbi = lb % T.cg.nxb, t = lb / T.cg.nxb;
  if constexpr (KIND == 1)
    col_adjoint_two<TwoRt, 1>(T.cg, xbi, t, T.zhat, T.b1, T.khz, tile, 0, twl, rml);
  else if constexpr (KIND == 3)
    col_adjoint_two<Two256, 1>(T.cg, xbi, t, T.zhat, T.b1, T.khz, tile, 0, twl, rml);
  else
    col_adjoint_fused<KIND == 2>(T.cg, xbi, t, T.zhat, T.b1, T.khz, tile, twl, rml);
}

template <bool DELTA, int K = 0>
static void col_fwd(const TaskGrid &gr, const Task *d_tasks, int n, hipStream_t s) {
  if constexpr (K < kColKinds) {
    const int nb = gr.col_hi[K] - gr.col_lo[K];
    if (nb > 0)
      hipLaunchKernelGGL((kt_col_forward<DELTA, K>), dim3(nb, gr.col_groups), dim3(NTC), 0, s, d_tasks, n,
                         gr.col_lo[K], gr.col_groups);
    col_fwd<DELTA, K + 1>(gr, d_tasks, n, s);
  }
}
void launch_task_col_forward(bool delta, const TaskGrid &gr, const Task *d_tasks, int n,
                             hipStream_t s) {
  if (delta)
    col_fwd<true>(gr, d_tasks, n, s);
  else
    col_fwd<false>(gr, d_tasks, n, s);
  AV_LAUNCH_CHECK();
}

template <int K = 0>
static void col_adj(const TaskGrid &gr, const Task *d_tasks, int n, hipStream_t s) {
  if constexpr (K < kColKinds) {
    const int nb = gr.col_hi[K] - gr.col_lo[K];
    if (nb > 0)
      hipLaunchKernelGGL((kt_col_adjoint<K>), dim3(nb), dim3(NTC), 0, s, d_tasks, n, gr.col_lo[K]);
    col_adj<K + 1>(gr, d_tasks, n, s);
  }
}
void launch_task_col_adjoint(const TaskGrid &gr, const Task *d_tasks, int n, hipStream_t s) {
  col_adj(gr, d_tasks, n, s);
  AV_LAUNCH_CHECK();
}

template <int MODE, int RK = 0>
static void row(const TaskGrid &gr, const Task *d_tasks, int n, hipStream_t s) {
  if constexpr (RK < kRowKinds) {
    const int nb = gr.row_hi[RK] - gr.row_lo[RK];
    if (nb > 0)
      hipLaunchKernelGGL((kt_row<MODE, RK>), dim3(nb), dim3(NT), 0, s, d_tasks, n, gr.row_lo[RK]);
    row<MODE, RK + 1>(gr, d_tasks, n, s);
  }
}
void launch_task_row(int mode, const TaskGrid &gr, const Task *d_tasks, int n, hipStream_t s) {
  if (mode == kRowDualUpdate)
    row<kRowDualUpdate>(gr, d_tasks, n, s);
  else
    row<kRowNorm2>(gr, d_tasks, n, s);
  AV_LAUNCH_CHECK();
}

}  // namespace avionic
