// Task-list kernels of the PD iteration (see tasks.hpp).  Each block finds
// its task, checks the task's device-side predicates (uniform per block, so a
// whole block returns together) and runs the shared block / voxel bodies.
#include <type_traits>

#include "reg_device.hpp"
#include "tasks_device.hpp"

namespace avionic {

// Dual and primal updates over the blocks of family F: kDp2 runs a pair of
// voxels of a row per lane (tasks of even width), kDp1 (tasks of odd width)
// and kVox (every task) one voxel per lane.
template <int F>
__device__ inline bool lane_voxels(const Task &T, int blk, Vox &v) {
  return vox_of_block<false>(T.g, blk - first_block<F>(T), threadIdx.x, v);
}
template <int F>
__device__ inline bool lane_voxels(const Task &T, int blk, Vox2 &v) {
  return vox2_of_block(T.g, blk - T.b_dp2, threadIdx.x, v);
}

template <int M, typename DT, int F>
__global__ __launch_bounds__(RT) void kt_dual(const Task *__restrict__ tasks, int n) {
  typedef typename std::conditional<F == kDp2, Vox2, Vox>::type V;
  const int blk = blockIdx.x;
  const Task &T = tasks[find_task<F>(tasks, n, blk)];
  if (!task_active(T.sc)) return;
  V v;
  if (!lane_voxels<F>(T, blk, v)) return;
  dual_voxel<M, DT>(T.g, T.rp, T.ext, (DT *)T.y, (float)T.sc->sigma, v);
}

template <int M, typename DT, int F>
__global__ __launch_bounds__(RT) void kt_primal(const Task *__restrict__ tasks, int n) {
  typedef typename std::conditional<F == kDp2, Vox2, Vox>::type V;
  const int blk = blockIdx.x;
  const Task &T = tasks[find_task<F>(tasks, n, blk)];
  if (!task_active(T.sc)) return;
  V v;
  if (!lane_voxels<F>(T, blk, v)) return;
  primal_voxel<M, DT>(T.g, T.rp, T.x, T.ext, (const DT *)T.y, T.khz, (float)T.sc->tau, v);
}

template <int M>
__global__ __launch_bounds__(RT) void kt_step_reg(const Task *__restrict__ tasks, int n) {
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const Task &T = tasks[find_task<kVox>(tasks, n, blk)];
  if (!task_active(T.sc) || !task_adapt(T.sc)) return;
  const int lb = blk - T.b_vox;
  Vox v;
  double ak = 0.0, ax = 0.0;
  if (vox_of_block<true>(T.g, lb, threadIdx.x, v)) step_voxel<M>(T.g, T.rp, T.ext, T.x, v, ak, ax);
  block_reduce2(ak, ax, T.part_reg + 2 * lb);
}

// One block per task: step rule for adapting tasks, then the iteration
// counter.  The reductions run in a fixed order (deterministic).
__global__ __launch_bounds__(RT) void kt_tail(const Task *__restrict__ tasks, int n) {
  const Task &T = tasks[blockIdx.x];
  DevScalars *sc = T.sc;
  if (!task_active(sc)) return;
  if (task_adapt(sc)) {
    __shared__ double ra[RT], rb[RT];
    const int tid = threadIdx.x;
    double a = 0.0, b = 0.0;
    for (int j = tid; j < T.nvox_blocks; j += RT) {
      a += T.part_reg[2 * j];
      b += T.part_reg[2 * j + 1];
    }
    for (int j = tid; j < T.npart_k; j += RT) a += T.part_k[j];
    ra[tid] = a;
    rb[tid] = b;
    __syncthreads();
    for (int s = RT / 2; s > 0; s >>= 1) {
      if (tid < s) {
        ra[tid] += ra[tid + s];
        rb[tid] += rb[tid + s];
      }
      __syncthreads();
    }
    if (tid == 0) {
      apply_step_rule(sc, ra[0], rb[0]);
      if (T.sig_log) T.sig_log[sc->iter] = sc->sigma;
      if (T.tau_log) T.tau_log[sc->iter] = sc->tau;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) sc->iter += 1;
}

const char *kernel_name(int id) {
  static const char *names[kNumKernels] = {"dual", "col_forward", "row_dual_update", "col_adjoint",
                                           "primal", "step_reg", "col_forward_delta",
                                           "row_norm2", "tail"};
  return (id >= 0 && id < kNumKernels) ? names[id] : "?";
}

// Dual (primal = false) or primal update over every task, in the grid's
// launch variant (TaskGrid::lanes).
template <int M, typename DT, int F>
static void launch_dp(bool primal, int nblk, hipStream_t s, const Task *t, int n) {
  if (primal)
    hipLaunchKernelGGL((kt_primal<M, DT, F>), dim3(nblk), dim3(RT), 0, s, t, n);
  else
    hipLaunchKernelGGL((kt_dual<M, DT, F>), dim3(nblk), dim3(RT), 0, s, t, n);
}
template <typename DT, int F>
static void launch_dp_m(int method, bool primal, int nblk, hipStream_t s, const Task *t, int n) {
  if (method == kTV) launch_dp<kTV, DT, F>(primal, nblk, s, t, n);
  else if (method == kTGV2) launch_dp<kTGV2, DT, F>(primal, nblk, s, t, n);
  else if (method == kICTGV2) launch_dp<kICTGV2, DT, F>(primal, nblk, s, t, n);
  else launch_dp<kICTV, DT, F>(primal, nblk, s, t, n);
}
template <int F>
static void launch_dp_v(int method, int ds, bool primal, int nblk, hipStream_t s, const Task *t,
                        int n) {
  if (ds == kDualF32) launch_dp_m<float2, F>(method, primal, nblk, s, t, n);
  else if (ds == kDualBF16) launch_dp_m<bf16x2, F>(method, primal, nblk, s, t, n);
  else launch_dp_m<q16x2, F>(method, primal, nblk, s, t, n);
}
static void launch_dual_primal(bool primal, int method, int ds, const TaskGrid &gr, hipStream_t s,
                               const Task *t, int n) {
  if (gr.lanes == 1) {
    if (gr.vox > 0) launch_dp_v<kVox>(method, ds, primal, gr.vox, s, t, n);
    return;
  }
  if (gr.dp2 > 0) launch_dp_v<kDp2>(method, ds, primal, gr.dp2, s, t, n);
  if (gr.dp1 > 0) launch_dp_v<kDp1>(method, ds, primal, gr.dp1, s, t, n);
}

void launch_kernel(int id, int method, int ds, const Task *d_tasks, int n, const TaskGrid &gr,
                   hipStream_t s) {
  if (n <= 0) return;
  const dim3 bRT(RT);
  switch (id) {
    case kKDual: launch_dual_primal(false, method, ds, gr, s, d_tasks, n); break;
    case kKColFwd: launch_task_col_forward(false, gr, d_tasks, n, s); break;
    case kKRowDual: launch_task_row(kRowDualUpdate, gr, d_tasks, n, s); break;
    case kKColAdj: launch_task_col_adjoint(gr, d_tasks, n, s); break;
    case kKPrimal: launch_dual_primal(true, method, ds, gr, s, d_tasks, n); break;
    case kKStepReg:
      if (gr.vox) {
        if (method == kTV) hipLaunchKernelGGL(kt_step_reg<kTV>, dim3(gr.vox), bRT, 0, s, d_tasks, n);
        else if (method == kTGV2) hipLaunchKernelGGL(kt_step_reg<kTGV2>, dim3(gr.vox), bRT, 0, s, d_tasks, n);
        else if (method == kICTGV2) hipLaunchKernelGGL(kt_step_reg<kICTGV2>, dim3(gr.vox), bRT, 0, s, d_tasks, n);
        else hipLaunchKernelGGL(kt_step_reg<kICTV>, dim3(gr.vox), bRT, 0, s, d_tasks, n);
      }
      break;
    case kKColFwdDelta: launch_task_col_forward(true, gr, d_tasks, n, s); break;
    case kKRowNorm2: launch_task_row(kRowNorm2, gr, d_tasks, n, s); break;
    case kKTail: hipLaunchKernelGGL(kt_tail, dim3(n), bRT, 0, s, d_tasks, n); break;
    default: break;
  }
  AV_LAUNCH_CHECK();
}

void launch_iteration(int method, int ds, const Task *d_tasks, int n, const TaskGrid &gr,
                      bool with_step, const IterStreams &st, const IterHooks &hooks) {
  if (n <= 0) return;
  hipStream_t s = st.main;
  const bool two = st.side != nullptr;
  hipStream_t s2 = two ? st.side : st.main;
  auto fork = [&]() {
    if (!two) return;
    AV_HIP(hipEventRecord(st.fork, s));
    AV_HIP(hipStreamWaitEvent(s2, st.fork, 0));
  };
  auto join = [&]() {
    if (!two) return;
    AV_HIP(hipEventRecord(st.join, s2));
    AV_HIP(hipStreamWaitEvent(s, st.join, 0));
  };
  const dim3 bRT(RT);
  // dual update (reads ext, writes y) beside the data-term chain (reads ext,
  // writes kcol / z / zhat / khz); the primal update needs both
  if (two && gr.col_first) {
    // Submitted first, the column pass's workgroups start and the dual fills the
    // rest of the CUs; the dual still depends only on what precedes the column
    // pass.  Measured on MI355X, dual first against this order on the same
    // buffers: 768 column workgroups (16 TV 128x128x12x8) +6% from replayed
    // graphs, +12% eagerly; 19 sets of 1536 to 12288 workgroups -1.5 to +1.2%
    // (mean 0) from graphs, 0 to +1.8% eagerly.
    AV_HIP(hipEventRecord(st.fork, s));
    launch_task_col_forward(false, gr, d_tasks, n, s);
    AV_HIP(hipStreamWaitEvent(s2, st.fork, 0));
    launch_dual_primal(false, method, ds, gr, s2, d_tasks, n);
  } else {
    fork();
    launch_dual_primal(false, method, ds, gr, s2, d_tasks, n);
    launch_task_col_forward(false, gr, d_tasks, n, s);
  }
  AV_LAUNCH_CHECK();
  launch_task_row(kRowDualUpdate, gr, d_tasks, n, s);
  launch_task_col_adjoint(gr, d_tasks, n, s);
  AV_LAUNCH_CHECK();
  if (hooks.fn) hooks.fn(hooks.ctx, 0, s);
  join();
  launch_dual_primal(true, method, ds, gr, s, d_tasks, n);
  AV_LAUNCH_CHECK();
  if (with_step) {
    // regulariser sums (read ext, x) beside K(ext - x); the tail needs both
    fork();
    if (gr.vox > 0) {
      if (method == kTV) hipLaunchKernelGGL(kt_step_reg<kTV>, dim3(gr.vox), bRT, 0, s2, d_tasks, n);
      else if (method == kTGV2) hipLaunchKernelGGL(kt_step_reg<kTGV2>, dim3(gr.vox), bRT, 0, s2, d_tasks, n);
      else if (method == kICTGV2) hipLaunchKernelGGL(kt_step_reg<kICTGV2>, dim3(gr.vox), bRT, 0, s2, d_tasks, n);
      else hipLaunchKernelGGL(kt_step_reg<kICTV>, dim3(gr.vox), bRT, 0, s2, d_tasks, n);
    }
    AV_LAUNCH_CHECK();
    launch_task_col_forward(true, gr, d_tasks, n, s);
    launch_task_row(kRowNorm2, gr, d_tasks, n, s);
    AV_LAUNCH_CHECK();
    if (hooks.fn) hooks.fn(hooks.ctx, 1, s);
    join();
  }
  hipLaunchKernelGGL(kt_tail, dim3(n), bRT, 0, s, d_tasks, n);
  AV_LAUNCH_CHECK();
}

}  // namespace avionic
