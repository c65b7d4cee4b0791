// Task lookup and predicates shared by the task-list kernels (k_tasks.hip,
// k_tasks_cart.hip).
#pragma once

#include "tasks.hpp"

namespace avionic {

enum Family { kVox = 0, kCol = 1, kRow = 2, kDp1 = 3, kDp2 = 4 };

template <int F>
__device__ inline int first_block(const Task &t) {
  switch (F) {
    case kVox: return t.b_vox;
    case kCol: return t.b_col;
    case kRow: return t.b_row;
    case kDp1: return t.b_dp1;
    default: return t.b_dp2;
  }
}

// Last task whose first block does not exceed b (tasks are in block order;
// a task with no blocks in this family shares its start with the next one):
// a binary search over the non-decreasing first blocks.
template <int F>
__device__ inline int find_task(const Task *__restrict__ tasks, int n, int b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first_block<F>(tasks[mid]) <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// Renumbering blocks so that every XCD walks one contiguous range keeps the
// neighbouring frames that the step-rule reduction reads in one XCD's L2 (a
// bijection on [0, n)).  Measured on MI355X it helps that kernel and slows
// the streaming dual / primal updates, which keep the hardware order.
__device__ inline int xcd_block(int b, int n) {
  constexpr int X = 8;
  const int q = n / X, r = n % X;
  const int x = b % X, k = b / X;
  return x * q + min(x, r) + k;
}

__device__ inline bool task_active(const DevScalars *sc) { return sc->iter < sc->maxit; }
__device__ inline bool task_adapt(const DevScalars *sc) {
  const int k = sc->iter;
  return sc->schedule == 1 || (sc->schedule == 0 && (k < 10 || (k % 50) == 0));
}

}  // namespace avionic
