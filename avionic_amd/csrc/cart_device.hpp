// Device-side helpers shared by the Cartesian operator passes (cart_two.hpp,
// cart_fused.hpp).
#pragma once

#include "cartesian.hpp"
#include "fft_device.hpp"

namespace avionic {

constexpr int NT = kFftThreads;
constexpr int EMAX = kFftTileElems;

// (i + n/2) mod n and (a + b) mod n for 0 <= i, a < n, 0 <= b <= n, without a
// division.
__device__ __forceinline__ int wrap_half(int i, int n) {
  const int v = i + n / 2;
  return v >= n ? v - n : v;
}
__device__ __forceinline__ int wrap_add(int a, int b, int n) {
  const int v = a + b;
  return v >= n ? v - n : v;
}

// Block sum of one value per lane (NT lanes) in a fixed order, in lane 0.
__device__ inline double block_sum(double v, double *red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int s = NT / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  return red[0];
}

}  // namespace avionic
