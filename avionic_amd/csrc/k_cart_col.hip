// Column passes of the Cartesian operator for one operator's calls (K, K^H,
// norms, the eager solver); the block bodies are in cart_two.hpp and
// cart_fused.hpp.
#include "cart_two.hpp"

namespace avionic {

template <bool DELTA, int KIND>
__global__ __launch_bounds__(NT) void k_col_forward(CartGeom g, const float2 *__restrict__ u,
                                                    const float2 *__restrict__ usub,
                                                    const float2 *__restrict__ b1,
                                                    float2 *__restrict__ kcol) {
  __shared__ float2 tile[KIND & 1 ? kColTwoElems : kColTileElems];
  __shared__ float2 twl[col_table_len(KIND)];
  __shared__ int rml[col_table_len(KIND)];
  if constexpr (KIND == 1)
    col_forward_two<DELTA, TwoRt>(g, blockIdx.x, blockIdx.y, 0, g.C, u, usub, b1, kcol, tile, twl, rml);
  else if constexpr (KIND == 3)
    col_forward_two<DELTA, Two256>(g, blockIdx.x, blockIdx.y, 0, g.C, u, usub, b1, kcol, tile, twl, rml);
  else
    col_forward_fused<DELTA, KIND == 2>(g, blockIdx.x, blockIdx.y, 0, g.C, u,
                                                          usub, b1, kcol, tile, twl, rml);
}

template <int KIND>
__global__ __launch_bounds__(NT) void k_col_adjoint(CartGeom g, const float2 *__restrict__ zhat,
                                                    const float2 *__restrict__ b1,
                                                    float2 *__restrict__ out) {
  __shared__ float2 tile[KIND & 1 ? kColTwoElems : kColTileElems];
  __shared__ float2 twl[col_table_len(KIND)];
  __shared__ int rml[col_table_len(KIND)];
  if constexpr (KIND == 1)
    col_adjoint_two<TwoRt>(g, blockIdx.x, blockIdx.y, zhat, b1, out, tile, twl, rml);
  else if constexpr (KIND == 3)
    col_adjoint_two<Two256>(g, blockIdx.x, blockIdx.y, zhat, b1, out, tile, twl, rml);
  else
    col_adjoint_fused<KIND == 2>(g, blockIdx.x, blockIdx.y, zhat, b1, out, tile,
                                                   twl, rml);
}

template <bool DELTA>
static void launch_col_fwd_kind(const CartGeom &g, const float2 *u, const float2 *usub,
                                const float2 *b1, float2 *kcol, hipStream_t s) {
  const dim3 grid(g.nxb, g.T), block(NT);
  switch (col_kind(g)) {
    case 1: hipLaunchKernelGGL((k_col_forward<DELTA, 1>), grid, block, 0, s, g, u, usub, b1, kcol); break;
    case 0: hipLaunchKernelGGL((k_col_forward<DELTA, 0>), grid, block, 0, s, g, u, usub, b1, kcol); break;
    case 3: hipLaunchKernelGGL((k_col_forward<DELTA, 3>), grid, block, 0, s, g, u, usub, b1, kcol); break;
    default: hipLaunchKernelGGL((k_col_forward<DELTA, 2>), grid, block, 0, s, g, u, usub, b1, kcol); break;
  }
  AV_LAUNCH_CHECK();
}

void launch_col_forward(const CartGeom &g, const float2 *u, const float2 *usub, const float2 *b1,
                        float2 *kcol, hipStream_t s) {
  if (usub)
    launch_col_fwd_kind<true>(g, u, usub, b1, kcol, s);
  else
    launch_col_fwd_kind<false>(g, u, usub, b1, kcol, s);
}

void launch_col_adjoint(const CartGeom &g, const float2 *zhat, const float2 *b1, float2 *out,
                        hipStream_t s) {
  const dim3 grid(g.nxb, g.T), block(NT);
  switch (col_kind(g)) {
    case 1: hipLaunchKernelGGL((k_col_adjoint<1>), grid, block, 0, s, g, zhat, b1, out); break;
    case 0: hipLaunchKernelGGL((k_col_adjoint<0>), grid, block, 0, s, g, zhat, b1, out); break;
    case 3: hipLaunchKernelGGL((k_col_adjoint<3>), grid, block, 0, s, g, zhat, b1, out); break;
    default: hipLaunchKernelGGL((k_col_adjoint<2>), grid, block, 0, s, g, zhat, b1, out); break;
  }
  AV_LAUNCH_CHECK();
}

}  // namespace avionic
