// Column passes of the Cartesian operator for one operator's calls (K, K^H,
// norms, the eager solver); the block bodies are in cart_two.hpp and
// cart_fused.hpp.
#include <algorithm>

#include "cart_two.hpp"

namespace avionic {

// Block (tile, frame, coil group): coils [z cpg, (z + 1) cpg).
template <bool DELTA, int KIND>
__global__ __launch_bounds__(NT) void k_col_forward(CartGeom g, int cpg,
                                                    const float2 *__restrict__ u,
                                                    const float2 *__restrict__ usub,
                                                    const float2 *__restrict__ b1,
                                                    float2 *__restrict__ kcol) {
  __shared__ float2 tile[KIND & 1 ? kColTwoElems : kColTileElems];
  __shared__ float2 twl[col_table_len(KIND)];
  __shared__ int rml[col_table_len(KIND)];
  const int xbi = blockIdx.x, t = blockIdx.y, c0 = blockIdx.z * cpg, c1 = min(g.C, c0 + cpg);
  if constexpr (KIND == 1)
    col_forward_two<DELTA, TwoRt>(g, xbi, t, c0, c1, u, usub, b1, kcol, tile, twl, rml);
  else if constexpr (KIND == 3)
    col_forward_two<DELTA, Two256>(g, xbi, t, c0, c1, u, usub, b1, kcol, tile, twl, rml);
  else
    col_forward_fused<DELTA, KIND == 2>(g, xbi, t, c0, c1, u, usub, b1, kcol, tile, twl, rml);
}

// Runtime plans.
template <bool WIDE>
__global__ __launch_bounds__(NT) void k_col_adjoint_rt(CartGeom g, const float2 *__restrict__ zhat,
                                                       const float2 *__restrict__ b1,
                                                       float2 *__restrict__ out) {
  constexpr int KIND = WIDE ? 2 : 0;
  __shared__ float2 tile[kColTileElems];
  __shared__ float2 twl[col_table_len(KIND)];
  __shared__ int rml[col_table_len(KIND)];
  col_adjoint_fused<WIDE>(g, blockIdx.x, blockIdx.y, zhat, b1, out, tile, twl, rml);
}

// Two-stage: G groups of NT lanes share the block's coils, with a tile of
// `elems` each in the dynamic LDS.
template <class P, int G>
__global__ __launch_bounds__(NT * G) void k_col_adjoint(CartGeom g, int elems,
                                                        const float2 *__restrict__ zhat,
                                                        const float2 *__restrict__ b1,
                                                        float2 *__restrict__ out) {
  extern __shared__ float2 tiles[];
  __shared__ float2 twl[kTwoMaxLen];
  __shared__ int rml[kTwoMaxLen];
  col_adjoint_two<P, G>(g, blockIdx.x, blockIdx.y, zhat, b1, out, tiles, elems, twl, rml);
}

template <bool DELTA, int K = 0>
static void col_fwd(int kind, const CartGeom &g, const float2 *u, const float2 *usub,
                    const float2 *b1, float2 *kcol, hipStream_t s) {
  if constexpr (K < kColKinds) {
    if (kind != K) return col_fwd<DELTA, K + 1>(kind, g, u, usub, b1, kcol, s);
    const int groups = col_coil_groups((long)g.nxb * g.T, g.C);
    const int cpg = (g.C + groups - 1) / groups;
    hipLaunchKernelGGL((k_col_forward<DELTA, K>), dim3(g.nxb, g.T, (g.C + cpg - 1) / cpg), dim3(NT),
                       0, s, g, cpg, u, usub, b1, kcol);
    AV_LAUNCH_CHECK();
  }
}

void launch_col_forward(const CartGeom &g, const float2 *u, const float2 *usub, const float2 *b1,
                        float2 *kcol, hipStream_t s) {
  if (usub)
    col_fwd<true>(g.ckind, g, u, usub, b1, kcol, s);
  else
    col_fwd<false>(g.ckind, g, u, usub, b1, kcol, s);
}

template <class P, int G>
static void col_adj(const CartGeom &g, const float2 *zhat, const float2 *b1, float2 *out,
                    hipStream_t s) {
  const int elems = g.ph.rb * (g.ph.ra + 1) * g.XB;
  hipLaunchKernelGGL((k_col_adjoint<P, G>), dim3(g.nxb, g.T), dim3(NT * G),
                     sizeof(float2) * elems * G, s, g, elems, zhat, b1, out);
}
// Up to 5 tiles for 4 CUs each CU's one or two blocks run the chain of coils
// with little else to fill the waits: four groups of lanes then share it.
// Measured on MI355X (K^H, 1 / 2 / 4 groups): 180x240x20x12 (300 tiles) 53 / 42
// / 36 us, 192x192x20x10 (240) 38 / 31 / 29, 160x160x12x8 (120) 28 / 22 / 19.5;
// 256x256x25x12 (400) 47.5 / 48 / 52, 256x256x30x16 (480) 59.5 / 59 / 65.
constexpr long kAdjGroupTiles = 320;
template <class P>
static void col_adj_groups(const CartGeom &g, const float2 *zhat, const float2 *b1, float2 *out,
                           hipStream_t s) {
  if ((long)g.nxb * g.T > kAdjGroupTiles || g.C < 2)
    col_adj<P, 1>(g, zhat, b1, out, s);
  else if (g.C < 4)
    col_adj<P, 2>(g, zhat, b1, out, s);
  else
    col_adj<P, 4>(g, zhat, b1, out, s);
}

void launch_col_adjoint(const CartGeom &g, const float2 *zhat, const float2 *b1, float2 *out,
                        hipStream_t s) {
  const dim3 grid(g.nxb, g.T), block(NT);
  switch (g.ckind) {
    case 0: hipLaunchKernelGGL(k_col_adjoint_rt<false>, grid, block, 0, s, g, zhat, b1, out); break;
    case 2: hipLaunchKernelGGL(k_col_adjoint_rt<true>, grid, block, 0, s, g, zhat, b1, out); break;
    case 1: col_adj_groups<TwoRt>(g, zhat, b1, out, s); break;
    default: col_adj_groups<Two256>(g, zhat, b1, out, s); break;
  }
  AV_LAUNCH_CHECK();
}

}  // namespace avionic
