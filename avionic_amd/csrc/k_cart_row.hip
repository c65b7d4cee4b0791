// Row passes of the Cartesian operator for one operator's calls (K, K^H,
// norms, the eager solver); the block bodies are in cart_two.hpp and
// cart_fused.hpp.
#include "cart_two.hpp"

namespace avionic {

template <int MODE, int KIND>
__global__ __launch_bounds__(NT) void k_row_pass(CartGeom g, const float2 *__restrict__ kcol,
                                                 float2 *__restrict__ z,
                                                 const float2 *__restrict__ d,
                                                 float2 *__restrict__ zhat,
                                                 float2 *__restrict__ out,
                                                 const float2 *__restrict__ zin,
                                                 const DevScalars *__restrict__ sc,
                                                 double *__restrict__ partial) {
  constexpr bool SUM = MODE == kRowNorm2 || MODE == kRowResidual;
  constexpr bool DUAL = MODE == kRowDualUpdate;
  __shared__ float2 tile[KIND == 0 ? kRowTwoElems : RTILE];
  __shared__ float2 tile2[DUAL && KIND != 0 ? RTILE : 1];
  __shared__ float2 twl[row_table_len(KIND)];
  __shared__ int mrl[KIND == 0 ? 1 : kRowMaxRows];
  __shared__ double red[SUM ? NT : 1];
  double a = 0.0;
  if constexpr (KIND == 0)
    a = row_two<MODE>(g, blockIdx.x, kcol, z, d, zhat, out, zin, sc, tile, twl);
  else if constexpr (DUAL)
    row_dual_fused<KIND == 2>(g, blockIdx.x, kcol, z, d, zhat, sc, tile, tile2, twl, mrl);
  else
    a = row_mode_fused<MODE, KIND == 2>(g, blockIdx.x, kcol, d, zhat, out, zin, tile, twl,
                                              mrl);
  if (SUM) {
    a = block_sum(a, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = a;
  }
}

template <int MODE>
static void launch_row_kind(const CartGeom &g, int nb, const float2 *kcol, float2 *z,
                            const float2 *d, float2 *zhat, float2 *out, const float2 *zin,
                            const DevScalars *sc, double *partial, hipStream_t s) {
  const dim3 grid(nb), block(NT);
  switch (g.rkind) {
    case kRowTwo:
    case kRow256: hipLaunchKernelGGL((k_row_pass<MODE, 0>), grid, block, 0, s, g, kcol, z, d, zhat, out, zin, sc, partial); break;
    case kRowRt: hipLaunchKernelGGL((k_row_pass<MODE, 1>), grid, block, 0, s, g, kcol, z, d, zhat, out, zin, sc, partial); break;
    default: hipLaunchKernelGGL((k_row_pass<MODE, 2>), grid, block, 0, s, g, kcol, z, d, zhat, out, zin, sc, partial); break;
  }
}

void launch_row_pass(int mode, const CartGeom &g, const float2 *kcol, float2 *z, const float2 *d,
                     float2 *zhat, float2 *out, const float2 *zin, const DevScalars *sc,
                     double *partial, hipStream_t s) {
  const int nb = (int)((g.nrows_c + g.RB - 1) / g.RB);
  if (nb == 0) return;
  switch (mode) {
    case kRowApplyK: launch_row_kind<kRowApplyK>(g, nb, kcol, z, d, zhat, out, zin, sc, partial, s); break;
    case kRowDualUpdate: launch_row_kind<kRowDualUpdate>(g, nb, kcol, z, d, zhat, out, zin, sc, partial, s); break;
    case kRowNorm2: launch_row_kind<kRowNorm2>(g, nb, kcol, z, d, zhat, out, zin, sc, partial, s); break;
    case kRowAdjDense: launch_row_kind<kRowAdjDense>(g, nb, kcol, z, d, zhat, out, zin, sc, partial, s); break;
    case kRowResidual: launch_row_kind<kRowResidual>(g, nb, kcol, z, d, zhat, out, zin, sc, partial, s); break;
    case kRowAdjCompact: launch_row_kind<kRowAdjCompact>(g, nb, kcol, z, d, zhat, out, zin, sc, partial, s); break;
    default: AV_CHECK(false, "bad row-pass mode");
  }
  AV_LAUNCH_CHECK();
}

}  // namespace avionic
