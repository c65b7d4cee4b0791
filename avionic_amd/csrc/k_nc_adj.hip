// Kaiser-Bessel gridding, K^H (noncart.hpp): column and row passes.
#include "nc_device.hpp"

namespace avionic {

namespace {

// --------------------------------------------------------- K^H, column pass
struct NcColAdjStore {
  float2 *tp;  // tmp of the plane: [H][Gx]
  int H, Gx, Gy, gx0;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int gx = gx0 + b;
    if (gx >= Gx) return;
    const int y = wrap_up(i + H / 2, Gy);
    if (y < H) tp[(unsigned)(y * Gx + gx)] = v;
  }
};

// Spreading by gathers, balanced over the lanes: a block takes its column
// tile's entries (NcGeom::tce, in cell order) in chunks; the lanes form the
// products z[m] w of a chunk, each lane NCC apart (their index and z loads
// issued together), into the LDS tile; then every cell sums the products of
// its own entries in entry order from LDS.  Dense cells at the k-space
// centre (a hundred entries) then cost LDS reads, not a chain of dependent
// global loads on one lane.  The sums keep each cell's entry order, so every
// application gives the same bits.
// NZ coils of a frame per block (3 in the compiled kernels, 2 at grid length 512;
// 2 and 4 measured slower than 3 at the 256x256x30x12 radial geometry;
// nc_adj_coils on runtime plans): the tile's offsets are
// staged and its entries loaded once for all of them, each entry's products
// of the NZ coils sit in NZ parts of the tile, and the transforms run one
// after the other.  Every coil's sums are the one-coil
// sums.  (Running a block over all coils of a frame, one after the other,
// measured slower: 0.43 against 0.37 ms at the 256x256x30x12 radial
// geometry.)
template <int WIDE, class PL, int NZ>
__global__ __launch_bounds__(NCC) void k_nc_col_adj(NcGeom g, const float2 *__restrict__ z,
                                                    float2 *__restrict__ tmp) {
  constexpr int CPL = NCE / NCC;  // cells per lane (XBa Gy <= NCE)
  constexpr int U = 4;            // products per lane issued together
  constexpr int CH = NCE / NZ;    // entries per chunk
  __shared__ float2 tile[NCE];
  __shared__ float2 twl[nc_table_len(WIDE)];
  extern __shared__ int cps[];  // XBa * Gy + 1 ints, sized at launch
  const int tid = threadIdx.x;
  const int ngrp = (g.C + NZ - 1) / NZ;  // coil groups per frame
  const int t = blockIdx.y / ngrp, cz = (blockIdx.y % ngrp) * NZ;
  const int nz = min(NZ, g.C - cz);  // coils of this block
  const int X = blockIdx.x, nX = gridDim.x;
  const float2 *tw = stage_twiddles(g.py, twl, tid, NCC);
  constexpr bool CT = PL::L != 0;
  const int XB = CT ? PL::XB : g.XBa, ncell = XB * (CT ? PL::L : g.Gy);
  const int *tc = g.tcell + ((long)t * nX + X) * (ncell + 1);
  for (int k = tid; k <= ncell; k += NCC) cps[k] = tc[k];
  const int2 *ent = g.tce + g.tstart[t * nX + X];
  const float2 *zp = z + ((long)t * g.C + cz) * g.M;  // coil cz + q at zp + q M
  __syncthreads();
  const int E = cps[ncell];
  float2 acc[NZ][CPL];
#pragma unroll
  for (int q = 0; q < NZ; ++q)
#pragma unroll
    for (int j = 0; j < CPL; ++j) acc[q][j] = czero();
  for (int c0 = 0; c0 < E; c0 += CH) {
    const int n = min(CH, E - c0);
    for (int e0 = 0; e0 < n; e0 += U * NCC) {
      int2 mw[U];
      float2 zv[NZ][U];
#pragma unroll
      for (int u = 0; u < U; ++u) mw[u] = ent[c0 + min(e0 + u * NCC + tid, n - 1)];
#pragma unroll
      for (int q = 0; q < NZ; ++q)
#pragma unroll
        for (int u = 0; u < U; ++u) zv[q][u] = zp[(long)(q < nz ? q : 0) * g.M + mw[u].x];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * NCC + tid;
        if (e < n)
#pragma unroll
          for (int q = 0; q < NZ; ++q) tile[q * CH + e] = cscale(zv[q][u], __int_as_float(mw[u].y));
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int k = tid + j * NCC;
      if (k < ncell) {
        const int e1 = min(cps[k + 1], c0 + n);
        for (int e = max(cps[k], c0); e < e1; ++e)
#pragma unroll
          for (int q = 0; q < NZ; ++q) acc[q][j] = cadd(acc[q][j], tile[q * CH + e - c0]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < NZ; ++q) {
    if (q >= nz) break;  // uniform over the block
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int k = tid + j * NCC;
      if (k < ncell) tile[k] = acc[q][j];
    }
    __syncthreads();
    NcColAdjStore st{tmp + ((long)t * g.C + cz + q) * g.H * g.Gx, g.H, CT ? PL::L : g.Gx,
                     CT ? PL::L : g.Gy, X * XB};
    NoLoad nl;
    if constexpr (CT)
      fft_io_ct<NCC, PL, PL::XB, true, false, true>(tile, PL::XB, 1, PL::XB, +1.f, tid,
                                                       tw, nl, st);
    else
      fft_io<NCC, NCE, true, false, true, WIDE>(tile, g.py, XB, 1, XB, +1.f, tid, tw, nl, st);
    __syncthreads();  // every lane has read the tile before the next coil writes it
  }
}

// ------------------------------------------------------------ K^H, row pass
struct NcRowAdjLoad {
  const float2 *tr;  // tmp rows y0.. of plane (t, c)
  int Gx;
  __device__ float2 operator()(int b, int i, int) const { return tr[(unsigned)(b * Gx + i)]; }
};
template <int SLOTS>
struct NcRowAdjStore {
  float2 acc[SLOTS];
  const float2 *bc;
  float2 *img;  // frame t
  const float *dxi, *dyi;
  int W, Gx, y0;
  bool last;
  __device__ void operator()(int b, int i, float2 v, int slot) {
    const int x = wrap_up(i + W / 2, Gx);
    if (x >= W) return;
    const int y = y0 + b;
    const unsigned o = (unsigned)(y * W + x);
    const float2 a = cadd(acc[slot], cmulc(bc[o], v));
    if (last)
      img[o] = cscale(a, dxi[x] * dyi[y]);
    else
      acc[slot] = a;
  }
};

template <int WIDE, class PL>
__global__ __launch_bounds__(NCR) void k_nc_row_adj(NcGeom g, const float2 *__restrict__ tmp,
                                                    const float2 *__restrict__ b1,
                                                    float2 *__restrict__ img) {
  __shared__ float2 tile[NCE];
  __shared__ float2 twl[nc_table_len(WIDE)];
  const int tid = threadIdx.x;
  const int t = blockIdx.y;
  const int y0 = blockIdx.x * g.RBa;
  const int nr = min(g.RBa, g.H - y0);
  const long HW = (long)g.H * g.W;
  constexpr bool CT = PL::L != 0;
  const int Gx = CT ? PL::L : g.Gx;
  const float2 *tw = stage_twiddles(g.px, twl, tid, NCR);
  __syncthreads();
  NcRowAdjLoad ld{nullptr, Gx};
  NcRowAdjStore<row_slots_nc(WIDE)> st;
#pragma unroll
  for (int k = 0; k < row_slots_nc(WIDE); ++k) st.acc[k] = czero();
  st.img = img + t * HW;
  st.dxi = g.dxi;
  st.dyi = g.dyi;
  st.W = g.W;
  st.Gx = Gx;
  st.y0 = y0;
  for (int c = 0; c < g.C; ++c) {
    ld.tr = tmp + (((long)t * g.C + c) * g.H + y0) * Gx;
    st.bc = b1 + c * HW;
    st.last = (c == g.C - 1);
    if constexpr (CT) {
      static_assert(((NCE / PL::L) * PL::L / PL::RL + NCR - 1) / NCR * PL::RL <= row_slots_nc(WIDE),
                    "coil-sum slots of the last stage");
      fft_io_ct<NCR, PL, NCE / PL::L, false, true, true>(tile, nr, PL::L, 1, +1.f, tid, tw, ld, st);
    }
    else
      fft_io<NCR, NCE, false, true, true, WIDE>(tile, g.px, nr, Gx, 1, +1.f, tid, tw, ld, st);
    __syncthreads();
  }
}

// K^H's grid passes on a compiled plan: adjoint column blocks of three coils
// (two at grid length 512, whose tiles hold more entries: a chunk of 2048
// entries per coil holds most of a tile's; measured 867 -> 923 it/s against
// three at the 256x256x30x12 radial geometry with osf 2).
template <class PL>
void nc_adjoint_ct(const NcGeom &g, const float2 *z, const float2 *b1, float2 *tmp, float2 *img,
                   hipStream_t s) {
  const size_t cps_bytes = sizeof(int) * ((size_t)g.XBa * g.Gy + 1);
  const int nXa = (g.Gx + g.XBa - 1) / g.XBa;
  constexpr int NZ = PL::L == 512 ? 2 : 3;
  hipLaunchKernelGGL((k_nc_col_adj<kPlanNarrow, PL, NZ>), dim3(nXa, g.T * ((g.C + NZ - 1) / NZ)), dim3(NCC),
                     cps_bytes, s, g, z, tmp);
  AV_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_nc_row_adj<kPlanNarrow, PL>), dim3((g.H + g.RBa - 1) / g.RBa, g.T), dim3(NCR), 0,
                     s, g, (const float2 *)tmp, b1, img);
  AV_LAUNCH_CHECK();
}

// Coils per adjoint column block on a runtime plan.  Two share the tile's tables,
// which pays where one coil per block already makes more than eleven blocks per
// CU; below that it only lengthens the chain.  Measured on MI355X, K^H with two
// coils against one (grid length, one-coil blocks): 288 (432) +23%, 336 (2016)
// +7%, 400 (2400) +1%, 448 (2688) +1%, 504 (3024) -4%, 288 (4608) -2%, 320 (5120)
// -6%, 448 (13440) -10%.  Two-stage grids: 225 to 240 +4 to +18%, 200 -4 to +26%.
// Wide kernels, whose two-coil form holds more registers, gain only on tiles of
// more than 3264 cells: 312 +9 to +23%, 528 to 792 +2 to +15%, 840 to 1024 -8 to
// -13% (1440 blocks: +2%).
int nc_adj_coils(int kind, const NcGeom &g, int nXa) {
  if ((long)nXa * g.T * g.C <= 2816) return 1;
  return kind == kPlanNarrow || g.XBa * g.Gy > 3264 ? 2 : 1;
}

// On the geometry's runtime plans.
template <int KIND, int NZ>
void nc_col_adj_rt(const NcGeom &g, int nXa, const float2 *z, float2 *tmp, hipStream_t s) {
  const size_t cps_bytes = sizeof(int) * ((size_t)g.XBa * g.Gy + 1);
  hipLaunchKernelGGL((k_nc_col_adj<KIND, NcPlanRt, NZ>), dim3(nXa, g.T * ((g.C + NZ - 1) / NZ)),
                     dim3(NCC), cps_bytes, s, g, z, tmp);
  AV_LAUNCH_CHECK();
}
template <int KIND>
void nc_adjoint_rt(const NcGeom &g, const float2 *z, const float2 *b1, float2 *tmp, float2 *img,
                   hipStream_t s) {
  const int nXa = (g.Gx + g.XBa - 1) / g.XBa;
  if constexpr (KIND == kPlanTwo)
    nc_col_adj_rt<KIND, 1>(g, nXa, z, tmp, s);
  else if (nc_adj_coils(KIND, g, nXa) == 1)
    nc_col_adj_rt<KIND, 1>(g, nXa, z, tmp, s);
  else
    nc_col_adj_rt<KIND, 2>(g, nXa, z, tmp, s);
  hipLaunchKernelGGL((k_nc_row_adj<KIND, NcPlanRt>), dim3((g.H + g.RBa - 1) / g.RBa, g.T), dim3(NCR),
                     0, s, g, (const float2 *)tmp, b1, img);
  AV_LAUNCH_CHECK();
}

}  // namespace

void launch_nc_adjoint(const NcGeom &g, const float2 *z, const float2 *b1, float2 *tmp,
                       float2 *img, hipStream_t s) {
  switch (nc_ct_len(g)) {
    case 384: nc_adjoint_ct<NcPlan384>(g, z, b1, tmp, img, s); return;
    case 512: nc_adjoint_ct<NcPlan512>(g, z, b1, tmp, img, s); return;
    case 192: nc_adjoint_ct<NcPlan192>(g, z, b1, tmp, img, s); return;
    case 256: nc_adjoint_ct<NcPlan256>(g, z, b1, tmp, img, s); return;
    default: break;
  }
  switch (g.wide) {
    case kPlanTwo: nc_adjoint_rt<kPlanTwo>(g, z, b1, tmp, img, s); break;
    case kPlanWide: nc_adjoint_rt<kPlanWide>(g, z, b1, tmp, img, s); break;
    default: nc_adjoint_rt<kPlanNarrow>(g, z, b1, tmp, img, s); break;
  }
}

}  // namespace avionic
