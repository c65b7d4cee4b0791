// Kaiser-Bessel gridding, K (noncart.hpp): column, row and sample passes.
#include "nc_device.hpp"

namespace avionic {

namespace {

// ------------------------------------------------------------ K, column pass
// The first stage's input b1_c (u - usub) dxi dyi, zero outside the image.
// With SLOTS (the compiled kernels) a lane keeps (u - usub) dxi dyi of its
// first-stage elements in registers from the block's first coil (`first`)
// and loads only the coil map for the others: the lane -> element mapping of
// a stage is the same for every coil.  The product is formed the same way
// either way.
template <int SLOTS>
struct NcColFwdLoad {
  const float2 *ut, *us, *bc;
  const float *dxi, *dyi;
  int W, H, Gy, xb0;
  bool delta, first;
  float2 img[SLOTS > 0 ? SLOTS : 1];
  __device__ float2 operator()(int b, int i, int slot) {
    const int x = xb0 + b;
    if (x >= W) return czero();
    const int y = wrap_up(i + H / 2, Gy);
    if (y >= H) return czero();
    const unsigned si = (unsigned)(y * W + x);
    if constexpr (SLOTS > 0) {
      if (first) img[slot] = cscale(delta ? csub(ut[si], us[si]) : ut[si], dxi[x] * dyi[y]);
      return cmul(bc[si], img[slot]);
    } else {
      const float2 v = delta ? csub(ut[si], us[si]) : ut[si];
      return cmul(bc[si], cscale(v, dxi[x] * dyi[y]));
    }
  }
};
// First-stage elements per lane of the compiled column forward pass.
template <class PL>
constexpr int nc_colf_slots() {
  if constexpr (PL::L == 0)
    return 0;
  else
    return (PL::XB * PL::L / PL::R0 + AVIONIC_NC_COLF_THREADS - 1) / AVIONIC_NC_COLF_THREADS * PL::R0;
}
struct NcColFwdStore {
  float2 *tc;  // tmp rows of (t, c): [Gy][W]
  int W, xb0;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int x = xb0 + b;
    if (x < W) tc[(unsigned)(i * W + x)] = v;
  }
};

template <int WIDE, class PL>
__global__ __launch_bounds__(NCF) void k_nc_col_fwd(NcGeom g, const float2 *__restrict__ u,
                                                    const float2 *__restrict__ usub,
                                                    const float2 *__restrict__ b1,
                                                    float2 *__restrict__ tmp) {
  __shared__ float2 tile[NCE];
  __shared__ float2 twl[nc_table_len(WIDE)];
  const int tid = threadIdx.x;
  const int t = blockIdx.y;
  const long HW = (long)g.H * g.W;
  constexpr bool CT = PL::L != 0;
  const int XB = CT ? PL::XB : g.XBf;
  const float2 *tw = stage_twiddles(g.py, twl, tid, NCF);
  __syncthreads();
  NcColFwdLoad<nc_colf_slots<PL>()> ld;
  ld.ut = u + t * HW;
  ld.us = usub ? usub + t * HW : nullptr;
  ld.delta = usub != nullptr;
  ld.dxi = g.dxi;
  ld.dyi = g.dyi;
  ld.W = g.W;
  ld.H = g.H;
  ld.Gy = CT ? PL::L : g.Gy;
  ld.xb0 = blockIdx.x * XB;
  NcColFwdStore st{nullptr, g.W, (int)blockIdx.x * XB};
  // coils [c0, c1) of this block (blockIdx.z picks the coil group)
  const int cpg = (g.C + gridDim.z - 1) / gridDim.z;
  const int c0 = blockIdx.z * cpg, c1 = min(g.C, c0 + cpg);
  for (int c = c0; c < c1; ++c) {
    ld.first = c == c0;
    ld.bc = b1 + c * HW;
    st.tc = tmp + ((long)t * g.C + c) * g.Gy * g.W;
    if constexpr (CT)
      fft_io_ct<NCF, PL, PL::XB, true, true, true>(tile, PL::XB, 1, PL::XB, -1.f, tid, tw,
                                                      ld, st);
    else
      fft_io<NCF, NCE, true, true, true, WIDE>(tile, g.py, XB, 1, XB, -1.f, tid, tw, ld, st);
    __syncthreads();
  }
}

// --------------------------------------------------------------- K, row pass
// Transform b of a block: coil cz + b / RB, grid row gy0 + b % RB of that
// coil's tmp plane (zero past the block's coils or rows).
template <int NZ>
struct NcRowFwdLoad {
  const float2 *tr;  // tmp row gy0 of plane (t, cz): [.][W]; coil planes GyW apart
  long plane;        // Gy W
  int W, Gx, RB, nr, nz;
  __device__ float2 operator()(int b, int i, int) const {
    const int x = wrap_up(i + W / 2, Gx);
    if constexpr (NZ == 1) {
      return x < W ? tr[(unsigned)(b * W + x)] : czero();
    } else {
      const int q = b / RB, r = b - q * RB;
      return x < W && q < nz && r < nr ? tr[q * plane + (unsigned)(r * W + x)] : czero();
    }
  }
};

// NZ coils of a frame per block (2 in the compiled kernels, RB = 5 grid rows
// each): the tile holds NZ x RB transformed rows, and the row table's entries
// of those rows are loaded once for all coils.  Each coil's partials are the
// one-coil partials.
template <int WIDE, class PL, int NZ>
__global__ __launch_bounds__(NCR) void k_nc_row_fwd(NcGeom g, const float2 *__restrict__ tmp,
                                                    float2 *__restrict__ part) {
  __shared__ float2 tile[NCE];
  __shared__ float2 twl[nc_table_len(WIDE)];
  constexpr bool CT = PL::L != 0;
  static_assert(CT || NZ == 1, "coil groups need the compiled kernels");
  const int tid = threadIdx.x;
  const int RB = CT ? NCE / PL::L / NZ : g.RBf;  // grid rows per coil
  const int ngrp = (g.C + NZ - 1) / NZ;
  const int t = blockIdx.y / ngrp, cz = (blockIdx.y % ngrp) * NZ;
  const int nz = min(NZ, g.C - cz);
  const int gy0 = blockIdx.x * RB;
  const int nr = min(RB, g.Gy - gy0);
  const int Gx = CT ? PL::L : g.Gx;
  const float2 *tw = stage_twiddles(g.px, twl, tid, NCR);
  __syncthreads();
  const long plane = (long)g.Gy * g.W;
  NcRowFwdLoad<NZ> ld{tmp + ((long)t * g.C + cz) * plane + (long)gy0 * g.W, plane, g.W, Gx, RB, nr,
                  nz};
  NoStore ns;
  if constexpr (CT)
    fft_io_ct<NCR, PL, NCE / PL::L, false, true, false>(tile, NZ * RB, PL::L, 1, -1.f, tid, tw, ld,
                                                        ns);
  else
    fft_io<NCR, NCE, false, true, false, WIDE>(tile, g.px, nr, Gx, 1, -1.f, tid, tw, ld, ns);
  // tile[(q RB + r) Gx + i] holds grid row gy0 + r of coil cz + q in natural order.
  const int *rp = g.rptr + (long)t * (g.Gy + 1);
  const int e0 = rp[gy0], e1 = rp[gy0 + nr];
  float2 *pp = part + ((long)t * g.C + cz) * g.M * kNcTaps;  // coil cz + q: M kNcTaps further
  for (int e = e0 + tid; e < e1; e += NCR) {
    // (partial index dy M + m, grid row, first grid column, row weight) and the
    // column weights: no load here depends on another.  Consecutive points of a
    // spoke stay consecutive in a plane of partials.
    const int4 h = g.rhdr[e];
    const float4 wx = g.rwx[e];
    const int qx = h.z;
#pragma unroll
    for (int q = 0; q < NZ; ++q) {
      if (q >= nz) break;
      const float2 *row = tile + (q * RB + h.y - gy0) * Gx;
      float2 acc = cscale(row[qx], wx.x);
      acc = cadd(acc, cscale(row[wrap_up(qx + 1, Gx)], wx.y));
      acc = cadd(acc, cscale(row[wrap_up(qx + 2, Gx)], wx.z));
      if (wx.w != 0.f) acc = cadd(acc, cscale(row[wrap_up(qx + 3, Gx)], wx.w));  // rare
      pp[(long)q * g.M * kNcTaps + (unsigned)h.x] = cscale(acc, __int_as_float(h.w));
    }
  }
}

// ------------------------------------------------------------- sample pass
__device__ inline double block_sum(double v, double *red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int s = NCR / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  return red[0];
}

template <int MODE>
__global__ __launch_bounds__(NCR) void k_nc_samples(NcGeom g, const float2 *__restrict__ part,
                                                    float2 *__restrict__ out, float2 *z,
                                                    const float2 *__restrict__ d,
                                                    const DevScalars *__restrict__ sc,
                                                    double *__restrict__ partial) {
  __shared__ double red[NCR];
  const long n = (long)g.T * g.C * g.M;
  float sigma = 0.f, inv = 0.f;
  if (MODE == kNcDualUpdate) {
    sigma = (float)sc->sigma;
    inv = (float)(1.0 / (1.0 + sc->sigma / sc->lambda));
  }
  double acc = 0.0;
  for (long e = (long)blockIdx.x * NCR + threadIdx.x; e < n; e += (long)gridDim.x * NCR) {
    const long pl = e / g.M, m = e - pl * g.M;  // plane (t, c), point
    const int t = (int)pl / g.C;
    const float2 *p = part + pl * g.M * kNcTaps + m;
    const float2 p0 = p[0], p1 = p[g.M], p2 = p[2L * g.M];
    float2 v = make_float2(p0.x + p1.x + p2.x, p0.y + p1.y + p2.y);
    if (g.last[t]) v = cadd(v, p[3L * g.M]);
    v = cscale(v, g.sw[(long)t * g.M + m]);
    if (MODE == kNcApplyK) {
      out[e] = v;
    } else if (MODE == kNcDualUpdate) {
      float2 zz = cadd(z[e], cscale(v, sigma));
      zz = cscale(csub(zz, cscale(d[e], sigma)), inv);
      z[e] = zz;
    } else if (MODE == kNcNorm2) {
      acc += (double)cabs2(v);
    } else {
      acc += (double)cabs2(csub(v, d[e]));
    }
  }
  if (MODE == kNcNorm2 || MODE == kNcResidual) {
    const double s = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
  }
}

// K's grid passes on a compiled plan: row blocks of two coils, NCE / L / 2
// grid rows each.
template <class PL>
void nc_forward_ct(const NcGeom &g, const float2 *u, const float2 *usub, const float2 *b1,
                   float2 *tmp, float2 *part, hipStream_t s) {
  constexpr int rb2 = NCE / PL::L / 2;
  const dim3 gc((g.W + g.XBf - 1) / g.XBf, g.T, g.CG);
  const dim3 gr2((g.Gy + rb2 - 1) / rb2, g.T * ((g.C + 1) / 2));
  hipLaunchKernelGGL((k_nc_col_fwd<kPlanNarrow, PL>), gc, dim3(NCF), 0, s, g, u, usub, b1, tmp);
  AV_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_nc_row_fwd<kPlanNarrow, PL, 2>), gr2, dim3(NCR), 0, s, g, (const float2 *)tmp, part);
  AV_LAUNCH_CHECK();
}

// On the geometry's runtime plans.
template <int KIND>
void nc_forward_rt(const NcGeom &g, const float2 *u, const float2 *usub, const float2 *b1,
                   float2 *tmp, float2 *part, hipStream_t s) {
  const dim3 gc((g.W + g.XBf - 1) / g.XBf, g.T, g.CG), gr((g.Gy + g.RBf - 1) / g.RBf, g.T * g.C);
  hipLaunchKernelGGL((k_nc_col_fwd<KIND, NcPlanRt>), gc, dim3(NCF), 0, s, g, u, usub, b1, tmp);
  AV_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_nc_row_fwd<KIND, NcPlanRt, 1>), gr, dim3(NCR), 0, s, g, (const float2 *)tmp,
                     part);
  AV_LAUNCH_CHECK();
}

}  // namespace

void launch_nc_forward_grid(const NcGeom &g, const float2 *u, const float2 *usub,
                            const float2 *b1, float2 *tmp, float2 *part, hipStream_t s) {
  switch (nc_ct_len(g)) {
    case 384: nc_forward_ct<NcFwd384>(g, u, usub, b1, tmp, part, s); return;
    case 512: nc_forward_ct<NcPlan512>(g, u, usub, b1, tmp, part, s); return;
    case 192: nc_forward_ct<NcFwd192>(g, u, usub, b1, tmp, part, s); return;
    case 256: nc_forward_ct<NcPlan256>(g, u, usub, b1, tmp, part, s); return;
    default: break;
  }
  switch (g.wide) {
    case kPlanTwo: nc_forward_rt<kPlanTwo>(g, u, usub, b1, tmp, part, s); break;
    case kPlanWide: nc_forward_rt<kPlanWide>(g, u, usub, b1, tmp, part, s); break;
    default: nc_forward_rt<kPlanNarrow>(g, u, usub, b1, tmp, part, s); break;
  }
}

int nc_sample_blocks(const NcGeom &g) {
  const long n = (long)g.T * g.C * g.M;
  return (int)std::max<long>(1, std::min<long>(1024, (n + NCR - 1) / NCR));
}

int launch_nc_samples(int mode, const NcGeom &g, const float2 *part, float2 *out, float2 *z,
                      const float2 *d, const DevScalars *sc, double *partial, hipStream_t s) {
  const int nb = nc_sample_blocks(g);
  switch (mode) {
    case kNcApplyK: hipLaunchKernelGGL(k_nc_samples<kNcApplyK>, dim3(nb), dim3(NCR), 0, s, g, part, out, z, d, sc, partial); break;
    case kNcDualUpdate: hipLaunchKernelGGL(k_nc_samples<kNcDualUpdate>, dim3(nb), dim3(NCR), 0, s, g, part, out, z, d, sc, partial); break;
    case kNcNorm2: hipLaunchKernelGGL(k_nc_samples<kNcNorm2>, dim3(nb), dim3(NCR), 0, s, g, part, out, z, d, sc, partial); break;
    case kNcResidual: hipLaunchKernelGGL(k_nc_samples<kNcResidual>, dim3(nb), dim3(NCR), 0, s, g, part, out, z, d, sc, partial); break;
    default: AV_CHECK(false, "bad sample-pass mode");
  }
  AV_LAUNCH_CHECK();
  return nb;
}

}  // namespace avionic
