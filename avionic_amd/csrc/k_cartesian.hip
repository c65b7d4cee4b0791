// Cartesian plans, the compact gather and the standalone 2D transform; the
// operator's column and row passes are in k_cart_col.hip and k_cart_row.hip.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "cart_device.hpp"
#include "pool.hpp"

namespace avionic {

// Dense [t][c][H][W] -> compact rows, times the mask.
__global__ void k_compact_gather(CartGeom g, const float2 *__restrict__ dense,
                                 float2 *__restrict__ compact) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = g.nrows_c * g.W;
  if (i >= n) return;
  const long row = i / g.W;
  const int x = (int)(i % g.W);
  const int4 ri = g.rowinfo[row];
  compact[i] = cscale(dense[(((long)ri.x * g.C + ri.y) * g.H + ri.w) * g.W + x],
                      g.mrows[(long)ri.z * g.W + x]);
}

// Standalone batched 2D FFT (used by avionic_fft2, the AGILE FFT
// replacement): rows out of place (the centred y shift permutes rows between
// blocks), then columns in place.  Each stage chain reads its first stage from
// global memory and writes its last stage there.
struct FftRowLoad {
  const float2 *base;  // image
  int H, W, y0, centered;
  __device__ float2 operator()(int b, int i, int) const {
    const int y = centered ? wrap_half(y0 + b, H) : y0 + b;
    return gld(base, (unsigned)(y * W + (centered ? wrap_half(i, W) : i)));
  }
};
struct FftRowStore {
  float2 *base;  // image row y0
  int W, centered;
  __device__ void operator()(int b, int i, float2 v, int) const {
    gst(base, (unsigned)(b * W + (centered ? wrap_half(i, W) : i)), v);
  }
};
template <int KIND>
__global__ __launch_bounds__(NT) void k_fft_rows_oop(const float2 *in, float2 *outp, FftPlan pw,
                                                     int H, int W, int RB, int sign,
                                                     int centered) {
  __shared__ float2 tile[EMAX];
  __shared__ float2 twl[KIND == kPlanWide ? kMaxFftLen : kMaxFftLenNarrow];
  const int tid = threadIdx.x;
  const long img = (long)blockIdx.y * H * W;
  const int y0 = blockIdx.x * RB;
  const float2 *tw = stage_twiddles(pw, twl, tid, NT);
  __syncthreads();
  FftRowLoad ld{in + img, H, W, y0, centered};
  FftRowStore st{outp + img + (long)y0 * W, W, centered};
  fft_io<NT, EMAX, false, true, true, KIND>(tile, pw, min(RB, H - y0), W, 1, (float)sign, tid, tw,
                                            ld, st);
}

struct FftColLoad {
  const float2 *base;  // image column xb0
  int W, nx;
  __device__ float2 operator()(int b, int i, int) const {
    return gld(base, (unsigned)(i * W + min(b, nx - 1)));  // columns past the last: dropped
  }
};
struct FftColStore {
  float2 *base;
  int H, W, nx, centered;
  float scale;
  __device__ void operator()(int b, int i, float2 v, int) const {
    if (b < nx) gst(base, (unsigned)((centered ? wrap_half(i, H) : i) * W + b), cscale(v, scale));
  }
};
template <int KIND>
__global__ __launch_bounds__(NT) void k_fft_cols(float2 *data, FftPlan ph, int H, int W, int XB,
                                                 int sign, int centered, float scale) {
  __shared__ float2 tile[EMAX];
  __shared__ float2 twl[KIND == kPlanWide ? kMaxFftLen : kMaxFftLenNarrow];
  const int tid = threadIdx.x;
  const int xb0 = blockIdx.x * XB;
  float2 *base = data + (long)blockIdx.y * H * W + xb0;
  const float2 *tw = stage_twiddles(ph, twl, tid, NT);
  __syncthreads();
  FftColLoad ld{base, W, min(XB, W - xb0)};
  FftColStore st{base, H, W, min(XB, W - xb0), centered, scale};
  fft_io<NT, EMAX, true, true, true, KIND>(tile, ph, XB, 1, XB, (float)sign, tid, tw, ld, st);
}

// ---------------------------------------------------------------------------
// host side

#ifndef AVIONIC_COL_MAXXB
#define AVIONIC_COL_MAXXB 64
#endif
static int pick_xb(int H, int W, int emax = EMAX) {
  int xb = 1;
  while (xb * 2 * H <= emax && xb * 2 <= AVIONIC_COL_MAXXB && xb < W) xb *= 2;
  return xb;
}

static int log2_ceil(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return l;
}
static int col_tile(const CartGeom &g, bool wide) {
  if (!g.ph.ra) return pick_xb(g.H, g.W, kColTileElems);
  const int lb = log2_ceil(g.ph.rb), la = log2_ceil(g.ph.ra);
  int xb = std::min(64, NT >> (wide ? std::max(lb, la - log2_ceil(two_most(g.ph.rb))) : la));
  while (xb >= 2 * g.W) xb /= 2;
  return xb;
}
void set_col_tiles(CartGeom &g, bool wide) {
  g.XB = col_tile(g, wide);
  g.lxb = log2_ceil(g.XB);
  g.nxb = (g.W + g.XB - 1) / g.XB;
  if (g.ph.ra)
    g.ckind = g.ph.L == 256 && g.lxb == 4 ? kCol256 : kColTwo;
  else
    g.ckind = plan_is_wide(g.ph) ? kColWide : kColRt;
}
void set_row_tiles(CartGeom &g, bool wide) {
  if (!g.pw.ra) {
    g.RB = std::max(1, std::min(kRowMaxRows, kRowTileElems / g.W));
    g.rkind = plan_is_wide(g.pw) ? kRowWide : kRowRt;
    return;
  }
  g.ljb = log2_ceil(g.pw.ra);
  g.lja = wide ? std::max(log2_ceil(g.pw.rb), g.ljb - log2_ceil(two_most(g.pw.rb))) : g.ljb;
  g.RB = NT >> g.lja;
  g.rkind = g.pw.L == 256 ? kRow256 : kRowTwo;
}
long wide_col_blocks(const CartGeom &g) {
  const int xb = col_tile(g, true);
  return (long)((g.W + xb - 1) / xb) * g.T;
}

// Radices of a two-stage transform: the pair closest to square (fewest idle
// lanes), the larger first.
static void pick_two_stage(FftPlan &p) {
  for (int rb = kMaxRadix; rb >= 1; --rb)
    if (rb * rb <= p.L && p.L % rb == 0 && p.L / rb <= kMaxRadix) {
      p.ra = p.L / rb;
      p.rb = rb;
      return;
    }
}

// Stages of the float transforms: over the factorisations of L into plan
// radices (largest first), the one with the least work per element: a
// radix's own operations, the twiddles after the first stage, and about 8
// operations for the stage's LDS round trip and indices.
static void pick_stages(int m, int most, double cost, int n, int *r, double &best, FftPlan &p) {
  static const double ops[kMaxRadix + 1] = {0, 0, 2, 5.3, 4, 8, 7.3, 11.5, 6.5, 10, 10, 17, 9.3,
                                            20, 0, 0, 10.5};
  if (m == 1) {
    if (cost < best) {
      best = cost;
      p.nx = n;
      std::copy(r, r + n, p.rx);
    }
    return;
  }
  if (n == kMaxStages) return;
  for (int q = std::min(most, m); q >= 2; --q)
    if (m % q == 0 && plan_radix(q, true)) {
      r[n] = q;
      pick_stages(m / q, q, cost + ops[q] + 8 + (n ? 4 : 0), n + 1, r, best, p);
    }
}

void fft_plan_host(int L, FftPlan &p, std::vector<float2> &tw) {
  AV_CHECK(L >= 1 && L <= kMaxFftLen, "FFT length out of range (1..1024)");
  p = FftPlan{};
  p.L = L;
  int m = L, ns = 1;
  const int order[] = {16, 8, 4, 2, 3, 5, 7, 11, 13};
  for (int r : order) {
    while (m % r == 0) {
      AV_CHECK(p.nst < kMaxStages, "FFT plan too long");
      p.radix[p.nst] = r;
      p.ns[p.nst] = ns;
      ns *= r;
      m /= r;
      p.nst++;
    }
  }
  AV_CHECK(m == 1, "FFT length must factor into 2, 3, 5, 7, 11 and 13");
  pick_two_stage(p);
  int r[kMaxStages];
  double best = 1e30;
  pick_stages(L, kMaxRadix, 0.0, 0, r, best, p);
  while (p.nx < 2) p.rx[p.nx++] = 1;
  tw.resize(L);
  for (int k = 0; k < L; ++k) {
    const double a = -2.0 * M_PI * (double)k / (double)L;
    tw[k] = make_float2((float)std::cos(a), (float)std::sin(a));
  }
}

void make_fft_plan(int L, FftPlan &p, void **d_tw) {
  std::vector<float2> tw;
  fft_plan_host(L, p, tw);
  *d_tw = device_alloc(sizeof(float2) * L);
  AV_HIP(hipMemcpy(*d_tw, tw.data(), sizeof(float2) * L, hipMemcpyHostToDevice));
  AV_HIP(hipStreamSynchronize(nullptr));  // landed before any stream reads it
  p.tw = (const float2 *)*d_tw;
}

// One block per mask row (t, y): its sum of squares, or -1 when no value is
// nonzero (a NaN counts as nonzero).
__global__ __launch_bounds__(NT) void k_mask_rows(const float *__restrict__ mask, int W,
                                                  double *__restrict__ out) {
  __shared__ double red[NT];
  __shared__ int any;
  if (threadIdx.x == 0) any = 0;
  __syncthreads();
  double acc = 0.0;
  int mine = 0;
  for (int x = threadIdx.x; x < W; x += NT) {
    const float v = mask[(long)blockIdx.x * W + x];
    acc += (double)v * v;
    mine |= v != 0.f;
  }
  if (mine) any = 1;
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) out[blockIdx.x] = any ? s : -1.0;
}
// Mask values of the sampled rows (ones without a mask), one block per row.
__global__ void k_mask_gather(const float *__restrict__ mask, const int *__restrict__ src, int W,
                              float *__restrict__ mrows) {
  const long r = blockIdx.x;
  for (int x = threadIdx.x; x < W; x += blockDim.x)
    mrows[r * W + x] = mask ? mask[(long)src[r] * W + x] : 1.f;
}

CartPlan::~CartPlan() {
  if (d_tables) (void)hipFree(d_tables);
}

void CartPlan::init(int W, int H, int C, int T, const float *mask, int centered, hipStream_t s) {
  AV_CHECK(W >= 1 && H >= 1 && C >= 1 && T >= 1, "invalid operator dimensions");
  AV_CHECK(H <= kMaxFftLen && W <= kMaxFftLen, "image dimensions exceed the longest FFT (1024)");
  g = CartGeom{};
  g.W = W; g.H = H; g.C = C; g.T = T;
  g.centered = centered ? 1 : 0;
  g.scale = (float)(1.0 / std::sqrt((double)H * W));
  has_mask = mask != nullptr;
  std::vector<double> sums((size_t)T * H, 0.0);  // -1: row not sampled
  if (mask) {
    double *d = (double *)device_alloc(sizeof(double) * sums.size());
    hipLaunchKernelGGL(k_mask_rows, dim3((unsigned)sums.size()), dim3(NT), 0, s, mask, W, d);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
      e = hipMemcpyAsync(sums.data(), d, sizeof(double) * sums.size(), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(d);
    AV_HIP(e);
  }
  h_row_off.assign(T + 1, 0);
  h_rows.clear();
  std::vector<int> src;  // mask row t H + y of each sampled row
  mask_norm2 = 0.0;
  for (int t = 0; t < T; ++t) {
    for (int y = 0; y < H; ++y) {
      const double v = sums[(size_t)t * H + y];
      if (v == -1.0) continue;
      mask_norm2 += v;
      h_rows.push_back(y);
      src.push_back(t * H + y);
    }
    h_row_off[t + 1] = (int)h_rows.size();
  }
  g.nrows = (long)h_rows.size();
  g.nrows_c = g.nrows * C;
  std::vector<int> rowmap((size_t)T * H, -1);
  for (int t = 0; t < T; ++t)
    for (int k = h_row_off[t]; k < h_row_off[t + 1]; ++k) rowmap[(size_t)t * H + h_rows[k]] = k - h_row_off[t];
  std::vector<int4> info;
  info.reserve(g.nrows_c);
  for (int t = 0; t < T; ++t) {
    const int r0 = h_row_off[t], S = h_row_off[t + 1] - r0;
    for (int c = 0; c < C; ++c)
      for (int k = 0; k < S; ++k) info.push_back(make_int4(t, c, r0 + k, h_rows[r0 + k]));
  }
  std::vector<float2> twx, twy;
  fft_plan_host(W, g.pw, twx);
  fft_plan_host(H, g.ph, twy);
  // one allocation and one copy for all tables, then the mask rows behind them
  std::vector<char> host;
  auto put = [&](const void *p, size_t bytes) {
    const size_t at = host.size();
    host.resize(at + (bytes + 255) / 256 * 256);
    if (bytes) std::memcpy(host.data() + at, p, bytes);
    return at;
  };
  const size_t o_off = put(h_row_off.data(), sizeof(int) * h_row_off.size());
  const size_t o_rows = put(h_rows.data(), sizeof(int) * h_rows.size());
  const size_t o_src = put(src.data(), sizeof(int) * src.size());
  const size_t o_info = put(info.data(), sizeof(int4) * info.size());
  const size_t o_map = put(rowmap.data(), sizeof(int) * rowmap.size());
  const size_t o_twx = put(twx.data(), sizeof(float2) * twx.size());
  const size_t o_twy = put(twy.data(), sizeof(float2) * twy.size());
  const size_t o_mrows = host.size();
  d_tables = device_alloc(o_mrows + sizeof(float) * (size_t)g.nrows * W + 256);
  char *base = (char *)d_tables;
  AV_HIP(hipMemcpy(base, host.data(), host.size(), hipMemcpyHostToDevice));
  g.row_off = (const int *)(base + o_off);
  g.rows = (const int *)(base + o_rows);
  g.rowinfo = (const int4 *)(base + o_info);
  g.rowmap = (const int *)(base + o_map);
  g.mrows = (const float *)(base + o_mrows);
  g.pw.tw = (const float2 *)(base + o_twx);
  g.ph.tw = (const float2 *)(base + o_twy);
  if (g.nrows > 0) {
    hipLaunchKernelGGL(k_mask_gather, dim3((unsigned)g.nrows), dim3(NT), 0, nullptr, mask,
                       (const int *)(base + o_src), W, (float *)(base + o_mrows));
    AV_LAUNCH_CHECK();
  }
  set_col_tiles(g, wide_col_blocks(g) >= kColWideBlocks);
  set_row_tiles(g, true);
  if (row_blocks() < kRowWideBlocks) set_row_tiles(g, false);
  // The tables above come from pageable host memory (such a copy, on the null
  // stream, may return before its data has landed) and from a kernel there, and
  // the kernels that index with them may run on non-blocking streams, which do
  // not wait for the null stream.  Waiting for the null stream alone leaves those streams'
  // own work running.
  AV_HIP(hipStreamSynchronize(nullptr));
}

void launch_compact_gather(const CartGeom &g, const float2 *dense, float2 *compact, hipStream_t s) {
  const long n = g.nrows_c * g.W;
  if (n == 0) return;
  hipLaunchKernelGGL(k_compact_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, dense,
                     compact);
  AV_LAUNCH_CHECK();
}

int plan_kind(const FftPlan &p, int B) {
  if (p.ra && B * p.ra <= NT) return kPlanTwo;
  return plan_is_wide(p) ? kPlanWide : kPlanNarrow;
}

static void launch_cols(float2 *data, const FftPlan &p, int L, int plane, int batch, int sign,
                        int centered, float scale, hipStream_t s) {
  int XB = pick_xb(L, plane);
  while (p.ra && XB > 1 && XB * p.ra > NT) XB /= 2;
  const dim3 grid((plane + XB - 1) / XB, batch), block(NT);
  switch (plan_kind(p, XB)) {
    case kPlanTwo: hipLaunchKernelGGL(k_fft_cols<kPlanTwo>, grid, block, 0, s, data, p, L, plane, XB, sign, centered, scale); break;
    case kPlanWide: hipLaunchKernelGGL(k_fft_cols<kPlanWide>, grid, block, 0, s, data, p, L, plane, XB, sign, centered, scale); break;
    default: hipLaunchKernelGGL(k_fft_cols<kPlanNarrow>, grid, block, 0, s, data, p, L, plane, XB, sign, centered, scale); break;
  }
  AV_LAUNCH_CHECK();
}

void launch_fft2(float2 *data, const FftPlan &pw, const FftPlan &ph, int H, int W, int batch,
                 int sign, int centered, float scale, hipStream_t s) {
  const int RB = pw.ra ? std::min(EMAX / W, NT / pw.ra) : EMAX / W;
  float2 *tmp = (float2 *)device_alloc_async(sizeof(float2) * (size_t)H * W * batch, s);
  const dim3 grid((H + RB - 1) / RB, batch), block(NT);
  switch (plan_kind(pw, RB)) {
    case kPlanTwo: hipLaunchKernelGGL(k_fft_rows_oop<kPlanTwo>, grid, block, 0, s, data, tmp, pw, H, W, RB, sign, centered); break;
    case kPlanWide: hipLaunchKernelGGL(k_fft_rows_oop<kPlanWide>, grid, block, 0, s, data, tmp, pw, H, W, RB, sign, centered); break;
    default: hipLaunchKernelGGL(k_fft_rows_oop<kPlanNarrow>, grid, block, 0, s, data, tmp, pw, H, W, RB, sign, centered); break;
  }
  AV_LAUNCH_CHECK();
  launch_cols(tmp, ph, H, W, batch, sign, centered, scale, s);
  AV_HIP(hipMemcpyAsync(data, tmp, sizeof(float2) * (size_t)H * W * batch, hipMemcpyDeviceToDevice, s));
  AV_HIP(hipFreeAsync(tmp, s));
}

// In-place transform along the slowest axis of `batch` arrays [L][plane]:
// one length-L transform per column of the plane (the depth axis of a volume).
void launch_fft_axis0(float2 *data, const FftPlan &p, int L, int plane, int batch, int sign,
                      float scale, hipStream_t s) {
  launch_cols(data, p, L, plane, batch, sign, 0, scale, s);
}

}  // namespace avionic
