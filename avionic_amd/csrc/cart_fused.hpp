// Fused Cartesian operator passes on a runtime plan: lengths that are not a
// product of two radices up to 16 (those run cart_two.hpp).
//
// Column passes: the first radix stage reads the image (times the coil map)
// straight from global memory and the last stage hands each output to its
// consumer: the forward pass keeps only the sampled phase-encode rows, the
// adjoint pass accumulates conj(b1_c) * value over the coils in registers and
// writes K^H z after the last coil.  Row pass: forward row transform, z dual
// update and prox per output, the masked z staged in LDS for the adjoint row
// transform, whose last stage writes zhat.  Only the exchanges between radix
// stages go through LDS; twiddles are staged in LDS once per block.
#pragma once

#include "cart_device.hpp"

namespace avionic {

#ifndef AVIONIC_COL_THREADS
#define AVIONIC_COL_THREADS 256
#endif

constexpr int RTILE = kRowTileElems;
constexpr int NTC = AVIONIC_COL_THREADS;  // threads of a column-pass block
// Outputs per lane of a column-pass stage (narrow / wide plans).
constexpr int col_slots(bool wide) { return max_slots(kColTileElems, NTC, wide); }

// Column transform of one tile on the runtime plan, first stage from `ld`,
// last stage to `st`.
template <bool WIDE, class LD, class ST>
__device__ __forceinline__ void col_fft(float2 *tile, const CartGeom &g, float sign, int tid,
                                        const float2 *tw, LD &ld, ST &st) {
  fft_io<NTC, kColTileElems, true, true, true, WIDE>(tile, g.ph, g.XB, 1, g.XB, sign, tid, tw, ld,
                                                     st);
}

// ------------------------------------------------------------ column forward
// 32-bit offsets from per-(t, c) base pointers (uniform, in SGPRs) keep one
// VGPR per in-flight address.  Lanes of columns past W load a valid element
// and drop it: a load in a divergent branch whose value is used after it gets
// its own wait, which serialises the lane's loads.  Index products use 24-bit
// multiplies (rows and columns are below 2^12).
template <bool DELTA>
struct ColFwdLoad {
  const float2 *ut, *st, *bc;
  int H, W, xb0, centered;
  __device__ float2 operator()(int b, int i, int) const {
    const bool cen = centered != 0;
    const int x = xb0 + b;
    const int xc = x < W ? x : W - 1;
    const int sy = cen ? wrap_half(i, H) : i;
    const int sx = cen ? wrap_half(xc, W) : xc;
    const unsigned si = __umul24((unsigned)sy, (unsigned)W) + (unsigned)sx;
    const float2 bv = gld(bc, si), uv = gld(ut, si);
    return cmul(bv, DELTA ? csub(uv, gld(st, si)) : uv);
  }
};
struct ColFwdStore {
  float2 *kc;       // kcol + (C r0 + c S) W : rows of (t, c)
  const int *rmap;  // LDS: compact row of each k-space row of frame t
  int H, W, xb0, centered;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int x = xb0 + b;
    const int k = rmap[centered ? wrap_half(i, H) : i];
    if (x < W && k >= 0) gst(kc, __umul24((unsigned)k, (unsigned)W) + (unsigned)x, v);
  }
};

// The frame's rowmap (compact row of each k-space row, -1 if not sampled)
// staged in LDS: the store / load functors then need no dependent global
// read before each k-space access.
__device__ inline const int *stage_rowmap(const CartGeom &g, int t, int *lds, int tid, int nt) {
  const int *rm = g.rowmap + (long)t * g.H;
  for (int i = tid; i < g.H; i += nt) lds[i] = rm[i];
  return lds;
}

// Coils [c0, c1) of frame t.
template <bool DELTA, bool WIDE>
__device__ inline void col_forward_fused(const CartGeom &g, int xbi, int t, int c0, int c1,
                                         const float2 *u, const float2 *usub, const float2 *b1,
                                         float2 *kcol, float2 *tile, float2 *twl, int *rml) {
  const int tid = threadIdx.x;
  const long HW = (long)g.H * g.W;
  const float2 *tw = stage_twiddles(g.ph, twl, tid, NTC);
  const int *rmap = stage_rowmap(g, t, rml, tid, NTC);
  __syncthreads();
  const int r0 = g.row_off[t], S = g.row_off[t + 1] - r0;
  ColFwdLoad<DELTA> ld{u + t * HW, DELTA ? usub + t * HW : nullptr, nullptr, g.H, g.W, xbi * g.XB,
                       g.centered};
  ColFwdStore st{nullptr, rmap, g.H, g.W, xbi * g.XB, g.centered};
  for (int c = c0; c < c1; ++c) {
    ld.bc = b1 + c * HW;
    st.kc = kcol + ((long)g.C * r0 + (long)c * S) * g.W;
    col_fft<WIDE>(tile, g, +1.f, tid, tw, ld, st);
    __syncthreads();
  }
}

// ------------------------------------------------------------ column adjoint
// Lanes of unsampled rows (and columns past W) load element 0 of zh, a
// cached dummy, so that the loads of a lane's outputs are not in divergent
// branches.
struct ColAdjLoad {
  const float2 *zh;  // zhat rows of (t, c); when the frame has none, any valid element
  const int *rmap;
  int H, W, xb0, centered;
  __device__ float2 operator()(int b, int i, int) const {
    const int x = xb0 + b;
    const int k = rmap[centered ? wrap_half(i, H) : i];
    const bool use = x < W && k >= 0;
    const float2 z = gld(zh, use ? __umul24((unsigned)k, (unsigned)W) + (unsigned)x : 0u);
    return use ? z : czero();
  }
};
// The coil sum stays in registers, one accumulator per output of the lane.
template <int SLOTS>
struct ColAdjStore {
  float2 acc[SLOTS];
  const float2 *bc;
  float2 *out;  // image frame t
  int H, W, xb0, centered;
  bool last;
  float scale;
  __device__ void operator()(int b, int i, float2 v, int slot) {
    const int x = xb0 + b;
    const int xc = x < W ? x : W - 1;  // b1 load in bounds for every lane: no branch
    const int y = centered ? wrap_half(i, H) : i;
    const unsigned o = __umul24((unsigned)y, (unsigned)W) + (unsigned)xc;
    const float2 a = cadd(acc[slot], cmulc(gld(bc, o), v));
    if (!last)
      acc[slot] = a;
    else if (x < W)
      gst(out, o, cscale(a, scale));
  }
};

template <bool WIDE>
__device__ inline void col_adjoint_fused(const CartGeom &g, int xbi, int t, const float2 *zhat,
                                         const float2 *b1, float2 *out, float2 *tile,
                                         float2 *twl, int *rml) {
  const int tid = threadIdx.x;
  const long HW = (long)g.H * g.W;
  const float2 *tw = stage_twiddles(g.ph, twl, tid, NTC);
  const int *rmap = stage_rowmap(g, t, rml, tid, NTC);
  __syncthreads();
  const int r0 = g.row_off[t], S = g.row_off[t + 1] - r0;
  ColAdjLoad ld{nullptr, rmap, g.H, g.W, xbi * g.XB, g.centered};
  constexpr int SLOTS = col_slots(WIDE);
  ColAdjStore<SLOTS> st;
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) st.acc[k] = czero();
  st.out = out + t * HW;
  st.H = g.H;
  st.W = g.W;
  st.xb0 = xbi * g.XB;
  st.centered = g.centered;
  st.scale = g.scale;
  for (int c = 0; c < g.C; ++c) {
    ld.zh = S > 0 ? zhat + ((long)g.C * r0 + (long)c * S) * g.W : zhat;
    st.bc = b1 + c * HW;
    st.last = (c == g.C - 1);
    col_fft<WIDE>(tile, g, -1.f, tid, tw, ld, st);
    __syncthreads();
  }
}

// ----------------------------------------------------------------- row pass
struct RowLoad {
  const float2 *src;  // kcol + g0 W
  int W;
  __device__ float2 operator()(int b, int i, int) const { return gld(src, (unsigned)(b * W + i)); }
};
// Mask row (index into mrows) of each row of the block, staged in LDS so
// that the mask load does not wait on a global rowinfo load.
__device__ inline const int *stage_mask_rows(const CartGeom &g, long g0, int nr, int *lds, int tid,
                                             int nt) {
  for (int b = tid; b < nr; b += nt) lds[b] = g.rowinfo[g0 + b].z;
  return lds;
}

struct RowDualStore {
  float2 *z;        // z + g0 W: rows of the block
  const float2 *d;  // d + g0 W
  const float *mrows;
  const int *mrow;  // LDS: mask row of local row b
  float2 *tile2;
  int W, wc, centered;
  float scale, sigma, inv;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int kx = centered ? wrap_half(i, W) : i;
    const float mk = gld(mrows, (unsigned)(mrow[b] * W + kx));
    const float2 val = cscale(v, scale * mk);
    const unsigned gi = (unsigned)(b * W + kx);
    float2 zz = gld(z, gi);
    zz = cadd(zz, cscale(val, sigma));
    zz = cscale(csub(zz, cscale(gld(d, gi), sigma)), inv);
    gst_stream(z, gi, zz);
    const int xp = centered ? wrap_add(kx, wc, W) : kx;
    tile2[b * W + xp] = cscale(zz, mk);
  }
};
struct RowAdjStore {
  float2 *zhat;  // zhat + g0 W
  int W, centered;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int kxp = centered ? wrap_half(i, W) : i;
    gst(zhat, (unsigned)(b * W + kxp), v);
  }
};
struct RowNorm2Store {
  const float *mrows;
  const int *mrow;  // LDS: mask row of local row b
  int W, centered;
  float scale;
  double acc;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int kx = centered ? wrap_half(i, W) : i;
    const float2 val = cscale(v, scale * gld(mrows, (unsigned)(mrow[b] * W + kx)));
    acc += (double)cabs2(val);
  }
};
// |K u - d|^2 on the compact data
struct RowResidualStore {
  const float *mrows;
  const int *mrow;
  const float2 *d;  // d + g0 W
  int W, centered;
  float scale;
  double acc;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int kx = centered ? wrap_half(i, W) : i;
    const float2 val = cscale(v, scale * gld(mrows, (unsigned)(mrow[b] * W + kx)));
    acc += (double)cabs2(csub(val, gld(d, (unsigned)(b * W + kx))));
  }
};
// K u into the dense k-space
struct RowApplyStore {
  const float *mrows;
  const int *mrow;
  const int4 *info;  // rowinfo + g0
  float2 *out;
  int W, C, H, centered;
  float scale;
  __device__ void operator()(int b, int i, float2 v, int) {
    const int kx = centered ? wrap_half(i, W) : i;
    const int4 ri = info[b];
    out[(((long)ri.x * C + ri.y) * H + ri.w) * W + kx] =
        cscale(v, scale * gld(mrows, (unsigned)(mrow[b] * W + kx)));
  }
};
// M z of dense or compact k-space
template <bool DENSE>
struct RowMaskLoad {
  const float *mrows;
  const int *mrow;
  const int4 *info;
  const float2 *z;  // dense: the whole k-space; compact: z + g0 W
  int W, C, H, centered;
  __device__ float2 operator()(int b, int i, int) const {
    const int kx = centered ? wrap_half(i, W) : i;
    const float mk = gld(mrows, (unsigned)(mrow[b] * W + kx));
    if (!DENSE) return cscale(gld(z, (unsigned)(b * W + kx)), mk);
    const int4 ri = info[b];
    return cscale(z[(((long)ri.x * C + ri.y) * H + ri.w) * W + kx], mk);
  }
};

template <bool WIDE>
__device__ inline void row_dual_fused(const CartGeom &g, int blk, const float2 *kcol, float2 *z,
                                      const float2 *d, float2 *zhat, const DevScalars *sc,
                                      float2 *tile, float2 *tile2, float2 *twl, int *mrl) {
  const int tid = threadIdx.x;
  const int W = g.W;
  const long g0 = (long)blk * g.RB;
  const int nr = (int)min((long)g.RB, g.nrows_c - g0);
  const float2 *tw = stage_twiddles(g.pw, twl, tid, NT);
  const int *mrow = stage_mask_rows(g, g0, nr, mrl, tid, NT);
  __syncthreads();
  RowLoad ld{kcol + g0 * W, W};
  RowDualStore st;
  st.z = z + g0 * W;
  st.d = d + g0 * W;
  st.mrows = g.mrows;
  st.mrow = mrow;
  st.tile2 = tile2;
  st.W = W;
  st.wc = (W + 1) / 2;
  st.centered = g.centered;
  st.scale = g.scale;
  st.sigma = (float)sc->sigma;
  st.inv = (float)(1.0 / (1.0 + sc->sigma / sc->lambda));
  fft_io<NT, RTILE, false, true, true, WIDE>(tile, g.pw, nr, W, 1, +1.f, tid, tw, ld, st);
  __syncthreads();  // tile2 holds M z for every row of the block
  RowAdjStore st2{zhat + g0 * W, W, g.centered};
  NoLoad nl;
  fft_io<NT, RTILE, false, false, true, WIDE>(tile2, g.pw, nr, W, 1, -1.f, tid, tw, nl, st2);
}

// The modes other than the dual update on a runtime plan; returns the lane's
// part of the sum (kRowNorm2, kRowResidual).
template <int MODE, bool WIDE>
__device__ inline double row_mode_fused(const CartGeom &g, int blk, const float2 *kcol,
                                        const float2 *d, float2 *zhat, float2 *out,
                                        const float2 *zin, float2 *tile, float2 *twl, int *mrl) {
  const int tid = threadIdx.x;
  const int W = g.W;
  const long g0 = (long)blk * g.RB;
  const int nr = (int)min((long)g.RB, g.nrows_c - g0);
  const float2 *tw = stage_twiddles(g.pw, twl, tid, NT);
  const int *mrow = stage_mask_rows(g, g0, nr, mrl, tid, NT);
  __syncthreads();
  if constexpr (MODE == kRowAdjDense || MODE == kRowAdjCompact) {
    constexpr bool DENSE = MODE == kRowAdjDense;
    RowMaskLoad<DENSE> ld{g.mrows, mrow, g.rowinfo + g0, DENSE ? zin : zin + g0 * W,
                          W, g.C, g.H, g.centered};
    RowAdjStore st{zhat + g0 * W, W, g.centered};
    fft_io<NT, RTILE, false, true, true, WIDE>(tile, g.pw, nr, W, 1, -1.f, tid, tw, ld, st);
    return 0.0;
  } else {
    RowLoad ld{kcol + g0 * W, W};
    if constexpr (MODE == kRowApplyK) {
      RowApplyStore st{g.mrows, mrow, g.rowinfo + g0, out, W, g.C, g.H, g.centered, g.scale};
      fft_io<NT, RTILE, false, true, true, WIDE>(tile, g.pw, nr, W, 1, +1.f, tid, tw, ld, st);
      return 0.0;
    } else if constexpr (MODE == kRowNorm2) {
      RowNorm2Store st{g.mrows, mrow, W, g.centered, g.scale, 0.0};
      fft_io<NT, RTILE, false, true, true, WIDE>(tile, g.pw, nr, W, 1, +1.f, tid, tw, ld, st);
      return st.acc;
    } else {
      RowResidualStore st{g.mrows, mrow, d + g0 * W, W, g.centered, g.scale, 0.0};
      fft_io<NT, RTILE, false, true, true, WIDE>(tile, g.pw, nr, W, 1, +1.f, tid, tw, ld, st);
      return st.acc;
    }
  }
}

}  // namespace avionic
