// Two-stage Cartesian passes: transforms whose length is a product of two
// radices of at most 16 (FftPlan::ra, rb), i.e. nearly every length up to 256.
//
// Every lane runs at most one butterfly of each stage, so a lane is one
// (column, butterfly) or (row, butterfly) pair for the whole pass and no index
// is ever divided: stage 0 takes elements j + r rb (r < ra) of butterfly
// j < rb, stage 1 elements j + r ra (r < rb) of butterfly j < ra, which are
// also its output positions.  Between the stages the values cross the LDS
// tile once.  The radices are runtime values; a switch around each stage
// selects its butterfly (with_radix).
//
// What bounds them: at 256 x 256 the VALU issue of the butterflies; below that
// the chain load -> stage -> barrier -> stage of each coil.  Measured on MI355X
// against the passes that moved every coil through LDS on a runtime plan (the
// operator calls before): K at 256 x 256 x 30 frames x 16 coils, acceleration
// 12, 291 -> 110 us (column pass 228 -> 62 us); K^H at 180 x 240 x 20 x 12,
// 191 -> 53 us; at 100 x 80 x 4 x 4, 71 -> 16.5 us; one eager TGV2 iteration
// at 256 x 256 x 25 x 12, 425 -> 220 us.
#pragma once

#include "cart_fused.hpp"

namespace avionic {

// Tile elements.  Columns: element i of column b at (i + i / ra) XB + b; the
// extra row after every ra elements puts the rows that a wave's lanes write
// together (ra apart) on different banks.  Rows: element i of row b at
// b row_pitch(W) + row_pos(i), one extra element in 16 for the same reason.
constexpr int kColTwoElems = 16 * 17 * 16;
constexpr int kRowTwoElems = 16 * 273;
constexpr int kTwoMaxLen = kMaxRadix * kMaxRadix;

__device__ __forceinline__ int row_pos(int i) { return i + (i >> 4); }
__device__ __forceinline__ int row_pitch(int W) { return W + (W >> 4) + 1; }

// v *= exp(sign i theta), tw = exp(-i theta)
__device__ __forceinline__ float2 twiddle(float2 v, float2 tw, float sign) {
  return sign > 0.f ? cmulc(tw, v) : cmul(tw, v);
}

// Loads past `bytes` return zero (the buffer instruction's range check), so a
// row that is not sampled needs no branch, no select and no memory traffic.
constexpr unsigned kNoRow = 0x7ffffff8u;
struct BoundedLoad {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ BoundedLoad(const float2 *p, unsigned bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<float2 *>(p), 0, (int)bytes, 0x00020000)) {}
  __device__ float2 operator()(unsigned byte) const {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)byte, 0, 0));
  }
};

// Image element j + r N (r < R) of column x: the centring shift by half of an
// even radix's length is a rotation of r, so the lane's offset is the same for
// every r and the rest is uniform, part of the scalar base.
template <int R>
struct ImageCol {
  int L, W;
  bool cen;
  unsigned o;
  int j, N, x;
  __device__ ImageCol(int j_, int N_, int L_, int W_, int x_, bool cen_)
      : L(L_), W(W_), cen(cen_), o(__umul24((unsigned)j_, (unsigned)W_) + (unsigned)x_), j(j_),
        N(N_), x(x_) {}
  __device__ unsigned base(int r) const {
    if constexpr (R % 2 == 0) return (unsigned)((cen ? (r + R / 2) % R : r) * N * W);
    return 0u;
  }
  __device__ unsigned lane(int r) const {
    if constexpr (R % 2 == 0) return o;
    const int i = j + r * N;
    return __umul24((unsigned)(cen ? wrap_half(i, L) : i), (unsigned)W) + (unsigned)x;
  }
  __device__ float2 load(const float2 *p, int r) const { return gld(p + base(r), lane(r)); }
  __device__ void store(float2 *p, int r, float2 v) const { gst(p + base(r), lane(r), v); }
};

// Keeps the index arithmetic of a pass's sixteen radices inside its coil loop:
// hoisted, all of them would be live at once.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// ------------------------------------------------------------ column forward
// Coils [c0, c1) of frame t, columns xbi XB ..: b1_c (u - usub), transform
// along y, sampled rows kept.  The image values of a lane's stage-0 elements
// and the k-space offsets of its outputs stay in registers across the coils.
template <bool DELTA>
__device__ __forceinline__ void col_forward_two(const CartGeom &g, int xbi, int t, int c0, int c1,
                                                const float2 *u, const float2 *usub,
                                                const float2 *b1, float2 *kcol, float2 *tile,
                                                float2 *twl, int *rml) {
  const int tid = threadIdx.x;
  const int H = g.H, W = g.W, Ra = g.ph.ra, Rb = g.ph.rb;
  const long HW = (long)H * W;
  const bool cen = g.centered != 0;
  const float2 *tw = stage_twiddles(g.ph, twl, tid, NT);
  for (int i = tid; i < H; i += NT) rml[i] = g.rowmap[(long)t * H + i];
  const int b = tid & (g.XB - 1);
  int j = tid >> g.lxb;
  const int x = xbi * g.XB + b;
  const int xc = x < W ? x : W - 1;  // lanes past the last column load in bounds, store nothing
  const int sx = cen ? wrap_half(xc, W) : xc;
  const int r0 = g.row_off[t], S = g.row_off[t + 1] - r0;
  float2 img[kMaxRadix];
  with_radix(Ra, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    if (j < Rb) {
      const ImageCol<R> ic(j, Rb, H, W, sx, cen);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        img[r] = ic.load(u + t * HW, r);
        if (DELTA) img[r] = csub(img[r], ic.load(usub + t * HW, r));
      }
    }
  });
  __syncthreads();
  unsigned ko[kMaxRadix];
  with_radix(Rb, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = j + r * Ra;
      const int k = j < Ra && x < W ? rml[cen ? wrap_half(i, H) : i] : -1;
      ko[r] = k >= 0 ? __umul24((unsigned)k, (unsigned)W) + (unsigned)x : kNoRow;
    }
  });
  for (int c = c0; c < c1; ++c) {
    j = opaque(j);
    const float2 *bc = b1 + c * HW;
    float2 *kc = kcol + ((long)g.C * r0 + (long)c * S) * W;
    with_radix(Ra, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (j < Rb) {
        float2 v[R];
        const ImageCol<R> ic(j, Rb, H, W, sx, cen);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = ic.load(bc, r);
        __builtin_amdgcn_sched_barrier(0);  // every load issued before the first use
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = cmul(v[r], img[r]);
        Dft<R>::run(v, +1.f);
        float2 *p = tile + ((j * (R + 1)) << g.lxb) + b;
#pragma unroll
        for (int r = 0; r < R; ++r) p[r << g.lxb] = v[r];
      }
    });
    __syncthreads();
    with_radix(Rb, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (j < Ra) {
        float2 v[R];
        const float2 *p = tile + (j << g.lxb) + b;
        const int pitch = (Ra + 1) << g.lxb;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = p[r * pitch];
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * j], +1.f);
        Dft<R>::run(v, +1.f);
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (ko[r] != kNoRow) gst(kc, ko[r], v[r]);
      }
    });
    __syncthreads();
  }
}

// ------------------------------------------------------------ column adjoint
// Frame t, columns xbi XB ..: transform of the sampled rows along y, times
// conj(b1_c), summed over the coils in registers.  The coil-map values of a
// lane's outputs are loaded with the coil's k-space, ahead of both stages.
__device__ __forceinline__ void col_adjoint_two(const CartGeom &g, int xbi, int t,
                                                const float2 *zhat, const float2 *b1, float2 *out,
                                                float2 *tile, float2 *twl, int *rml) {
  const int tid = threadIdx.x;
  const int H = g.H, W = g.W, Ra = g.ph.ra, Rb = g.ph.rb;
  const long HW = (long)H * W;
  const bool cen = g.centered != 0;
  const float2 *tw = stage_twiddles(g.ph, twl, tid, NT);
  for (int i = tid; i < H; i += NT) rml[i] = g.rowmap[(long)t * H + i];
  const int b = tid & (g.XB - 1);
  int j = tid >> g.lxb;
  const int x = xbi * g.XB + b;
  const int xc = x < W ? x : W - 1;
  const int r0 = g.row_off[t], S = g.row_off[t + 1] - r0;
  __syncthreads();
  unsigned ko[kMaxRadix];  // byte offsets
  with_radix(Ra, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = j + r * Rb;
      const int k = j < Rb ? rml[cen ? wrap_half(i, H) : i] : -1;
      ko[r] = k >= 0 ? 8u * (__umul24((unsigned)k, (unsigned)W) + (unsigned)xc) : kNoRow;
    }
  });
  float2 acc[kMaxRadix];
#pragma unroll
  for (int r = 0; r < kMaxRadix; ++r) acc[r] = czero();
  for (int c = 0; c < g.C; ++c) {
    j = opaque(j);
    const float2 *bc = b1 + c * HW;
    const BoundedLoad zh(zhat + ((long)g.C * r0 + (long)c * S) * W, 8u * (unsigned)(S * W));
    with_radix(Ra, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (j < Rb) {
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = zh(ko[r]);
        __builtin_amdgcn_sched_barrier(0);
        Dft<R>::run(v, -1.f);
        float2 *p = tile + ((j * (R + 1)) << g.lxb) + b;
#pragma unroll
        for (int r = 0; r < R; ++r) p[r << g.lxb] = v[r];
      }
    });
    __syncthreads();
    with_radix(Rb, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (j < Ra) {
        float2 m[R], v[R];
        const ImageCol<R> ic(j, Ra, H, W, xc, cen);
#pragma unroll
        for (int r = 0; r < R; ++r) m[r] = ic.load(bc, r);
        __builtin_amdgcn_sched_barrier(0);
        const float2 *p = tile + (j << g.lxb) + b;
        const int pitch = (Ra + 1) << g.lxb;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = p[r * pitch];
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * j], -1.f);
        Dft<R>::run(v, -1.f);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = cadd(acc[r], cmulc(m[r], v[r]));
      }
    });
    __syncthreads();
  }
  with_radix(Rb, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    if (j < Ra && x < W) {
      const ImageCol<R> ic(j, Ra, H, W, xc, cen);
#pragma unroll
      for (int r = 0; r < R; ++r) ic.store(out + t * HW, r, cscale(acc[r], g.scale));
    }
  });
}

// ------------------------------------------------------------------ row pass
// g.RBT sampled rows per block, NT / RBT lanes per row (butterfly j fastest, so
// that the loads of a row are contiguous).  The modes that end in k-space run
// the forward transform; the dual update keeps M z of a lane's outputs in
// registers, where they are the inputs of its first inverse butterfly: the
// centring shifts of K and K^H cancel, and the inverse runs the radices in the
// opposite order (rb, then ra).  The adjoint modes load M z there instead.
template <int MODE>
__device__ __forceinline__ double row_two(const CartGeom &g, int blk, const float2 *kcol,
                                          float2 *z, const float2 *d, float2 *zhat, float2 *out,
                                          const float2 *zin, const DevScalars *sc, float2 *tile,
                                          float2 *twl) {
  constexpr bool FWD = MODE != kRowAdjDense && MODE != kRowAdjCompact;
  constexpr bool INV = !FWD || MODE == kRowDualUpdate;
  const int tid = threadIdx.x;
  const int W = g.W, Ra = g.pw.ra, Rb = g.pw.rb;
  const bool cen = g.centered != 0;
  const long g0 = (long)blk * g.RBT;
  const int nr = (int)min((long)g.RBT, g.nrows_c - g0);
  const float2 *tw = stage_twiddles(g.pw, twl, tid, NT);
  const int j = tid & ((1 << g.ljw) - 1), b = tid >> g.ljw;
  const int bc = min(b, nr - 1);  // lanes past the last row work on it, store nothing
  const int4 ri = g.rowinfo[g0 + bc];
  const unsigned mbase = (unsigned)(ri.z * W);
  const unsigned rbase = (unsigned)(bc * W);
  const long dense = (((long)ri.x * g.C + ri.y) * g.H + ri.w) * W;
  float2 *row = tile + b * row_pitch(W);
  auto kx_of = [&](int i) { return cen ? wrap_half(i, W) : i; };
  double acc = 0.0;
  if (FWD) {
    with_radix(Ra, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (j < Rb) {
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = gld(kcol + g0 * W, rbase + (unsigned)(j + r * Rb));
        __builtin_amdgcn_sched_barrier(0);
        Dft<R>::run(v, +1.f);
#pragma unroll
        for (int r = 0; r < R; ++r) row[row_pos(j * R + r)] = v[r];
      }
    });
  }
  __syncthreads();
  // forward stage 1 (or the adjoint's load) and inverse stage 0, both radix rb
  // on the elements j + r ra
  with_radix(Rb, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    float2 v[R];
    if (j < Ra) {
      float mk[R];
#pragma unroll
      for (int r = 0; r < R; ++r) mk[r] = gld(g.mrows, mbase + (unsigned)kx_of(j + r * Ra));
      if constexpr (!FWD) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int kx = kx_of(j + r * Ra);
          v[r] = MODE == kRowAdjDense ? zin[dense + kx] : gld(zin + g0 * W, rbase + (unsigned)kx);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = cscale(v[r], mk[r]);
      } else {
        float2 zz[MODE == kRowDualUpdate ? R : 1], dd[MODE == kRowDualUpdate || MODE == kRowResidual ? R : 1];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const unsigned gi = rbase + (unsigned)kx_of(j + r * Ra);
          if (MODE == kRowDualUpdate) zz[r] = gld(z + g0 * W, gi);
          if (MODE == kRowDualUpdate || MODE == kRowResidual) dd[r] = gld(d + g0 * W, gi);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = row[row_pos(j + r * Ra)];
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * j], +1.f);
        Dft<R>::run(v, +1.f);
        float sigma = 0.f, inv = 0.f;
        if (MODE == kRowDualUpdate) {
          sigma = (float)sc->sigma;
          inv = (float)(1.0 / (1.0 + sc->sigma / sc->lambda));
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int kx = kx_of(j + r * Ra);
          const float2 val = cscale(v[r], g.scale * mk[r]);
          if (MODE == kRowApplyK) {
            if (b < nr) out[dense + kx] = val;
          } else if (MODE == kRowNorm2) {
            if (b < nr) acc += (double)cabs2(val);
          } else if (MODE == kRowResidual) {
            if (b < nr) acc += (double)cabs2(csub(val, dd[r]));
          } else {
            float2 zn = cadd(zz[r], cscale(val, sigma));
            zn = cscale(csub(zn, cscale(dd[r], sigma)), inv);
            if (b < nr) gst_stream(z + g0 * W, rbase + (unsigned)kx, zn);
            v[r] = cscale(zn, mk[r]);
          }
        }
      }
    }
    if constexpr (INV) {
      if (MODE == kRowDualUpdate) __syncthreads();  // every lane has read the forward exchange
      if (j < Ra) {
        Dft<R>::run(v, -1.f);
#pragma unroll
        for (int r = 0; r < R; ++r) row[row_pos(j * R + r)] = v[r];
      }
    }
  });
  if constexpr (INV) {
    __syncthreads();
    with_radix(Ra, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (j < Rb) {
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = row[row_pos(j + r * Rb)];
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * j], -1.f);
        Dft<R>::run(v, -1.f);
        if (b < nr)
#pragma unroll
          for (int r = 0; r < R; ++r)
            gst(zhat + g0 * W, rbase + (unsigned)kx_of(j + r * Rb), v[r]);
      }
    });
  }
  return acc;
}

// One kernel per kind of transform: two-stage, narrow or wide runtime plan.
enum ApiKind { kTwo = 0, kRt = 1, kRtWide = 2 };
inline int api_kind(const FftPlan &p) { return p.ra ? kTwo : (plan_is_wide(p) ? kRtWide : kRt); }
constexpr int api_table_len(int kind) {
  return kind == kTwo ? kTwoMaxLen : (kind == kRt ? kMaxFftLenNarrow : kMaxFftLen);
}

}  // namespace avionic
