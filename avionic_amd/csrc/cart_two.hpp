// Two-stage Cartesian passes: transforms whose length is a product of two
// radices of at most 16 (FftPlan::ra >= rb): every supported length below 125 and
// 53 of the 69 from 64 to 256.
//
// Stage a takes elements j + r rb (r < ra) of butterfly j < rb, stage b
// elements j + r ra (r < rb) of butterfly j < ra, which are also its output
// positions; between the stages the values cross the LDS tile once.  A lane is
// one (column, butterfly) or (row, butterfly) pair of each stage, so no index
// is ever divided; a radix rb <= 8 lets a lane run up to two_most(rb)
// butterflies of stage b, which keeps every lane busy in stage a.  The radices
// are runtime values; a switch around each stage selects its butterfly
// (with_radix).
//
// What bounds them: at 256 x 256 the VALU issue of the butterflies; below that
// the chain load -> stage -> barrier -> stage of each coil.  Measured on MI355X
// against the passes that moved every coil through LDS on a runtime plan (the
// operator calls before): K at 256 x 256 x 30 frames x 16 coils, acceleration
// 12, 291 -> 99 us (column pass 228 -> 49 us); K^H at 180 x 240 x 20 x 12,
// 191 -> 35 us; at 100 x 80 x 4 x 4, 71 -> 12.7 us; one eager TGV2 iteration
// at 256 x 256 x 25 x 12, 425 -> 184 us.
#pragma once

#include "cart_fused.hpp"

namespace avionic {

// Tile elements.  Columns: element i of column b at (i + i / ra) XB + b; the
// extra row after every ra elements puts the rows that a wave's lanes write
// together (ra apart) on different banks.  Rows: element i of row b at
// b row_pitch(W) + row_pos(i), one extra element in 16 for the same reason.
constexpr int kColTwoElems = 16 * 17 * 16;
constexpr int kRowTwoElems = 64 * 69;  // 64 rows of 64 (the largest: 32 of 128 and 16 of 256 less)
constexpr int kTwoMaxLen = kMaxRadix * kMaxRadix;

__device__ __forceinline__ int row_pos(int i) { return i + (i >> 4); }
__device__ __forceinline__ int row_pitch(int W) { return W + (W >> 4) + 1; }

// The radices and tile width of a column pass: runtime values (a switch around
// each stage), or 16 x 16 with 16 columns as constants.  The constant form has
// no switch, constant LDS offsets and fewer live scalars; length 256 is the
// most common one, and there it measured col_forward 296 -> 255 us and
// col_adjoint 400 -> 355 us (ICTGV2 256x256x30x16, 8 reconstructions).
struct TwoRt {
  int ra, rb, lxb;
  __device__ explicit TwoRt(const CartGeom &g) : ra(g.ph.ra), rb(g.ph.rb), lxb(g.lxb) {}
  template <class F> __device__ __forceinline__ void stage_a(F &&f) const { with_radix(ra, f); }
  template <class F> __device__ __forceinline__ void stage_b(F &&f) const { with_radix(rb, f); }
  static constexpr int most(int r) { return two_most(r); }
};
struct Two256 {
  static constexpr int ra = 16, rb = 16, lxb = 4;
  __device__ explicit Two256(const CartGeom &) {}
  template <class F> __device__ __forceinline__ void stage_a(F &&f) const { f(std::integral_constant<int, 16>{}); }
  template <class F> __device__ __forceinline__ void stage_b(F &&f) const { f(std::integral_constant<int, 16>{}); }
  static constexpr int most(int) { return 1; }
};

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
__device__ __forceinline__ int opaque_s(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// ------------------------------------------------------------ column forward
// Coils [c0, c1) of frame t, columns xbi XB ..: b1_c (u - usub), transform
// along y, sampled rows kept.  The image values of a lane's stage-a elements
// and the k-space offsets of its outputs stay in registers across the coils.
template <bool DELTA, class P>
__device__ __forceinline__ void col_forward_two(const CartGeom &g, int xbi, int t, int c0, int c1,
                                                const float2 *u, const float2 *usub,
                                                const float2 *b1, float2 *kcol, float2 *tile,
                                                float2 *twl, int *rml) {
  const int tid = threadIdx.x;
  const P plan(g);
  const int Ra = plan.ra, Rb = plan.rb, lxb = plan.lxb, H = Ra * Rb;
  int W = g.W;
  const long HW = (long)H * W;
  const bool cen = g.centered != 0;
  const float2 *tw = stage_twiddles(g.ph, twl, tid, NT);
  for (int i = tid; i < H; i += NT) rml[i] = g.rowmap[(long)t * H + i];
  const int b = tid & ((1 << lxb) - 1);
  int j = tid >> lxb;
  const int jq = NT >> lxb;  // stage b: butterflies j + q jq
  const int x = (xbi << lxb) + b;
  const int xc = x < W ? x : W - 1;  // lanes past the last column load in bounds, store nothing
  const int sx = cen ? wrap_half(xc, W) : xc;
  const int r0 = g.row_off[t], S = g.row_off[t + 1] - r0;
  float2 img[kMaxRadix];
  plan.stage_a([&](auto rc) {
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
  plan.stage_b([&](auto rc) {
    constexpr int R = decltype(rc)::value;
#pragma unroll
    for (int q = 0; q < P::most(R); ++q)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int jj = j + q * jq, i = jj + r * Ra;
        const int k = jj < Ra && x < W ? rml[cen ? wrap_half(i, H) : i] : -1;
        ko[q * R + r] = k >= 0 ? __umul24((unsigned)k, (unsigned)W) + (unsigned)x : kNoRow;
      }
  });
  for (int c = c0; c < c1; ++c) {
    j = opaque(j);
    W = opaque_s(W);
    const float2 *bc = b1 + c * HW;
    float2 *kc = kcol + ((long)g.C * r0 + (long)c * S) * W;
    plan.stage_a([&](auto rc) {
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
        float2 *p = tile + ((j * (R + 1)) << lxb) + b;
#pragma unroll
        for (int r = 0; r < R; ++r) p[r << lxb] = v[r];
      }
    });
    __syncthreads();
    plan.stage_b([&](auto rc) {
      constexpr int R = decltype(rc)::value;
      const int pitch = (Ra + 1) << lxb;
#pragma unroll
      for (int q = 0; q < P::most(R); ++q) {
        const int jj = j + q * jq;
        if (jj < Ra) {
          float2 v[R];
          const float2 *p = tile + (jj << lxb) + b;
#pragma unroll
          for (int r = 0; r < R; ++r) v[r] = p[r * pitch];
#pragma unroll
          for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * jj], +1.f);
          Dft<R>::run(v, +1.f);
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (ko[q * R + r] != kNoRow) gst(kc, ko[q * R + r], v[r]);
        }
      }
    });
    __syncthreads();
  }
}

// ------------------------------------------------------------ column adjoint
// Frame t, columns xbi XB ..: transform of the sampled rows along y, times
// conj(b1_c), summed over the coils in registers.  The coil-map values of a
// lane's outputs are loaded before its stage-b reads.  G groups of NT lanes
// each take a contiguous share of the coils on a tile of their own (`elems`
// apart) and add their sums in group order at the end.
template <class P, int G>
__device__ __forceinline__ void col_adjoint_two(const CartGeom &g, int xbi, int t,
                                                const float2 *zhat, const float2 *b1, float2 *out,
                                                float2 *tile, int elems, float2 *twl, int *rml) {
  const int tid = G > 1 ? threadIdx.x & (NT - 1) : threadIdx.x;
  const int grp = G > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
  float2 *const tiles = tile;
  tile += grp * elems;
  const P plan(g);
  const int Ra = plan.ra, Rb = plan.rb, lxb = plan.lxb, H = Ra * Rb;
  int W = g.W;
  const long HW = (long)H * W;
  const bool cen = g.centered != 0;
  const float2 *tw = stage_twiddles(g.ph, twl, threadIdx.x, NT * G);
  for (int i = threadIdx.x; i < H; i += NT * G) rml[i] = g.rowmap[(long)t * H + i];
  const int b = tid & ((1 << lxb) - 1);
  int j = tid >> lxb;
  const int jq = NT >> lxb;
  const int x = (xbi << lxb) + b;
  const int xc = x < W ? x : W - 1;
  const int r0 = g.row_off[t], S = g.row_off[t + 1] - r0;
  __syncthreads();
  unsigned ko[kMaxRadix];  // byte offsets
  plan.stage_a([&](auto rc) {
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
  const int share = (g.C + G - 1) / G;
  for (int ci = 0; ci < share; ++ci) {
    const int c = grp * share + ci;
    const bool live = G == 1 || c < g.C;  // uniform over a wave
    j = opaque(j);
    W = opaque_s(W);
    const float2 *bc = b1 + c * HW;
    const BoundedLoad zh(zhat + ((long)g.C * r0 + (long)c * S) * W, 8u * (unsigned)(S * W));
    plan.stage_a([&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (live && j < Rb) {
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = zh(ko[r]);
        __builtin_amdgcn_sched_barrier(0);
        Dft<R>::run(v, -1.f);
        float2 *p = tile + ((j * (R + 1)) << lxb) + b;
#pragma unroll
        for (int r = 0; r < R; ++r) p[r << lxb] = v[r];
      }
    });
    __syncthreads();
    plan.stage_b([&](auto rc) {
      constexpr int R = decltype(rc)::value;
      const int pitch = (Ra + 1) << lxb;
#pragma unroll
      for (int q = 0; q < P::most(R); ++q) {
        const int jj = j + q * jq;
        if (live && jj < Ra) {
          float2 m[R], v[R];
          const ImageCol<R> ic(jj, Ra, H, W, xc, cen);
#pragma unroll
          for (int r = 0; r < R; ++r) m[r] = ic.load(bc, r);
          __builtin_amdgcn_sched_barrier(0);
          const float2 *p = tile + (jj << lxb) + b;
#pragma unroll
          for (int r = 0; r < R; ++r) v[r] = p[r * pitch];
#pragma unroll
          for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * jj], -1.f);
          Dft<R>::run(v, -1.f);
#pragma unroll
          for (int r = 0; r < R; ++r) acc[q * R + r] = cadd(acc[q * R + r], cmulc(m[r], v[r]));
        }
      }
    });
    __syncthreads();
  }
  if constexpr (G > 1) {
    // every group's sums to its tile, then each group finishes its part
    plan.stage_b([&](auto rc) {
      constexpr int R = decltype(rc)::value;
#pragma unroll
      for (int q = 0; q < P::most(R); ++q) {
        const int jj = j + q * jq;
        if (jj < Ra)
#pragma unroll
          for (int r = 0; r < R; ++r) tile[((jj + r * Ra) << lxb) + b] = acc[q * R + r];
      }
    });
    __syncthreads();
    plan.stage_b([&](auto rc) {
      constexpr int R = decltype(rc)::value;
#pragma unroll
      for (int q = 0; q < P::most(R); ++q) {
        const int jj = j + q * jq;
        if (jj < Ra && x < W) {
          const ImageCol<R> ic(jj, Ra, H, W, xc, cen);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (r % G != grp) continue;
            const float2 *p = tiles + ((jj + r * Ra) << lxb) + b;
            float2 a = p[0];
#pragma unroll
            for (int k = 1; k < G; ++k) a = cadd(a, p[k * elems]);
            ic.store(out + t * HW, r, cscale(a, g.scale));
          }
        }
      }
    });
    return;
  }
  plan.stage_b([&](auto rc) {
    constexpr int R = decltype(rc)::value;
#pragma unroll
    for (int q = 0; q < P::most(R); ++q) {
      const int jj = j + q * jq;
      if (jj < Ra && x < W) {
        const ImageCol<R> ic(jj, Ra, H, W, xc, cen);
#pragma unroll
        for (int r = 0; r < R; ++r) ic.store(out + t * HW, r, cscale(acc[q * R + r], g.scale));
      }
    }
  });
}

// ------------------------------------------------------------------ row pass
// g.RB sampled rows per block; 2^lja lanes per row in the radix-ra stages and
// 2^ljb in the radix-rb ones (butterfly fastest, so that the loads of a row are
// contiguous).  The modes that end in k-space run the forward transform; the
// dual update keeps M z of a lane's outputs in registers, where they are the
// inputs of its first inverse butterfly: the centring shifts of K and K^H
// cancel, and the inverse runs the radices in the opposite order (rb, then
// ra).  The adjoint modes load M z there instead.
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
  const long g0 = (long)blk * g.RB;
  const int nr = (int)min((long)g.RB, g.nrows_c - g0);
  const float2 *tw = stage_twiddles(g.pw, twl, tid, NT);
  // stage a: butterfly ja of row ba; stage b: butterfly jb of rows bb + q bq.
  // Lanes past the last row work on it and store nothing.
  const int ja = tid & ((1 << g.lja) - 1), ba = tid >> g.lja;
  const int jb = tid & ((1 << g.ljb) - 1), bb = tid >> g.ljb, bq = NT >> g.ljb;
  const int nq = g.RB / bq;
  const int pitch = row_pitch(W);
  auto kx_of = [&](int i) { return cen ? wrap_half(i, W) : i; };
  double acc = 0.0;
  if (FWD) {
    with_radix(Ra, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (ja < Rb) {
        float2 v[R];
        const unsigned o = (unsigned)(min(ba, nr - 1) * W + ja);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = gld(kcol + g0 * W, o + (unsigned)(r * Rb));
        __builtin_amdgcn_sched_barrier(0);
        Dft<R>::run(v, +1.f);
        float2 *row = tile + ba * pitch;
#pragma unroll
        for (int r = 0; r < R; ++r) row[row_pos(ja * R + r)] = v[r];
      }
    });
  }
  __syncthreads();
  // forward stage b (or the adjoint's load) and inverse stage b, both radix rb
  // on the elements jb + r ra
  with_radix(Rb, [&](auto rc) {
    constexpr int R = decltype(rc)::value, Q = two_most(R);
    float2 v[Q][R];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int b = bb + q * bq, bc = min(b, nr - 1);
      if (q < nq && jb < Ra) {
        const int4 ri = g.rowinfo[g0 + bc];
        const unsigned mbase = (unsigned)(ri.z * W), rbase = (unsigned)(bc * W);
        const long dense = (((long)ri.x * g.C + ri.y) * g.H + ri.w) * W;
        float mk[R];
#pragma unroll
        for (int r = 0; r < R; ++r) mk[r] = gld(g.mrows, mbase + (unsigned)kx_of(jb + r * Ra));
        if constexpr (!FWD) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int kx = kx_of(jb + r * Ra);
            v[q][r] = MODE == kRowAdjDense ? zin[dense + kx] : gld(zin + g0 * W, rbase + (unsigned)kx);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int r = 0; r < R; ++r) v[q][r] = cscale(v[q][r], mk[r]);
        } else {
          constexpr bool Z = MODE == kRowDualUpdate, D = Z || MODE == kRowResidual;
          float2 zz[Z ? R : 1], dd[D ? R : 1];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const unsigned gi = rbase + (unsigned)kx_of(jb + r * Ra);
            if (Z) zz[r] = gld(z + g0 * W, gi);
            if (D) dd[r] = gld(d + g0 * W, gi);
          }
          __builtin_amdgcn_sched_barrier(0);
          const float2 *row = tile + b * pitch;
#pragma unroll
          for (int r = 0; r < R; ++r) v[q][r] = row[row_pos(jb + r * Ra)];
#pragma unroll
          for (int r = 1; r < R; ++r) v[q][r] = twiddle(v[q][r], tw[r * jb], +1.f);
          Dft<R>::run(v[q], +1.f);
          float sigma = 0.f, inv = 0.f;
          if (Z) {
            sigma = (float)sc->sigma;
            inv = (float)(1.0 / (1.0 + sc->sigma / sc->lambda));
          }
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int kx = kx_of(jb + r * Ra);
            const float2 val = cscale(v[q][r], g.scale * mk[r]);
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
              v[q][r] = cscale(zn, mk[r]);
            }
          }
        }
      }
    }
    if constexpr (INV) {
      if (MODE == kRowDualUpdate) __syncthreads();  // every lane has read the forward exchange
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (q < nq && jb < Ra) {
          Dft<R>::run(v[q], -1.f);
          float2 *row = tile + (bb + q * bq) * pitch;
#pragma unroll
          for (int r = 0; r < R; ++r) row[row_pos(jb * R + r)] = v[q][r];
        }
    }
  });
  if constexpr (INV) {
    __syncthreads();
    with_radix(Ra, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      if (ja < Rb) {
        float2 v[R];
        const float2 *row = tile + ba * pitch;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = row[row_pos(ja + r * Rb)];
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twiddle(v[r], tw[r * ja], -1.f);
        Dft<R>::run(v, -1.f);
        if (ba < nr)
#pragma unroll
          for (int r = 0; r < R; ++r)
            gst(zhat + g0 * W, (unsigned)(ba * W + kx_of(ja + r * Rb)), v[r]);
      }
    });
  }
  return acc;
}

// Twiddle and rowmap entries staged in LDS by the kernel of each kind.
__host__ __device__ constexpr int col_table_len(int kind) {
  return kind & 1 ? kTwoMaxLen : (kind == 2 ? kMaxFftLen : kMaxFftLenNarrow);
}
__host__ __device__ constexpr int row_table_len(int kind) {
  return kind == kRowTwo || kind == kRow256 ? kTwoMaxLen : (kind == kRowWide ? kMaxFftLen : kMaxFftLenNarrow);
}

}  // namespace avionic
