// In-LDS mixed-radix Stockham FFT for one workgroup (gfx950, 64-wide waves).
//
// A tile of `B` transforms of length L lives in LDS; element (b, i) sits at
// b*bstride + i*istride.  Each stage of radix R reads R inputs per butterfly
// into registers, twiddles them, runs an in-register DFT_R, synchronises, and
// writes the outputs to their Stockham positions in place; the next stage
// starts after a second barrier.  Lanes are mapped so that consecutive lanes
// touch consecutive LDS words (unit stride on whichever of b / i has it).
#pragma once

#include "common.hpp"

namespace avionic {

template <int R>
struct RootTable;  // cos / sin (2 pi m / R), m < R
template <> struct RootTable<3> {
  static constexpr float c[3] = {1.000000000e+00f, -5.000000000e-01f, -5.000000000e-01f};
  static constexpr float s[3] = {0.000000000e+00f, 8.660254038e-01f, -8.660254038e-01f};
};
template <> struct RootTable<5> {
  static constexpr float c[5] = {1.000000000e+00f, 3.090169944e-01f, -8.090169944e-01f, -8.090169944e-01f, 3.090169944e-01f};
  static constexpr float s[5] = {0.000000000e+00f, 9.510565163e-01f, 5.877852523e-01f, -5.877852523e-01f, -9.510565163e-01f};
};
template <> struct RootTable<7> {
  static constexpr float c[7] = {1.000000000e+00f, 6.234898019e-01f, -2.225209340e-01f, -9.009688679e-01f, -9.009688679e-01f, -2.225209340e-01f, 6.234898019e-01f};
  static constexpr float s[7] = {0.000000000e+00f, 7.818314825e-01f, 9.749279122e-01f, 4.338837391e-01f, -4.338837391e-01f, -9.749279122e-01f, -7.818314825e-01f};
};
template <> struct RootTable<11> {
  static constexpr float c[11] = {1.000000000e+00f, 8.412535328e-01f, 4.154150130e-01f, -1.423148383e-01f, -6.548607339e-01f, -9.594929736e-01f, -9.594929736e-01f, -6.548607339e-01f, -1.423148383e-01f, 4.154150130e-01f, 8.412535328e-01f};
  static constexpr float s[11] = {0.000000000e+00f, 5.406408175e-01f, 9.096319954e-01f, 9.898214419e-01f, 7.557495744e-01f, 2.817325568e-01f, -2.817325568e-01f, -7.557495744e-01f, -9.898214419e-01f, -9.096319954e-01f, -5.406408175e-01f};
};
template <> struct RootTable<13> {
  static constexpr float c[13] = {1.000000000e+00f, 8.854560257e-01f, 5.680647467e-01f, 1.205366803e-01f, -3.546048870e-01f, -7.485107482e-01f, -9.709418174e-01f, -9.709418174e-01f, -7.485107482e-01f, -3.546048870e-01f, 1.205366803e-01f, 5.680647467e-01f, 8.854560257e-01f};
  static constexpr float s[13] = {0.000000000e+00f, 4.647231720e-01f, 8.229838659e-01f, 9.927088741e-01f, 9.350162427e-01f, 6.631226582e-01f, 2.393156643e-01f, -2.393156643e-01f, -6.631226582e-01f, -9.350162427e-01f, -9.927088741e-01f, -8.229838659e-01f, -4.647231720e-01f};
};
// exp(sign * i * theta) applied as (c, sign * s).
__device__ inline float2 crot(float2 a, float c, float s, float sign) {
  float ss = sign * s;
  return make_float2(a.x * c - a.y * ss, a.x * ss + a.y * c);
}

// 4-point DFT, X[k] = sum_n x[n] exp(sign 2 pi i n k / 4).
__device__ inline void dft4(float2 &x0, float2 &x1, float2 &x2, float2 &x3, float sign) {
  float2 a = cadd(x0, x2), b = csub(x0, x2), c = cadd(x1, x3), d = csub(x1, x3);
  float2 di = make_float2(-sign * d.y, sign * d.x);  // d * (sign i)
  x0 = cadd(a, c);
  x2 = csub(a, c);
  x1 = cadd(b, di);
  x3 = csub(b, di);
}

template <int R>
struct Dft {
  // Odd radix via conjugate pairs: X_r = v0 + sum_{q<=(R-1)/2}
  //   (v_q + v_{R-q}) cos(2 pi q r / R) + sign i (v_q - v_{R-q}) sin(2 pi q r / R).
  __device__ static inline void run(float2 *v, float sign) {
    constexpr int Hh = (R - 1) / 2;
    float2 sp[Hh], sm[Hh];
#pragma unroll
    for (int q = 1; q <= Hh; ++q) {
      sp[q - 1] = cadd(v[q], v[R - q]);
      sm[q - 1] = csub(v[q], v[R - q]);
    }
    float2 o0 = v[0];
#pragma unroll
    for (int q = 0; q < Hh; ++q) o0 = cadd(o0, sp[q]);
#pragma unroll
    for (int r = 1; r <= Hh; ++r) {
      float ar = v[0].x, ai = v[0].y, br = 0.f, bi = 0.f;
#pragma unroll
      for (int q = 1; q <= Hh; ++q) {
        const int m = (q * r) % R;
        const float c = RootTable<R>::c[m], sn = RootTable<R>::s[m];
        ar += sp[q - 1].x * c;
        ai += sp[q - 1].y * c;
        br += sm[q - 1].x * sn;
        bi += sm[q - 1].y * sn;
      }
      // sign i (br + i bi) = (-sign bi, sign br)
      v[r] = make_float2(ar - sign * bi, ai + sign * br);
      v[R - r] = make_float2(ar + sign * bi, ai - sign * br);
    }
    v[0] = o0;
  }
};

template <>
struct Dft<2> {
  __device__ static inline void run(float2 *v, float) {
    float2 a = v[0];
    v[0] = cadd(a, v[1]);
    v[1] = csub(a, v[1]);
  }
};

template <>
struct Dft<4> {
  __device__ static inline void run(float2 *v, float sign) { dft4(v[0], v[1], v[2], v[3], sign); }
};

template <>
struct Dft<8> {
  // radix-2 split of two 4-point DFTs.
  __device__ static inline void run(float2 *v, float sign) {
    float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4(e0, e1, e2, e3, sign);
    dft4(o0, o1, o2, o3, sign);
    const float h = 0.70710678118654752f;
    o1 = crot(o1, h, h, sign);
    o2 = make_float2(-sign * o2.y, sign * o2.x);
    o3 = crot(o3, -h, h, sign);
    v[0] = cadd(e0, o0); v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1); v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2); v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3); v[7] = csub(e3, o3);
  }
};

template <>
struct Dft<16> {
  // 4 x 4: n = 4 n1 + n2, k = k1 + 4 k2.
  __device__ static inline void run(float2 *v, float sign) {
    float2 a[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
      a[n2][0] = v[n2]; a[n2][1] = v[4 + n2]; a[n2][2] = v[8 + n2]; a[n2][3] = v[12 + n2];
      dft4(a[n2][0], a[n2][1], a[n2][2], a[n2][3], sign);
    }
    // twiddles w16^(n2 k1)
    const float c1 = 0.92387953251128674f, s1 = 0.38268343236508978f;
    const float h = 0.70710678118654752f;
    a[1][1] = crot(a[1][1], c1, s1, sign);
    a[1][2] = crot(a[1][2], h, h, sign);
    a[1][3] = crot(a[1][3], s1, c1, sign);
    a[2][1] = crot(a[2][1], h, h, sign);
    a[2][2] = make_float2(-sign * a[2][2].y, sign * a[2][2].x);
    a[2][3] = crot(a[2][3], -h, h, sign);
    a[3][1] = crot(a[3][1], s1, c1, sign);
    a[3][2] = crot(a[3][2], -h, h, sign);
    a[3][3] = crot(a[3][3], -c1, -s1, sign);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      float2 b0 = a[0][k1], b1 = a[1][k1], b2 = a[2][k1], b3 = a[3][k1];
      dft4(b0, b1, b2, b3, sign);
      v[k1] = b0; v[k1 + 4] = b1; v[k1 + 8] = b2; v[k1 + 12] = b3;
    }
  }
};

template <>
struct Dft<1> {
  __device__ static inline void run(float2 *, float) {}
};

// Composite radix N = P Q, P and Q coprime, by the prime-factor mapping:
// inputs at (Q n1 + P n2) mod N, outputs at the k with k = k1 mod P and
// k = k2 mod Q, so that no twiddles stand between the two factors.
template <int P, int Q>
struct DftPfa {
  static constexpr int N = P * Q;
  __host__ __device__ static constexpr int out_index(int k1, int k2) {
    for (int k = 0; k < N; ++k)
      if (k % P == k1 && k % Q == k2) return k;
    return 0;
  }
  __device__ static inline void run(float2 *v, float sign) {
    float2 a[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1) a[n2][n1] = v[(Q * n1 + P * n2) % N];
      Dft<P>::run(a[n2], sign);
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      float2 b[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) b[n2] = a[n2][k1];
      Dft<Q>::run(b, sign);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) v[out_index(k1, k2)] = b[k2];
    }
  }
};
template <> struct Dft<6> : DftPfa<2, 3> {};
template <> struct Dft<10> : DftPfa<2, 5> {};
template <> struct Dft<12> : DftPfa<4, 3> {};
template <> struct Dft<14> : DftPfa<2, 7> {};
template <> struct Dft<15> : DftPfa<3, 5> {};

template <>
struct Dft<9> {
  // 3 x 3: n = 3 n1 + n2, k = k1 + 3 k2, twiddles w9^(n2 k1) between.
  __device__ static inline void run(float2 *v, float sign) {
    float2 a[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
      a[n2][0] = v[n2]; a[n2][1] = v[3 + n2]; a[n2][2] = v[6 + n2];
      Dft<3>::run(a[n2], sign);
    }
    a[1][1] = crot(a[1][1], 0.76604444311897801f, 0.64278760968653925f, sign);
    a[1][2] = crot(a[1][2], 0.17364817766693041f, 0.98480775301220802f, sign);
    a[2][1] = crot(a[2][1], 0.17364817766693041f, 0.98480775301220802f, sign);
    a[2][2] = crot(a[2][2], -0.93969262078590832f, 0.34202014332566888f, sign);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      float2 b[3] = {a[0][k1], a[1][k1], a[2][k1]};
      Dft<3>::run(b, sign);
      v[k1] = b[0]; v[k1 + 3] = b[1]; v[k1 + 6] = b[2];
    }
  }
};

// Calls f(std::integral_constant<int, R>) for a runtime radix 1 .. kMaxRadix.
constexpr int kMaxRadix = 16;
template <class F>
__device__ __forceinline__ void with_radix(int R, F &&f) {
  switch (R) {
    case 16: f(std::integral_constant<int, 16>{}); break;
    case 15: f(std::integral_constant<int, 15>{}); break;
    case 14: f(std::integral_constant<int, 14>{}); break;
    case 13: f(std::integral_constant<int, 13>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 11: f(std::integral_constant<int, 11>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    default: f(std::integral_constant<int, 1>{}); break;
  }
}

// a / n for 0 <= a < 2^13, 1 <= n: folded where n is a constant, else one
// reciprocal (its error is far below the 0.5 / n that separates a + 0.5 from
// the next multiple of n).
__device__ __forceinline__ int small_div(int a, int n) {
  if (__builtin_constant_p(n)) return a / n;
  return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)n));
}
// Butterfly j of transform b from a lane's index: BFAST (B a power of two)
// takes consecutive transforms on consecutive lanes, else consecutive
// butterflies.
template <bool BFAST>
__device__ __forceinline__ void butterfly_of(int idx, int nbf, int B, int &b, int &j) {
  if (BFAST) {
    b = idx & (B - 1);
    j = idx >> (31 - __clz(B));
  } else {
    b = small_div(idx, nbf);
    j = idx - b * nbf;
  }
}

// ---------------------------------------------------------------------------
// Fused transforms: the first stage may take its inputs from a load functor
// (global memory) instead of LDS, and the last stage may hand its outputs to
// a store functor instead of writing LDS.  Only the exchanges between stages
// touch LDS.  `tw` may point to LDS (a per-block copy of the twiddles).
//
//   ld(b, i, slot) -> float2  input element i of transform b   (natural order)
//   st(b, i, v, slot)        output element i of transform b   (natural order)
// The lane -> (b, j) mapping of a stage is the same for every call with the
// same plan and B, so a store functor may keep per-lane state across calls:
// `slot` (a compile-time constant once the stage is unrolled) numbers the
// outputs a lane produces, at most kMaxSlots of them.

template <int R, int NT, int EMAX, bool BFAST, bool FROMG, bool TOG, class LD, class ST>
__device__ __forceinline__ void fft_stage_io(float2 *buf, int L, int B, int bstride, int istride, int Ns,
                                    float sign, const float2 *__restrict__ tw, int tid, LD &ld,
                                    ST &st) {
  constexpr int MAXB = (EMAX / R + NT - 1) / NT;
  asm volatile("" : "+v"(tid));
  const int nbf = L / R;
  const int total = nbf * B;
  const int twstep = L / (Ns * R);
  const int rstride = nbf * istride;
  float2 v[MAXB][R];
#pragma unroll
  for (int c = 0; c < MAXB; ++c) {
    const int idx = tid + c * NT;
    if (idx < total) {
      int b, j;
      butterfly_of<BFAST>(idx, nbf, B, b, j);
      const int m = Ns > 1 ? small_div(j, Ns) : j, k = j - m * Ns;
      if (FROMG) {
#pragma unroll
        for (int r = 0; r < R; ++r) v[c][r] = ld(b, j + r * nbf, c * R + r);
      } else {
        const int base = b * bstride + j * istride;
#pragma unroll
        for (int r = 0; r < R; ++r) v[c][r] = buf[base + r * rstride];
      }
      if (Ns > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          float2 w = tw[r * k * twstep];
          w.y = -sign * w.y;
          v[c][r] = cmul(v[c][r], w);
        }
      }
      Dft<R>::run(v[c], sign);
    }
  }
  if (!FROMG && !TOG) __syncthreads();  // in place: all reads before any write
#pragma unroll
  for (int c = 0; c < MAXB; ++c) {
    const int idx = tid + c * NT;
    if (idx < total) {
      int b, j;
      butterfly_of<BFAST>(idx, nbf, B, b, j);
      const int m = Ns > 1 ? small_div(j, Ns) : j, k = j - m * Ns;
      const int o = m * Ns * R + k;
      if (TOG) {
#pragma unroll
        for (int r = 0; r < R; ++r) st(b, o + r * Ns, v[c][r], c * R + r);
      } else {
        const int base = b * bstride + o * istride;
        const int ostride = Ns * istride;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[base + r * ostride] = v[c][r];
      }
    }
  }
  if (!TOG) __syncthreads();
}

template <int NT, int EMAX, bool BFAST, bool FROMG, bool TOG, int WIDE, class LD, class ST>
__device__ __forceinline__ void fft_stage_io_dispatch(int R, float2 *buf, int L, int B, int bstride,
                                             int istride, int Ns, float sign, const float2 *tw,
                                             int tid, LD &ld, ST &st) {
  // (written out: through with_radix's closure the functors' per-lane arrays
  // stay in scratch memory)
#define AV_CASE(r)                                                                            \
  if constexpr (plan_radix(r, WIDE == kPlanWide))                                             \
  fft_stage_io<r, NT, EMAX, BFAST, FROMG, TOG>(buf, L, B, bstride, istride, Ns, sign, tw, tid, \
                                               ld, st)
  switch (R) {
    case 16: AV_CASE(16); break;
    case 15: AV_CASE(15); break;
    case 14: AV_CASE(14); break;
    case 13: AV_CASE(13); break;
    case 12: AV_CASE(12); break;
    case 11: AV_CASE(11); break;
    case 10: AV_CASE(10); break;
    case 9: AV_CASE(9); break;
    case 8: AV_CASE(8); break;
    case 7: AV_CASE(7); break;
    case 6: AV_CASE(6); break;
    case 5: AV_CASE(5); break;
    case 4: AV_CASE(4); break;
    case 3: AV_CASE(3); break;
    case 2: AV_CASE(2); break;
    default: AV_CASE(1); break;
  }
#undef AV_CASE
}
// Two-stage transforms (plan_kind kPlanTwo) whose lanes hold at most one butterfly of each stage
// (B ra <= NT): any radix up to 16 with one butterfly's registers.
template <int NT, bool BFAST, bool FROMG, bool TOG, class LD, class ST>
__device__ __forceinline__ void fft_stage_one(int R, float2 *buf, int L, int B, int bstride, int istride,
                                     int Ns, float sign, const float2 *tw, int tid, LD &ld,
                                     ST &st) {
#define AV_CASE(r)                                                                               \
  fft_stage_io<r, NT, r * NT, BFAST, FROMG, TOG>(buf, L, B, bstride, istride, Ns, sign, tw, tid, \
                                                 ld, st)
  switch (R) {
    case 16: AV_CASE(16); break;
    case 15: AV_CASE(15); break;
    case 14: AV_CASE(14); break;
    case 13: AV_CASE(13); break;
    case 12: AV_CASE(12); break;
    case 11: AV_CASE(11); break;
    case 10: AV_CASE(10); break;
    case 9: AV_CASE(9); break;
    case 8: AV_CASE(8); break;
    case 7: AV_CASE(7); break;
    case 6: AV_CASE(6); break;
    case 5: AV_CASE(5); break;
    case 4: AV_CASE(4); break;
    case 3: AV_CASE(3); break;
    case 2: AV_CASE(2); break;
    default: AV_CASE(1); break;
  }
#undef AV_CASE
}

struct NoLoad {
  __device__ float2 operator()(int, int, int) const { return make_float2(0.f, 0.f); }
};
struct NoStore {
  __device__ void operator()(int, int, float2, int) {}
};

// Outputs per lane of one stage: max over a plan's radices of
// ceil(EMAX/R/NT) * R.
constexpr int max_slots(int emax, int nt, int kind) {
  if (kind == kPlanTwo) return kMaxRadix;
  int m = 0;
  for (int r = 2; r <= kMaxRadix; ++r) {
    if (!plan_radix(r, kind == kPlanWide)) continue;
    const int v = ((emax / r + nt - 1) / nt) * r;
    m = v > m ? v : m;
  }
  return m;
}

// Transform with optional global input / output.  With FROMG the LDS tile's
// previous contents may still be being read by other lanes: callers sync
// before re-using a tile.  With TOG the LDS tile is free once this returns
// (the last stage read it before the function's final store loop; lanes may
// still be reading it, so callers sync before writing the tile again).
template <int NT, int EMAX, bool BFAST, bool FROMG, bool TOG, int WIDE, class LD, class ST>
__device__ __forceinline__ void fft_io(float2 *buf, const FftPlan &p, int B, int bstride, int istride,
                              float sign, int tid, const float2 *tw, LD &ld, ST &st) {
  NoStore ns;
  NoLoad nl;
  if constexpr (WIDE == kPlanTwo) {
    fft_stage_one<NT, BFAST, FROMG, false>(p.ra, buf, p.L, B, bstride, istride, 1, sign, tw, tid,
                                           ld, ns);
    fft_stage_one<NT, BFAST, false, TOG>(p.rb, buf, p.L, B, bstride, istride, p.ra, sign, tw, tid,
                                         nl, st);
  } else {
  const int n = p.nx;  // at least 2
  fft_stage_io_dispatch<NT, EMAX, BFAST, FROMG, false, WIDE>(p.rx[0], buf, p.L, B, bstride, istride,
                                                       1, sign, tw, tid, ld, ns);
  int Ns = p.rx[0];
  for (int s = 1; s < n - 1; ++s) {
    fft_stage_io_dispatch<NT, EMAX, BFAST, false, false, WIDE>(p.rx[s], buf, p.L, B, bstride, istride,
                                                         Ns, sign, tw, tid, nl, ns);
    Ns *= p.rx[s];
  }
  fft_stage_io_dispatch<NT, EMAX, BFAST, false, TOG, WIDE>(p.rx[n - 1], buf, p.L, B, bstride, istride,
                                                     Ns, sign, tw, tid, nl, st);
  }
}

// A plan known at compile time: length L = R0 R1 R2, stages in that order
// (R2 = 1: two stages).  fft_io_ct runs the stages fft_io runs on
// a plan of the same radices (same butterflies, twiddle indices
// and Stockham positions), with the length, the stage strides and, for
// BFAST, the transform count folded into constants: the per-element index
// divisions and remainders of the runtime plan become multiplies and shifts.
// `tw` holds the length-L twiddle table (stage_twiddles of that plan).
template <int L_, int R0_, int R1_, int R2_ = 1>
struct FftCt {
  static constexpr int L = L_, R0 = R0_, R1 = R1_, R2 = R2_;
  static_assert(R0_ * R1_ * R2_ == L_, "radices must multiply to the length");
};
// BMAX: most transforms per call (sizes the per-lane register arrays).  For
// BFAST the transform count is the constant BMAX and `B` is ignored.
template <int NT, class P, int BMAX, bool BFAST, bool FROMG, bool TOG, class LD, class ST>
__device__ __forceinline__ void fft_io_ct(float2 *buf, int B, int bstride, int istride, float sign,
                                          int tid, const float2 *tw, LD &ld, ST &st) {
  constexpr int L = P::L, E = L * BMAX;
  const int nb = BFAST ? BMAX : B;
  NoStore ns;
  NoLoad nl;
  if constexpr (P::R2 == 1) {
    fft_stage_io<P::R0, NT, E, BFAST, FROMG, false>(buf, L, nb, bstride, istride, 1, sign, tw, tid, ld, ns);
    fft_stage_io<P::R1, NT, E, BFAST, false, TOG>(buf, L, nb, bstride, istride, P::R0, sign, tw, tid, nl, st);
  } else {
    fft_stage_io<P::R0, NT, E, BFAST, FROMG, false>(buf, L, nb, bstride, istride, 1, sign, tw, tid, ld, ns);
    fft_stage_io<P::R1, NT, E, BFAST, false, false>(buf, L, nb, bstride, istride, P::R0, sign, tw, tid, nl, ns);
    fft_stage_io<P::R2, NT, E, BFAST, false, TOG>(buf, L, nb, bstride, istride, P::R0 * P::R1, sign, tw, tid, nl, st);
  }
}

// Copy a plan's twiddles to LDS (L <= kMaxFftLen) and return the LDS view.
__device__ inline const float2 *stage_twiddles(const FftPlan &p, float2 *lds, int tid, int nt) {
  for (int i = tid; i < p.L; i += nt) lds[i] = p.tw[i];
  return lds;
}

}  // namespace avionic
