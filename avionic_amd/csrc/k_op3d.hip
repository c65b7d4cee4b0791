// Volumetric Cartesian operator pair for TGV2_3D
// (CartesianOperator3D, cartesian_operator3d.cpp:64-345):
//   K  (image -> k-space): z_c = M . F^{+}(b1_c . u) / sqrt(N)
//   K^H (k-space -> image): u = sum_c conj(b1_c) . F^{-}(M . z_c) / sqrt(N)
// with 3D transforms over [depth][height][width] (F^{+}: e^{+i}, F^{-}:
// e^{-i}) and k-space stored coil-major [c][depth][height][width], as the
// reference stores it.  The reference's `centered` flag changes nothing in
// this operator (both branches run the same transform), so there is none here.
// Separable passes, each reading its first stage from global memory and writing
// its last stage there (44 MB per array at 128 x 112 x 48 x 8 coils: the passes
// are bound by memory traffic, so everything elementwise is folded into one):
//   x: b1_c (u - usub), rows along x           x^H: rows along x, conj(b1_c) coil sum
//   y: columns along y, in place               y^H: the same
//   z: columns along depth, then what the mode asks for: mask into k-space, the
//      z update and the adjoint's depth transform, or a sum of squares
// K is x, y, z; K^H is z^H, y^H, x^H; the dual update runs z and z^H in one
// kernel.  One iteration's data term is 5 passes for the 14 of separate
// expand / 2D transform / copy / depth / mask kernels: 240 -> 142 us.
#include <cmath>
#include <vector>

#include "cart_device.hpp"
#include "reg_device.hpp"
#include "solver.hpp"

namespace avionic {

namespace {

constexpr int kT3 = 256;

// out = in . mask (mask over one coil's N elements; null = ones)
__global__ __launch_bounds__(kT3) void k3_mask(const float2 *__restrict__ in,
                                               const float *__restrict__ mask,
                                               float2 *__restrict__ out, long N, long n) {
  for (long e = (long)blockIdx.x * kT3 + threadIdx.x; e < n; e += (long)gridDim.x * kT3)
    out[e] = mask ? cscale(in[e], mask[e % N]) : in[e];
}

constexpr int table3(int kind) { return kind == kPlanWide ? kMaxFftLen : kMaxFftLenNarrow; }

// Rows of the C volumes: block x takes rows [y0, y0 + RB) of the D H rows of
// coil blockIdx.y (x), or of every coil in turn (x^H).
struct V3 {
  int W, H, D, C;
  long N;  // W H D
};
struct XLoad {
  const float2 *u, *us, *b1;  // row y0
  int W;
  __device__ float2 operator()(int b, int i, int) const {
    const unsigned o = (unsigned)(b * W + i);
    const float2 bv = gld(b1, o), uv = gld(u, o);
    return cmul(bv, us ? csub(uv, gld(us, o)) : uv);
  }
};
struct XStore {
  float2 *out;
  int W;
  __device__ void operator()(int b, int i, float2 v, int) const { gst(out, (unsigned)(b * W + i), v); }
};
template <int KIND>
__global__ __launch_bounds__(kT3) void k3_x(V3 g, FftPlan px, int RB, const float2 *u,
                                            const float2 *usub, const float2 *b1, float2 *out) {
  __shared__ float2 tile[EMAX];
  __shared__ float2 twl[table3(KIND)];
  const int tid = threadIdx.x, y0 = blockIdx.x * RB;
  const long o = (long)y0 * g.W, oc = (long)blockIdx.y * g.N + o;
  const float2 *tw = stage_twiddles(px, twl, tid, kT3);
  __syncthreads();
  XLoad ld{u + o, usub ? usub + o : nullptr, b1 + oc, g.W};
  XStore st{out + oc, g.W};
  fft_io<kT3, EMAX, false, true, true, KIND>(tile, px, min(RB, g.H * g.D - y0), g.W, 1, +1.f, tid,
                                             tw, ld, st);
}

struct XAdjLoad {
  const float2 *in;
  int W;
  __device__ float2 operator()(int b, int i, int) const { return gld(in, (unsigned)(b * W + i)); }
};
// Each of the block's kXG waves runs its own rows tile over a contiguous share
// of the coils (the coils in one wave's sequence: 51 us at 128 x 112 x 48 x 8,
// four waves 36 us); a wave's sum stays in registers, one accumulator
// per output of the lane, and the waves' sums are added in order at the end.
constexpr int kXG = 4, kXLanes = kT3 / kXG, kXElems = EMAX / kXG;
template <int SLOTS>
struct XAdjStore {
  float2 acc[SLOTS];
  const float2 *b1;
  float2 *sum;  // LDS
  int W;
  bool live, last;
  __device__ void operator()(int b, int i, float2 v, int slot) {
    const unsigned o = (unsigned)(b * W + i);
    if (live) acc[slot] = cadd(acc[slot], cmulc(gld(b1, o), v));
    if (last) sum[o] = acc[slot];
  }
};
template <int KIND>
__global__ __launch_bounds__(kT3) void k3_x_adj(V3 g, FftPlan px, int RB, const float2 *in,
                                                const float2 *b1, float2 *img) {
  extern __shared__ float2 lds[];  // kXG transform tiles, kXG sums, RB W each
  __shared__ float2 twl[table3(KIND)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kXLanes);
  const int lane = threadIdx.x % kXLanes, y0 = blockIdx.x * RB, elems = RB * g.W;
  const int nr = min(RB, g.H * g.D - y0);
  const long o = (long)y0 * g.W;
  const float2 *tw = stage_twiddles(px, twl, threadIdx.x, kT3);
  __syncthreads();
  XAdjLoad ld{nullptr, g.W};
  constexpr int SLOTS = max_slots(kXElems, kXLanes, KIND);
  XAdjStore<SLOTS> st;
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) st.acc[k] = czero();
  st.sum = lds + (kXG + wave) * elems;
  st.W = g.W;
  const int share = (g.C + kXG - 1) / kXG;
  for (int ci = 0; ci < share; ++ci) {
    const int c = min(wave * share + ci, g.C - 1);
    ld.in = in + c * g.N + o;
    st.b1 = b1 + c * g.N + o;
    st.live = wave * share + ci < g.C;
    st.last = ci == share - 1;
    fft_io<kXLanes, kXElems, false, true, true, KIND>(lds + wave * elems, px, nr, g.W, 1, -1.f,
                                                      lane, tw, ld, st);
    __syncthreads();
  }
  const float2 *sum = lds + kXG * elems;
  for (int e = threadIdx.x; e < nr * g.W; e += kT3) {
    float2 a = sum[e];
#pragma unroll
    for (int k = 1; k < kXG; ++k) a = cadd(a, sum[k * elems + e]);
    gst(img + o, (unsigned)e, a);
  }
}

// Depth pass: block (columns p0 .. of the plane, coil).
enum DepthMode { kDApplyK = 0, kDDual = 1, kDNorm2 = 2, kDResidual = 3, kDAdjoint = 4 };
struct ZLoad {
  const float2 *in;  // coil volume, column p0
  int plane, np;
  __device__ float2 operator()(int b, int i, int) const {
    return gld(in, (unsigned)(i * plane + min(b, np - 1)));  // columns past the last: dropped
  }
};
struct ZMaskLoad {
  const float2 *in;
  const float *mask;
  int plane, np;
  __device__ float2 operator()(int b, int i, int) const {
    const unsigned o = (unsigned)(i * plane + min(b, np - 1));
    const float2 v = gld(in, o);
    return mask ? cscale(v, gld(mask, o)) : v;
  }
};
struct ZStore {
  float2 *out;
  int plane, np;
  float scale;
  __device__ void operator()(int b, int i, float2 v, int) const {
    if (b < np) gst(out, (unsigned)(i * plane + b), cscale(v, scale));
  }
};
// Output of K's depth transform: mask . scale . v into k-space, into the z
// update (M z to the tile of the adjoint's transform), or into a sum.
template <int MODE>
struct ZOut {
  const float *mask;
  float2 *out;      // kDApplyK: k-space; kDDual: z
  const float2 *d;  // kDDual, kDResidual
  float2 *tile2;
  int plane, np, XB;
  float scale, sigma, inv;
  double acc;
  __device__ void operator()(int b, int i, float2 v, int) {
    const unsigned o = (unsigned)(i * plane + min(b, np - 1));
    const float mk = mask ? gld(mask, o) : 1.f;
    const float2 val = cscale(cscale(v, scale), mk);
    if constexpr (MODE == kDApplyK) {
      if (b < np) gst(out, o, val);
    } else if constexpr (MODE == kDNorm2) {
      if (b < np) acc += (double)cabs2(val);
    } else if constexpr (MODE == kDResidual) {
      if (b < np) acc += (double)cabs2(csub(val, gld(d, o)));
    } else {
      // z = (z + sigma K u - sigma d) / (1 + sigma / lambda)  (tgv2_3d.cpp loop)
      float2 zz = cadd(gld(out, o), cscale(val, sigma));
      zz = cscale(csub(zz, cscale(gld(d, o), sigma)), inv);
      if (b < np) gst(out, o, zz);
      tile2[i * XB + b] = cscale(zz, mk);
    }
  }
};
template <int MODE, int KIND>
__global__ __launch_bounds__(kT3) void k3_z(V3 g, FftPlan pz, int XB, float scale, const float2 *in,
                                            const float *mask, float2 *out, const float2 *d,
                                            float2 *zhat, const DevScalars *sc, double *partial) {
  constexpr bool SUM = MODE == kDNorm2 || MODE == kDResidual;
  // L XB elements, twice for kDDual: a short depth leaves room for more blocks
  extern __shared__ float2 tile[];
  float2 *const tile2 = tile + pz.L * XB;
  __shared__ float2 twl[table3(KIND)];
  __shared__ double red[SUM ? kT3 : 1];
  const int tid = threadIdx.x, plane = g.W * g.H, p0 = blockIdx.x * XB, np = min(XB, plane - p0);
  const long oc = (long)blockIdx.y * g.N + p0;
  const float2 *tw = stage_twiddles(pz, twl, tid, kT3);
  __syncthreads();
  const float *mk = mask ? mask + p0 : nullptr;
  if constexpr (MODE == kDAdjoint) {
    ZMaskLoad ld{in + oc, mk, plane, np};
    ZStore st{zhat + oc, plane, np, scale};
    fft_io<kT3, EMAX, true, true, true, KIND>(tile, pz, XB, 1, XB, -1.f, tid, tw, ld, st);
    return;
  } else {
    ZLoad ld{in + oc, plane, np};
    ZOut<MODE> st;
    st.mask = mk;
    st.out = out ? out + oc : nullptr;
    st.d = d ? d + oc : nullptr;
    st.tile2 = tile2;
    st.plane = plane;
    st.np = np;
    st.XB = XB;
    st.scale = scale;
    st.acc = 0.0;
    if (MODE == kDDual) {
      st.sigma = (float)sc->sigma;
      st.inv = (float)(1.0 / (1.0 + sc->sigma / sc->lambda));
    }
    fft_io<kT3, EMAX, true, true, true, KIND>(tile, pz, XB, 1, XB, +1.f, tid, tw, ld, st);
    if constexpr (MODE == kDDual) {
      __syncthreads();  // tile2 holds M z of the block's columns
      NoLoad nl;
      ZStore st2{zhat + oc, plane, np, scale};
      fft_io<kT3, EMAX, true, false, true, KIND>(tile2, pz, XB, 1, XB, -1.f, tid, tw, nl, st2);
    }
    if constexpr (SUM) {
      const double a = block_sum(st.acc, red);
      if (tid == 0) partial[(long)blockIdx.y * gridDim.x + blockIdx.x] = a;
    }
  }
}

int blocks_for(long n) { return (int)std::max<long>(1, std::min<long>(1024, (n + kT3 - 1) / kT3)); }

class CartesianOperator3D : public Operator {
 public:
  CartesianOperator3D(int W_, int H_, int D_, int C_, const float *mask) {
    W = W_; H = H_; T = D_; C = C_;
    AV_CHECK(W > 0 && H > 0 && T > 0 && C > 0, "invalid operator dimensions");
    check_grid(Grid3{W, H, T, (long)W * H * T});
    AV_CHECK((long)C * N() < (1L << 31), "coils x volume exceeds 2^31 elements");
    const long n = N();
    if (mask) {
      std::vector<float> hm((size_t)n);
      AV_HIP(hipMemcpy(hm.data(), mask, sizeof(float) * n, hipMemcpyDeviceToHost));
      mask_norm2_ = 0.0;
      for (float v : hm) mask_norm2_ += (double)v * v;
      mask_.ensure(sizeof(float) * n);
      AV_HIP(hipMemcpy(mask_.p, hm.data(), sizeof(float) * n, hipMemcpyHostToDevice));
    }
    make_fft_plan(W, pw_, &twx_.p);
    make_fft_plan(H, ph_, &twy_.p);
    make_fft_plan(T, pd_, &twz_.p);
    AV_HIP(hipStreamSynchronize(nullptr));  // the copies above have landed
    v_ = V3{W, H, T, C, n};
    scale_ = (float)(1.0 / std::sqrt((double)n));
    rb_ = fft_tile(pw_, H * T, EMAX, kT3);
    rba_ = fft_tile(pw_, H * T, kXElems, kXLanes);
    xb_ = 1;
    while (xb_ * 2 <= fft_tile(pd_, W * H, EMAX, kT3)) xb_ *= 2;
    tmp_.ensure(sizeof(float2) * (size_t)C * n);
  }
  long dense_elems() const override { return (long)C * N(); }
  long compact_elems() const override { return dense_elems(); }

  // K^H (ForwardOperation, cartesian_operator3d.cpp:64-133): the input is
  // masked as it is read, not in place.
  void forward(const float2 *kd, float2 *img, const float2 *b1, hipStream_t s) override {
    depth<kDAdjoint>(kd, nullptr, nullptr, tmp_.as<float2>(), nullptr, nullptr, s);
    adjoint_yx(img, b1, s);
  }
  // K (BackwardOperation, cartesian_operator3d.cpp:216-280)
  void backward(const float2 *img, float2 *kd, const float2 *b1, hipStream_t s) override {
    xy(img, nullptr, b1, kd, s);
    depth<kDApplyK>(kd, kd, nullptr, nullptr, nullptr, nullptr, s);
  }
  // CartesianOperator3D::AdaptLambda (cartesian_operator3d.cpp:47-62)
  double adapt_lambda(double k, double d) const override {
    const double n = (double)N();
    const double subfac = mask_.p ? n / mask_norm2_ : 1.0;
    return subfac * k + d;
  }
  void gather(const float2 *kd, float2 *out, hipStream_t s) override {
    const long n = dense_elems();
    hipLaunchKernelGGL(k3_mask, dim3(blocks_for(n)), dim3(kT3), 0, s, kd, mask_.as<float>(), out,
                       N(), n);
    AV_LAUNCH_CHECK();
  }
  void dual_update(const float2 *u, const float2 *b1, float2 *z, const float2 *d, float2 *khz,
                   const DevScalars *sc, hipStream_t s) override {
    float2 *t = tmp_.as<float2>();
    xy(u, nullptr, b1, t, s);
    depth<kDDual>(t, z, d, t, sc, nullptr, s);
    adjoint_yx(khz, b1, s);
  }
  void adjoint_compact(const float2 *z, const float2 *b1, float2 *img, hipStream_t s) override {
    forward(z, img, b1, s);
  }
  int norm2(const float2 *u, const float2 *usub, const float2 *b1, double *partial,
            hipStream_t s) override {
    xy(u, usub, b1, tmp_.as<float2>(), s);
    depth<kDNorm2>(tmp_.as<float2>(), nullptr, nullptr, nullptr, nullptr, partial, s);
    return max_partials();
  }
  int residual2(const float2 *u, const float2 *b1, const float2 *d, double *partial,
                hipStream_t s) override {
    xy(u, nullptr, b1, tmp_.as<float2>(), s);
    depth<kDResidual>(tmp_.as<float2>(), nullptr, d, nullptr, nullptr, partial, s);
    return max_partials();
  }
  int max_partials() const override { return (W * H + xb_ - 1) / xb_ * C; }
  bool volumetric() const override { return true; }
  bool khk_fp64(const double2 *u, double2 *out, const float2 *b1, Fp64Scratch &ws,
                hipStream_t s) const override {
    cart3_khk_fp64(W, H, T, C, mask_.as<float>(), u, out, b1, ws, s);
    return true;
  }

 private:
  DevBuf mask_, twx_, twy_, twz_, tmp_;
  FftPlan pw_{}, ph_{}, pd_{};
  V3 v_{};
  int rb_ = 1, rba_ = 1, xb_ = 1;  // rows per x / x^H block, columns per depth block
  float scale_ = 1.f;    // unitary 3D transform
  double mask_norm2_ = 0.0;

  // Transforms per block: the LDS tile, and one butterfly per lane where the
  // plan is two-stage.
  static int fft_tile(const FftPlan &p, int n, int elems, int lanes) {
    const int t = std::max(1, elems / p.L);
    return std::max(1, std::min(n, p.ra ? std::min(t, lanes / p.ra) : t));
  }
  // x and y transforms of b1_c (u - usub) into the C volumes of out.
  void xy(const float2 *u, const float2 *usub, const float2 *b1, float2 *out, hipStream_t s) {
    const dim3 grid((H * T + rb_ - 1) / rb_, C), block(kT3);
    switch (plan_kind(pw_, rb_)) {
      case kPlanTwo: hipLaunchKernelGGL(k3_x<kPlanTwo>, grid, block, 0, s, v_, pw_, rb_, u, usub, b1, out); break;
      case kPlanWide: hipLaunchKernelGGL(k3_x<kPlanWide>, grid, block, 0, s, v_, pw_, rb_, u, usub, b1, out); break;
      default: hipLaunchKernelGGL(k3_x<kPlanNarrow>, grid, block, 0, s, v_, pw_, rb_, u, usub, b1, out); break;
    }
    AV_LAUNCH_CHECK();
    launch_fft_axis0(out, ph_, H, W, C * T, +1, 1.f, s);
  }
  template <int MODE>
  void depth(const float2 *in, float2 *out, const float2 *d, float2 *zhat, const DevScalars *sc,
             double *partial, hipStream_t s) {
    const dim3 grid((W * H + xb_ - 1) / xb_, C), block(kT3);
    const float *m = mask_.as<float>();
    const size_t lds = sizeof(float2) * (size_t)pd_.L * xb_ * (MODE == kDDual ? 2 : 1);
    switch (plan_kind(pd_, xb_)) {
      case kPlanTwo: hipLaunchKernelGGL((k3_z<MODE, kPlanTwo>), grid, block, lds, s, v_, pd_, xb_, scale_, in, m, out, d, zhat, sc, partial); break;
      case kPlanWide: hipLaunchKernelGGL((k3_z<MODE, kPlanWide>), grid, block, lds, s, v_, pd_, xb_, scale_, in, m, out, d, zhat, sc, partial); break;
      default: hipLaunchKernelGGL((k3_z<MODE, kPlanNarrow>), grid, block, lds, s, v_, pd_, xb_, scale_, in, m, out, d, zhat, sc, partial); break;
    }
    AV_LAUNCH_CHECK();
  }
  // y and x adjoint transforms of tmp_, summed over the coils.
  void adjoint_yx(float2 *img, const float2 *b1, hipStream_t s) {
    float2 *t = tmp_.as<float2>();
    launch_fft_axis0(t, ph_, H, W, C * T, -1, 1.f, s);
    const dim3 grid((H * T + rba_ - 1) / rba_), block(kT3);
    const size_t lds = sizeof(float2) * 2 * kXG * (size_t)rba_ * W;
    switch (pw_.ra ? kPlanTwo : (plan_is_wide(pw_) ? kPlanWide : kPlanNarrow)) {
      case kPlanTwo: hipLaunchKernelGGL(k3_x_adj<kPlanTwo>, grid, block, lds, s, v_, pw_, rba_, t, b1, img); break;
      case kPlanWide: hipLaunchKernelGGL(k3_x_adj<kPlanWide>, grid, block, lds, s, v_, pw_, rba_, t, b1, img); break;
      default: hipLaunchKernelGGL(k3_x_adj<kPlanNarrow>, grid, block, lds, s, v_, pw_, rba_, t, b1, img); break;
    }
    AV_LAUNCH_CHECK();
  }
};

}  // namespace

Operator *make_cartesian3d(int W, int H, int D, int C, const float *mask) {
  return new CartesianOperator3D(W, H, D, C, mask);
}

}  // namespace avionic
