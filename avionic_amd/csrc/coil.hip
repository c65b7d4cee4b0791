// Coil-sensitivity estimation on the GPU: CoilConstruction
// (CUDA/src/coil_construction.cpp:22-557) with the Cartesian
// TimeAveragedReconstruction (cartesian_coil_construction.cpp:23-87).
//
//   1. time-averaged coil images crec_c = F(sum_t d_{t,c} / max(1, sum_t M_t))
//      and u0 = sqrt(sum_c |crec_c|^2) (phase of sum_c crec_c);
//   2. |b1_c| from (mu |u0|^2 + L) x_c = mu |u0| |crec_c| (L the periodic 2D
//      Laplacian, cg_forward_operation.h:46-67), all coils in one batched
//      conjugate-gradient solve with per-coil scalars on the device, then
//      |x_c| / sqrt(sum_c |x_c|^2) (B1FromUH1 :363-446);
//   3. a greedy coil order (FindMaximumSum :52-73, then the coil overlapping
//      most with the previous one); per coil a TGV2 image estimate from the
//      coils so far (UTGV2Recon :75-216) and the phase of the next map from a
//      quadratically regularised fit (B1Recon :217-362);
//   4. a final B1Recon over all coils (:553-556).
// Images are [coils][height][width] complex float; arithmetic is float (the
// reference's precision), reductions are double in a fixed order.  The PD loops
// run several iterations per launch on regions held in LDS.
#include <algorithm>
#include <cmath>
#include <memory>
#include <vector>

#include "coil.hpp"

namespace avionic {

namespace {

constexpr int kTC = 256;

inline unsigned nblocks(long n) { return (unsigned)std::max<long>(1, std::min<long>(4096, (n + kTC - 1) / kTC)); }

// ------------------------------------------------------------ time average
// davg[c] = sum_t d[t][c] / max(1, sum_t M_t), mask from the compact rows.
__global__ void k_tar_average(const CartGeom g, const float2 *__restrict__ kd,
                              float2 *__restrict__ avg) {
  const long HW = (long)g.H * g.W, n = HW * g.C;
  for (long e = (long)blockIdx.x * kTC + threadIdx.x; e < n; e += (long)gridDim.x * kTC) {
    const long c = e / HW, p = e % HW;
    const int y = (int)(p / g.W), x = (int)(p % g.W);
    float ms = 0.f;
    float2 s = czero();
    for (int t = 0; t < g.T; ++t) {
      const int k = g.rowmap[t * g.H + y];
      ms += k >= 0 ? g.mrows[((long)g.row_off[t] + k) * g.W + x] : 0.f;
      s = cadd(s, kd[((long)t * g.C + c) * HW + p]);
    }
    avg[e] = cscale(s, 1.f / fmaxf(1.f, ms));
  }
}
// u = sqrt(sum_c |crec_c|^2) (times the phase of sum_c crec_c)
__global__ void k_tar_combine(const float2 *__restrict__ crec, float2 *__restrict__ u, int C,
                              long N, int apply_phase) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    float2 s = czero();
    float m = 0.f;
    for (int c = 0; c < C; ++c) {
      const float2 v = crec[c * N + i];
      s = cadd(s, v);
      m += cabs2(v);
    }
    const float a = sqrtf(m);
    if (apply_phase) {
      const float ph = atan2f(s.y, s.x);
      u[i] = make_float2(a * cosf(ph), a * sinf(ph));
    } else {
      u[i] = make_float2(a, 0.f);
    }
  }
}

// --------------------------------------------------------- reductions
// block-wide sum of v, stored by thread 0 at *out
__device__ inline void block_sum_store(double v, double *out) {
  __shared__ double red[kTC];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = kTC / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}
// per coil: sum |a| (b == null) or sum |a| |b| (b: one image)
__global__ void k_coil_abs_sum(const float2 *__restrict__ a, const float2 *__restrict__ b, long N,
                               double *__restrict__ partial) {
  const int c = blockIdx.y, nb = gridDim.x;
  double acc = 0.0;
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)nb * kTC) {
    const float2 v = a[c * N + i];
    double t = sqrt((double)cabs2(v));
    if (b) t *= sqrt((double)cabs2(b[i]));
    acc += t;
  }
  block_sum_store(acc, partial + (long)c * nb + blockIdx.x);
}
// max |a| over one image (block partials)
__global__ void k_abs_max(const float2 *__restrict__ a, long N, double *__restrict__ partial) {
  __shared__ double red[kTC];
  double m = 0.0;
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC)
    m = fmax(m, sqrt((double)cabs2(a[i])));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = kTC / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// ------------------------------------------------------------- B1FromUH1
// Batched CG over the coils: A = diag(mu |u|^2) + L, L the periodic 2D
// Laplacian (D^T D with wrap-around forward differences).  Images of this size
// are bound by launches, so an iteration is two kernels: the direction update
// and A p (the neighbours' new directions are recomputed), and the step.  Each
// block sums the other kernel's block partials itself, in one fixed order; the
// scalars alternate between two slots, written by block 0 of a coil.
struct CgScal {
  double rho, rho0;
  int active;
};
// Sum of n <= kTC partials, in every lane.
__device__ inline double sum_partials(const double *p, int n) {
  __shared__ double red[kTC];
  red[threadIdx.x] = (int)threadIdx.x < n ? p[threadIdx.x] : 0.0;
  __syncthreads();
  for (int s = kTC / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  const double v = red[0];
  __syncthreads();
  return v;
}
// x = 0, p = 0, r = conj(u) mu |crec|; partial = sum |r|^2
__global__ void k_cg_init(const float2 *__restrict__ u, const float2 *__restrict__ crec, float mu,
                          float2 *__restrict__ x, float2 *__restrict__ r, float2 *__restrict__ p,
                          long N, double *__restrict__ partial) {
  const int c = blockIdx.y, nb = gridDim.x;
  double acc = 0.0;
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)nb * kTC) {
    const long e = c * N + i;
    const float a = mu * sqrtf(cabs2(crec[e]));
    const float2 uu = u[i];
    const float2 rhs = make_float2(uu.x * a, -uu.y * a);
    x[e] = czero();
    p[e] = czero();
    r[e] = rhs;
    acc += (double)cabs2(rhs);
  }
  block_sum_store(acc, partial + (long)c * nb + blockIdx.x);
}
// Convergence (squared residual <= 1e-12 rho0 or <= 1e-12), then for active
// coils p' = r + beta p and Ap = (mu |u|^2 + L) p'; pap = sum Re(conj(p') Ap).
// rr: block partials of |r|^2; first: the first iteration (rho0 = |r|^2,
// beta = 0).
__global__ __launch_bounds__(kTC) void k_cg_apply(const float2 *__restrict__ u, float mu,
                                                  const float2 *__restrict__ r,
                                                  const float2 *__restrict__ pin,
                                                  float2 *__restrict__ pout,
                                                  float2 *__restrict__ ap,
                                                  const CgScal *__restrict__ sin,
                                                  CgScal *__restrict__ sout, int first, int W,
                                                  int H, const double *__restrict__ rr,
                                                  double *__restrict__ pap) {
  const int c = blockIdx.y, nb = gridDim.x;
  const long N = (long)W * H;
  const double rn = sum_partials(rr + (long)c * nb, nb);
  CgScal s = sin[c];
  double beta = 0.0;
  if (first) {
    s.rho = s.rho0 = rn;
    s.active = rn > 1e-12 ? 1 : 0;
  } else if (s.active) {
    if (rn <= 1e-12 * s.rho0 || rn <= 1e-12) {
      s.active = 0;
    } else {
      beta = rn / s.rho;
      s.rho = rn;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) sout[c] = s;
  double acc = 0.0;
  if (s.active) {
    const float be = (float)beta;
    const float2 *rc = r + c * N, *pc = pin + c * N;
    auto dir = [&](int i) { return cadd(rc[i], cscale(pc[i], be)); };
    for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)nb * kTC) {
      const int x = (int)(i % W), y = (int)(i / W);
      const int xp = x + 1 < W ? x + 1 : 0, xm = x > 0 ? x - 1 : W - 1;
      const int yp = y + 1 < H ? y + 1 : 0, ym = y > 0 ? y - 1 : H - 1;
      const float2 pv = dir((int)i);
      const float2 bx = cadd(csub(dir(y * W + xp), cscale(pv, 2.f)), dir(y * W + xm));
      const float2 by = cadd(csub(dir(yp * W + x), cscale(pv, 2.f)), dir(ym * W + x));
      const float2 v = cadd(cscale(cadd(bx, by), -1.f), cscale(pv, mu * cabs2(u[i])));
      pout[c * N + i] = pv;
      ap[c * N + i] = v;
      acc += (double)pv.x * v.x + (double)pv.y * v.y;
    }
  }
  block_sum_store(acc, pap + (long)c * nb + blockIdx.x);
}
// alpha = rho / <p, Ap>; x += alpha p; r -= alpha Ap; rr = sum |r|^2
__global__ __launch_bounds__(kTC) void k_cg_update(float2 *__restrict__ x, float2 *__restrict__ r,
                                                   const float2 *__restrict__ p,
                                                   const float2 *__restrict__ ap,
                                                   const CgScal *__restrict__ sc, long N,
                                                   const double *__restrict__ pap,
                                                   double *__restrict__ rr) {
  const int c = blockIdx.y, nb = gridDim.x;
  if (!sc[c].active) return;
  const float al = (float)(sc[c].rho / sum_partials(pap + (long)c * nb, nb));
  double acc = 0.0;
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)nb * kTC) {
    const long e = c * N + i;
    x[e] = cadd(x[e], cscale(p[e], al));
    const float2 rn = csub(r[e], cscale(ap[e], al));
    r[e] = rn;
    acc += (double)cabs2(rn);
  }
  block_sum_store(acc, rr + (long)c * nb + blockIdx.x);
}
// b1_c = |x_c| / sqrt(sum_c |x_c|^2)
__global__ void k_cg_finish(const float2 *__restrict__ x, float2 *__restrict__ b1, int C, long N) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    float s = 0.f;
    for (int c = 0; c < C; ++c) s += cabs2(x[c * N + i]);
    const float inv = 1.f / sqrtf(s);
    for (int c = 0; c < C; ++c) b1[c * N + i] = make_float2(sqrtf(cabs2(x[c * N + i])) * inv, 0.f);
  }
}

// ------------------------------------------------------------- UTGV2Recon
// Lw = sum_{c in inds} conj(b1_c) crec_c; ib = 1 / (1 + tau sum |b1_c|^2)
__global__ void k_ut_pre(const float2 *__restrict__ b1, const float2 *__restrict__ crec,
                         const int *__restrict__ inds, int n_inds, float tau, long N,
                         float2 *__restrict__ lw, float *__restrict__ ib) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    float2 l = czero();
    float s = 0.f;
    for (int k = 0; k < n_inds; ++k) {
      const long o = (long)inds[k] * N + i;
      l = cadd(l, cmulc(b1[o], crec[o]));
      s += cabs2(b1[o]);
    }
    lw[i] = l;
    ib[i] = 1.f / (1.f + tau * s);
  }
}
// Several iterations of a PD loop per launch: a block holds a REG x REG region
// in LDS and advances it `its` <= kHalo iterations.  An iteration reaches one
// pixel in each direction, so after them the inner CORE x CORE pixels are the
// ones the whole image would have given; the block writes those to the other
// half of a double buffer.  The loops were bound by launches (4 us each, two per
// iteration): coil estimation at 192 x 160, 12 frames, 6 coils, 38 -> 10.6
// to 12.5 ms, by process (the two-kernel conjugate gradients above included).
constexpr int kHalo = 8;
// Region side REG, lanes per block, pixels per lane (ROW rows apart).
template <int REG_>
struct Region {
  static constexpr int REG = REG_, CORE = REG - 2 * kHalo, LANES = REG == 32 ? 1024 : 768,
                       PIX = REG * REG / LANES, ROW = LANES / REG;
};

// A lane's k-th pixel: its place l in the region and i in the image.
template <class G>
struct RegPix {
  int l, x, y, i;
  bool in, core;
  __device__ RegPix(int k, int W, int H) {
    const int lx = (int)threadIdx.x % G::REG, ly = (int)threadIdx.x / G::REG + k * G::ROW;
    l = ly * G::REG + lx;
    x = (int)blockIdx.x * G::CORE - kHalo + lx;
    y = (int)blockIdx.y * G::CORE - kHalo + ly;
    in = x >= 0 && x < W && y >= 0 && y < H;
    i = in ? y * W + x : 0;
    core = in && lx >= kHalo && lx < G::REG - kHalo && ly >= kHalo && ly < G::REG - kHalo;
  }
};
// Differences on the region; a neighbour outside it (clamped) only reaches
// pixels that the launch does not write.
template <class G>
struct RegDiff {
  int W, H;
  __device__ float2 at(const float2 *a, int l) const { return a[min(max(l, 0), G::REG * G::REG - 1)]; }
  __device__ float2 fx(const float2 *a, const RegPix<G> &p, float2 c) const {
    return p.x < W - 1 ? csub(at(a, p.l + 1), c) : czero();
  }
  __device__ float2 fy(const float2 *a, const RegPix<G> &p, float2 c) const {
    return p.y < H - 1 ? csub(at(a, p.l + G::REG), c) : czero();
  }
  __device__ float2 bx(const float2 *a, const RegPix<G> &p, float2 c) const {
    if (W == 1) return czero();
    if (p.x == 0) return c;
    const float2 m = at(a, p.l - 1);
    return p.x == W - 1 ? cscale(m, -1.f) : csub(c, m);
  }
  __device__ float2 by(const float2 *a, const RegPix<G> &p, float2 c) const {
    if (H == 1) return czero();
    if (p.y == 0) return c;
    const float2 m = at(a, p.l - G::REG);
    return p.y == H - 1 ? cscale(m, -1.f) : csub(c, m);
  }
};

// x1, ext1, x2 (2), ext2 (2), y1 (2), y2 (3): N elements each
constexpr int kUtState = 11;
template <class G>
__global__ __launch_bounds__(G::LANES) void k_ut_iterations(const float2 *__restrict__ in,
                                                            float2 *__restrict__ out,
                                                            const float2 *__restrict__ lw,
                                                            const float *__restrict__ ib, int W,
                                                            int H, float sigma, float tau, float r1,
                                                            float r2, int its) {
  extern __shared__ float2 sh[];  // ext1, ext2 (2), y1 (2), y2 (3)
  constexpr int A = G::REG * G::REG;
  float2 *e1 = sh, *v0 = sh + A, *v1 = sh + 2 * A, *p0 = sh + 3 * A, *p1 = sh + 4 * A,
         *q0 = sh + 5 * A, *q1 = sh + 6 * A, *q2 = sh + 7 * A;
  const long N = (long)W * H;
  const RegDiff<G> d{W, H};
  float2 x1[G::PIX], xa[G::PIX], xb[G::PIX], l[G::PIX];
  float b[G::PIX];
#pragma unroll
  for (int k = 0; k < G::PIX; ++k) {
    const RegPix<G> p(k, W, H);
    auto ld = [&](int c) { return p.in ? in[c * N + p.i] : czero(); };
    x1[k] = ld(0);
    xa[k] = ld(2);
    xb[k] = ld(3);
    l[k] = p.in ? lw[p.i] : czero();
    b[k] = p.in ? ib[p.i] : 0.f;
    e1[p.l] = ld(1);
    v0[p.l] = ld(4);
    v1[p.l] = ld(5);
    p0[p.l] = ld(6);
    p1[p.l] = ld(7);
    q0[p.l] = ld(8);
    q1[p.l] = ld(9);
    q2[p.l] = ld(10);
  }
  __syncthreads();
  for (int it = 0; it < its; ++it) {
    // y1 += sigma (grad ext1 - ext2); y2 += sigma E ext2; projections (radii
    // alpha1 nu and alpha0 nu; |y2| with the off-diagonal weight 2)
#pragma unroll
    for (int k = 0; k < G::PIX; ++k) {
      const RegPix<G> p(k, W, H);
      const float2 e = e1[p.l], a = v0[p.l], c = v1[p.l];
      const float2 s0 = cadd(p0[p.l], cscale(csub(d.fx(e1, p, e), a), sigma));
      const float2 s1 = cadd(p1[p.l], cscale(csub(d.fy(e1, p, e), c), sigma));
      const float2 g2 = cscale(cadd(d.by(v0, p, a), d.bx(v1, p, c)), 0.5f);
      const float2 t0 = cadd(q0[p.l], cscale(d.bx(v0, p, a), sigma));
      const float2 t1 = cadd(q1[p.l], cscale(d.by(v1, p, c), sigma));
      const float2 t2 = cadd(q2[p.l], cscale(g2, sigma));
      const float n1 = fmaxf(1.f, sqrtf(cabs2(s0) + cabs2(s1)) / r1);
      const float n2 = fmaxf(1.f, sqrtf(cabs2(t0) + cabs2(t1) + 2.f * cabs2(t2)) / r2);
      p0[p.l] = cscale(s0, 1.f / n1);
      p1[p.l] = cscale(s1, 1.f / n1);
      q0[p.l] = cscale(t0, 1.f / n2);
      q1[p.l] = cscale(t1, 1.f / n2);
      q2[p.l] = cscale(t2, 1.f / n2);
    }
    __syncthreads();
    // x1+ = (x1 + tau div y1 + tau Lw) ib; x2+ = x2 + tau (y1 + divsym y2);
    // ext = 2 x+ - x; x = x+
#pragma unroll
    for (int k = 0; k < G::PIX; ++k) {
      const RegPix<G> p(k, W, H);
      const float2 a = p0[p.l], c = p1[p.l], t0 = q0[p.l], t1 = q1[p.l], t2 = q2[p.l];
      const float2 dv = cadd(d.bx(p0, p, a), d.by(p1, p, c));
      const float2 sd0 = cadd(d.fx(q0, p, t0), d.fy(q2, p, t2));
      const float2 sd1 = cadd(d.fx(q2, p, t2), d.fy(q1, p, t1));
      const float2 xn = cscale(cadd(cadd(x1[k], cscale(dv, tau)), cscale(l[k], tau)), b[k]);
      const float2 n0 = cadd(xa[k], cscale(cadd(a, sd0), tau));
      const float2 n1 = cadd(xb[k], cscale(cadd(c, sd1), tau));
      e1[p.l] = csub(cscale(xn, 2.f), x1[k]);
      v0[p.l] = csub(cscale(n0, 2.f), xa[k]);
      v1[p.l] = csub(cscale(n1, 2.f), xb[k]);
      x1[k] = xn;
      xa[k] = n0;
      xb[k] = n1;
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < G::PIX; ++k) {
    const RegPix<G> p(k, W, H);
    if (!p.core) continue;
    auto st = [&](int c, float2 v) { out[c * N + p.i] = v; };
    st(0, x1[k]);
    st(1, e1[p.l]);
    st(2, xa[k]);
    st(3, xb[k]);
    st(4, v0[p.l]);
    st(5, v1[p.l]);
    st(6, p0[p.l]);
    st(7, p1[p.l]);
    st(8, q0[p.l]);
    st(9, q1[p.l]);
    st(10, q2[p.l]);
  }
}

// --------------------------------------------------------------- B1Recon
// un = u0 / max|u0|: lw_c = conj(un) crec_c, iu = 1 / (1 + tau |un|^2); the
// maximum from nmx <= kTC block partials, stored at *mx
__global__ __launch_bounds__(kTC) void k_b1_pre(const float2 *__restrict__ u0,
                                                const float2 *__restrict__ crec,
                                                const double *__restrict__ part, int nmx,
                                                double *__restrict__ mx, float tau, int coils,
                                                long N, float2 *__restrict__ lw,
                                                float *__restrict__ iu) {
  __shared__ double red[kTC];
  red[threadIdx.x] = (int)threadIdx.x < nmx ? part[threadIdx.x] : 0.0;
  __syncthreads();
  for (int s = kTC / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *mx = red[0];
  const float inv = (float)(1.0 / red[0]);
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    const float2 un = cscale(u0[i], inv);
    iu[i] = 1.f / (1.f + tau * cabs2(un));
    for (int c = 0; c < coils; ++c) lw[c * N + i] = cmulc(un, crec[c * N + i]);
  }
}
// Iterations of one coil (blockIdx.z) on the region form above; a coil's state
// is x, ext, y (2): N elements each.
//   y = (y + sigma grad ext) / (1 + sigma / mu)
//   x+ = (x + tau div y + tau lw) iu; ext = 2 x+ - x; x = x+
constexpr int kB1State = 4;
template <class G>
__global__ __launch_bounds__(G::LANES) void k_b1_iterations(const float2 *__restrict__ in,
                                                            float2 *__restrict__ out,
                                                            const float2 *__restrict__ lw,
                                                            const float *__restrict__ iu, int W,
                                                            int H, float sigma, float shrink,
                                                            float tau, int its) {
  __shared__ float2 e1[G::REG * G::REG], y0[G::REG * G::REG], y1[G::REG * G::REG];
  const long N = (long)W * H;
  const RegDiff<G> d{W, H};
  in += (long)blockIdx.z * kB1State * N;
  out += (long)blockIdx.z * kB1State * N;
  lw += (long)blockIdx.z * N;
  float2 x[G::PIX], ext[G::PIX], a[G::PIX], c[G::PIX], l[G::PIX];
  float b[G::PIX];
#pragma unroll
  for (int k = 0; k < G::PIX; ++k) {
    const RegPix<G> p(k, W, H);
    x[k] = p.in ? in[p.i] : czero();
    ext[k] = p.in ? in[N + p.i] : czero();
    a[k] = p.in ? in[2 * N + p.i] : czero();
    c[k] = p.in ? in[3 * N + p.i] : czero();
    l[k] = p.in ? lw[p.i] : czero();
    b[k] = p.in ? iu[p.i] : 0.f;
    e1[p.l] = ext[k];
  }
  __syncthreads();
  for (int it = 0; it < its; ++it) {
#pragma unroll
    for (int k = 0; k < G::PIX; ++k) {
      const RegPix<G> p(k, W, H);
      a[k] = cscale(cadd(a[k], cscale(d.fx(e1, p, ext[k]), sigma)), shrink);
      c[k] = cscale(cadd(c[k], cscale(d.fy(e1, p, ext[k]), sigma)), shrink);
      y0[p.l] = a[k];
      y1[p.l] = c[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < G::PIX; ++k) {
      const RegPix<G> p(k, W, H);
      const float2 dv = cadd(d.bx(y0, p, a[k]), d.by(y1, p, c[k]));
      const float2 xn = cscale(cadd(cadd(x[k], cscale(dv, tau)), cscale(l[k], tau)), b[k]);
      ext[k] = csub(cscale(xn, 2.f), x[k]);
      x[k] = xn;
      e1[p.l] = ext[k];
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < G::PIX; ++k) {
    const RegPix<G> p(k, W, H);
    if (!p.core) continue;
    out[p.i] = x[k];
    out[N + p.i] = ext[k];
    out[2 * N + p.i] = a[k];
    out[3 * N + p.i] = c[k];
  }
}
// x_c = s_c / sqrt(sum_c |s_c|^2) from the coils' states
__global__ void k_b1_normalize(const float2 *__restrict__ s, float2 *__restrict__ x, int coils,
                               long N) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    float m = 0.f;
    for (int c = 0; c < coils; ++c) m += cabs2(s[c * kB1State * N + i]);
    const float inv = 1.f / sqrtf(m);
    for (int c = 0; c < coils; ++c) x[c * N + i] = cscale(s[c * kB1State * N + i], inv);
  }
}

// ------------------------------------------------------ outer loop helpers
// w = sqrt(w^2 + |b|^2)
__global__ void k_weight_update(float *__restrict__ w, const float2 *__restrict__ b, long N) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC)
    w[i] = sqrtf(w[i] * w[i] + cabs2(b[i]));
}
// bm = |b1_m| u_prev w; cm = crec_m w
__global__ void k_weighted_inputs(const float2 *__restrict__ absb, const float2 *__restrict__ u,
                                  const float2 *__restrict__ crec, const float *__restrict__ w,
                                  float2 *__restrict__ bm, float2 *__restrict__ cm, long N) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    bm[i] = cscale(cmul(absb[i], u[i]), w[i]);
    cm[i] = cscale(crec[i], w[i]);
  }
}
// b1_m = |b1_m| exp(i arg x)
__global__ void k_apply_phase(const float2 *__restrict__ absb, const float2 *__restrict__ x,
                              float2 *__restrict__ out, long N) {
  for (long i = (long)blockIdx.x * kTC + threadIdx.x; i < N; i += (long)gridDim.x * kTC) {
    const float ph = atan2f(x[i].y, x[i].x);
    out[i] = cmul(absb[i], make_float2(cosf(ph), sinf(ph)));
  }
}

}  // namespace

// ======================================================================= host
// CoilConstruction::InitParams (coil_construction.cpp:22-46)
void coil_default_params(avionic_coil_params *p) {
  *p = avionic_coil_params{};
  p->uH1mu = 1e-5;
  p->uReg = 0.2;
  p->uNrIt = 100;
  p->uSigma = p->uTau = std::sqrt(1.0 / 12.0);
  p->uAlpha0 = std::sqrt(2.0);
  p->uAlpha1 = 1.0;
  p->b1Reg = 2.0;
  p->b1NrIt = 500;
  p->b1Sigma = p->b1Tau = std::sqrt(1.0 / 8.0);
  p->b1FinalReg = 0.1;
  p->b1FinalNrIt = 1000;
}

// sum over each coil of |crec_c| (or |crec_c| |ref|), fixed-order
std::vector<double> coil_abs_sums(const CoilCtx &k, const float2 *crec, const float2 *ref,
                                  int coils) {
  const int nb = (int)std::min<long>(256, (k.N + kTC - 1) / kTC);
  DevBuf part;
  part.ensure(sizeof(double) * (size_t)nb * coils);
  hipLaunchKernelGGL(k_coil_abs_sum, dim3(nb, coils), dim3(kTC), 0, k.s, crec, ref, k.N,
                     part.as<double>());
  AV_LAUNCH_CHECK();
  std::vector<double> h((size_t)nb * coils), out(coils, 0.0);
  AV_HIP(hipMemcpyAsync(h.data(), part.p, sizeof(double) * h.size(), hipMemcpyDeviceToHost, k.s));
  AV_HIP(hipStreamSynchronize(k.s));
  for (int c = 0; c < coils; ++c)
    for (int b = 0; b < nb; ++b) out[c] += h[(size_t)c * nb + b];
  return out;
}

int coil_find_max_sum(const CoilCtx &k, const float2 *crec) {
  const std::vector<double> sums = coil_abs_sums(k, crec, nullptr, k.C);
  int best = -1;
  for (int c = 0; c < k.C; ++c)
    if (best < 0 || sums[c] > sums[best]) best = c;
  return best;
}

void coil_time_averaged(const Operator &op, const float2 *kdata, float2 *u, float2 *crec,
                        bool apply_phase, hipStream_t s) {
  const long HW = (long)op.W * op.H;
  if (const auto *c = dynamic_cast<const CartesianOperator *>(&op)) {
    // cartesian_coil_construction.cpp:23-87: per coil the sampled average
    // over frames, then the image transform of the operator
    const CartGeom &g = c->plan().g;
    hipLaunchKernelGGL(k_tar_average, dim3(nblocks(HW * g.C)), dim3(kTC), 0, s, g, kdata, crec);
    AV_LAUNCH_CHECK();
    launch_fft2(crec, g.pw, g.ph, g.H, g.W, g.C, -1, g.centered, g.scale, s);
  } else {
    // noncartesian_coil_construction.cpp:21-123: per coil, every frame's
    // points gridded together into one image (kernel width 3, oversampling 2)
    std::unique_ptr<Operator> all(make_noncartesian_all_frames(op));
    if (!all)
      throw Error(AVIONIC_E_UNSUPPORTED, "time-averaged coil images need a 2D+t operator");
    const long M = op.dense_elems() / ((long)op.T * op.C);  // points per frame
    DevBuf z, ones;
    z.ensure(sizeof(float2) * M * op.T);
    ones.ensure(sizeof(float2) * HW);
    const std::vector<float2> one((size_t)HW, make_float2(1.f, 0.f));
    AV_HIP(hipMemcpyAsync(ones.p, one.data(), sizeof(float2) * HW, hipMemcpyHostToDevice, s));
    for (int c = 0; c < op.C; ++c) {
      // [frames][coils][M] -> coil c's [frames * M]
      AV_HIP(hipMemcpy2DAsync(z.p, sizeof(float2) * M, kdata + (long)c * M,
                              sizeof(float2) * M * op.C, sizeof(float2) * M, op.T,
                              hipMemcpyDeviceToDevice, s));
      all->forward(z.as<float2>(), crec + (long)c * HW, ones.as<float2>(), s);
    }
    AV_HIP(hipStreamSynchronize(s));  // `one` and the operator end with this call
  }
  hipLaunchKernelGGL(k_tar_combine, dim3(nblocks(HW)), dim3(kTC), 0, s, crec, u, op.C, HW,
                     apply_phase ? 1 : 0);
  AV_LAUNCH_CHECK();
}

void coil_b1_from_uh1(const CoilCtx &k, const float2 *u, const float2 *crec, double mu,
                      float2 *b1) {
  const long n = k.N * k.C;
  DevBuf x, r, p, ap, sc, part;
  x.ensure(sizeof(float2) * n);
  r.ensure(sizeof(float2) * n);
  p.ensure(sizeof(float2) * 2 * n);
  ap.ensure(sizeof(float2) * n);
  sc.ensure(sizeof(CgScal) * 2 * k.C);
  const int nb = (int)std::min<long>(kTC, (k.N + kTC - 1) / kTC);
  part.ensure(sizeof(double) * 2 * (size_t)nb * k.C);
  double *rr = part.as<double>(), *pap = rr + (size_t)nb * k.C;
  float2 *pb[2] = {p.as<float2>(), p.as<float2>() + n};
  CgScal *sb[2] = {sc.as<CgScal>(), sc.as<CgScal>() + k.C};
  const dim3 grid(nb, k.C);
  AV_HIP(hipMemsetAsync(sc.p, 0, sc.bytes, k.s));
  hipLaunchKernelGGL(k_cg_init, grid, dim3(kTC), 0, k.s, u, crec, (float)mu, x.as<float2>(),
                     r.as<float2>(), pb[0], k.N, rr);
  AV_LAUNCH_CHECK();
  for (int it = 0; it < 800; ++it) {
    const int a = it & 1, b = 1 - a;
    hipLaunchKernelGGL(k_cg_apply, grid, dim3(kTC), 0, k.s, u, (float)mu, r.as<float2>(), pb[a],
                       pb[b], ap.as<float2>(), sb[a], sb[b], it == 0 ? 1 : 0, k.W, k.H, rr, pap);
    hipLaunchKernelGGL(k_cg_update, grid, dim3(kTC), 0, k.s, x.as<float2>(), r.as<float2>(), pb[b],
                       ap.as<float2>(), sb[b], k.N, pap, rr);
    AV_LAUNCH_CHECK();
    if ((it & 15) == 0 && it > 0) {  // stop once every coil had converged before this iteration
      std::vector<CgScal> hs(k.C);
      AV_HIP(hipMemcpyAsync(hs.data(), sb[b], sizeof(CgScal) * k.C, hipMemcpyDeviceToHost, k.s));
      AV_HIP(hipStreamSynchronize(k.s));
      bool any = false;
      for (const CgScal &c : hs) any = any || c.active;
      if (!any) break;
    }
  }
  hipLaunchKernelGGL(k_cg_finish, dim3(nblocks(k.N)), dim3(kTC), 0, k.s, x.as<float2>(), b1, k.C,
                     k.N);
  AV_LAUNCH_CHECK();
}

template <class G>
static dim3 region_grid(const CoilCtx &k, int coils) {
  return dim3((k.W + G::CORE - 1) / G::CORE, (k.H + G::CORE - 1) / G::CORE, coils);
}
// Small regions (one pixel per lane, four times the core's pixels computed)
// where they make at most four blocks per CU, large ones (2.25 times) above.
// Measured on MI355X, large / small: one image of 192 x 160, 14.2 / 7.3 us per
// launch of B1Recon iterations; whole estimation 192x160x6 14.7 / 11 ms, 256x256x8
// 19.6 / 14.6 ms with small ones for the single images only.
static bool small_regions(const CoilCtx &k, int coils) {
  const dim3 g = region_grid<Region<32>>(k, coils);
  return (long)g.x * g.y * g.z <= 1024;
}
template <class G>
static void ut_iterations(const CoilCtx &k, const float2 *in, float2 *out, const float2 *lw,
                          const float *ib, float sigma, float tau, float r1, float r2, int its) {
  hipLaunchKernelGGL(k_ut_iterations<G>, region_grid<G>(k, 1), dim3(G::LANES),
                     sizeof(float2) * 8 * G::REG * G::REG, k.s, in, out, lw, ib, k.W, k.H, sigma, tau,
                     r1, r2, its);
}
template <class G>
static void b1_iterations(const CoilCtx &k, int coils, const float2 *in, float2 *out,
                          const float2 *lw, const float *iu, float sigma, float shrink, float tau,
                          int its) {
  hipLaunchKernelGGL(k_b1_iterations<G>, region_grid<G>(k, coils), dim3(G::LANES), 0, k.s, in, out,
                     lw, iu, k.W, k.H, sigma, shrink, tau, its);
}

void coil_utgv2(const CoilCtx &k, const float2 *b1, const float2 *crec, const std::vector<int> &inds,
                const avionic_coil_params &p, float2 *x_inout) {
  const long N = k.N;
  DevBuf bi, lw, ib, st;
  bi.ensure(sizeof(int) * inds.size());
  AV_HIP(hipMemcpyAsync(bi.p, inds.data(), sizeof(int) * inds.size(), hipMemcpyHostToDevice, k.s));
  lw.ensure(sizeof(float2) * N);
  ib.ensure(sizeof(float) * N);
  st.ensure(sizeof(float2) * N * kUtState * 2);
  float2 *sb[2] = {st.as<float2>(), st.as<float2>() + N * kUtState};
  AV_HIP(hipMemsetAsync(sb[0], 0, sizeof(float2) * N * kUtState, k.s));
  for (int c = 0; c < 2; ++c)  // x1, ext1
    AV_HIP(hipMemcpyAsync(sb[0] + c * N, x_inout, sizeof(float2) * N, hipMemcpyDeviceToDevice, k.s));
  const float tau = (float)p.uTau, sigma = (float)p.uSigma;
  hipLaunchKernelGGL(k_ut_pre, dim3(nblocks(N)), dim3(kTC), 0, k.s, b1, crec, bi.as<int>(),
                     (int)inds.size(), tau, N, lw.as<float2>(), ib.as<float>());
  AV_LAUNCH_CHECK();
  const float r1 = (float)(p.uAlpha1 * p.uReg), r2 = (float)(p.uAlpha0 * p.uReg);
  int cur = 0;
  const auto iterate = small_regions(k, 1) ? ut_iterations<Region<32>> : ut_iterations<Region<48>>;
  for (unsigned it = 0; it < p.uNrIt; it += kHalo, cur = 1 - cur)
    iterate(k, sb[cur], sb[1 - cur], lw.as<float2>(), ib.as<float>(), sigma, tau, r1, r2,
            (int)std::min<unsigned>(kHalo, p.uNrIt - it));
  AV_LAUNCH_CHECK();
  AV_HIP(hipMemcpyAsync(x_inout, sb[cur], sizeof(float2) * N, hipMemcpyDeviceToDevice, k.s));
  AV_HIP(hipStreamSynchronize(k.s));  // the index table stays alive until here
}

void coil_b1_recon(const CoilCtx &k, const float2 *u0, const float2 *crec, int coils,
                   unsigned maxit, double mu, const avionic_coil_params &p, float2 *x1) {
  const long N = k.N, n = N * coils;
  DevBuf st, lw, iu, part;
  st.ensure(sizeof(float2) * n * kB1State * 2);
  lw.ensure(sizeof(float2) * n);
  iu.ensure(sizeof(float) * N);
  const int nb = (int)std::min<long>(kTC, (N + kTC - 1) / kTC);
  part.ensure(sizeof(double) * (nb + 1));
  float2 *sb[2] = {st.as<float2>(), st.as<float2>() + n * kB1State};
  AV_HIP(hipMemsetAsync(sb[0], 0, sizeof(float2) * n * kB1State, k.s));
  hipLaunchKernelGGL(k_abs_max, dim3(nb), dim3(kTC), 0, k.s, u0, N, part.as<double>());
  AV_LAUNCH_CHECK();
  const float tau = (float)p.b1Tau, sigma = (float)p.b1Sigma;
  hipLaunchKernelGGL(k_b1_pre, dim3(nblocks(N)), dim3(kTC), 0, k.s, u0, crec, part.as<double>(), nb,
                     part.as<double>() + nb, tau, coils, N, lw.as<float2>(), iu.as<float>());
  AV_LAUNCH_CHECK();
  const float shrink = (float)(1.0 / (1.0 + p.b1Sigma / mu));
  int cur = 0;
  const auto iterate = small_regions(k, coils) ? b1_iterations<Region<32>> : b1_iterations<Region<48>>;
  for (unsigned it = 0; it < maxit; it += kHalo, cur = 1 - cur)
    iterate(k, coils, sb[cur], sb[1 - cur], lw.as<float2>(), iu.as<float>(), sigma, shrink, tau,
            (int)std::min<unsigned>(kHalo, maxit - it));
  AV_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_b1_normalize, dim3(nblocks(N)), dim3(kTC), 0, k.s, sb[cur], x1, coils, N);
  AV_LAUNCH_CHECK();
  double mx = 0.0;
  AV_HIP(hipMemcpyAsync(&mx, part.as<double>() + nb, sizeof(double), hipMemcpyDeviceToHost, k.s));
  AV_HIP(hipStreamSynchronize(k.s));
  AV_CHECK(mx > 0.0, "coil construction: the image estimate is zero");
}

// PerformCoilConstruction (coil_construction.cpp:447-557) from the
// time-averaged images.  u_out, b1_out: [C][H][W]; order: the coil order.
void coil_construction_from(const CoilCtx &k, const float2 *crec, const float2 *u0c,
                            const avionic_coil_params &p, float2 *u, float2 *b1,
                            std::vector<int> *order) {
  const long N = k.N;
  DevBuf u0, absb1, w, bm, cm, x1, umax;
  u0.ensure(sizeof(float2) * N);
  absb1.ensure(sizeof(float2) * N * k.C);
  w.ensure(sizeof(float) * N);
  bm.ensure(sizeof(float2) * N);
  cm.ensure(sizeof(float2) * N);
  x1.ensure(sizeof(float2) * N);
  umax.ensure(sizeof(float2) * N);
  // |u0| (coil_construction.cpp:459-461)
  hipLaunchKernelGGL(k_tar_combine, dim3(nblocks(N)), dim3(kTC), 0, k.s, u0c, u0.as<float2>(), 1,
                     N, 0);
  AV_LAUNCH_CHECK();
  coil_b1_from_uh1(k, u0.as<float2>(), crec, p.uH1mu, absb1.as<float2>());
  AV_HIP(hipMemsetAsync(b1, 0, sizeof(float2) * N * k.C, k.s));
  AV_HIP(hipMemsetAsync(u, 0, sizeof(float2) * N * k.C, k.s));
  AV_HIP(hipMemsetAsync(w.p, 0, w.bytes, k.s));
  AV_HIP(hipMemsetAsync(umax.p, 0, umax.bytes, k.s));
  std::vector<int> inds{coil_find_max_sum(k, crec)};
  AV_HIP(hipMemcpyAsync(b1 + inds[0] * N, absb1.as<float2>() + inds[0] * N, sizeof(float2) * N,
                        hipMemcpyDeviceToDevice, k.s));
  coil_utgv2(k, b1, crec, inds, p, umax.as<float2>());
  AV_HIP(hipMemcpyAsync(u, umax.p, sizeof(float2) * N, hipMemcpyDeviceToDevice, k.s));
  for (int cnt = 1; cnt < k.C; ++cnt) {
    const int prev = inds[cnt - 1];
    hipLaunchKernelGGL(k_weight_update, dim3(nblocks(N)), dim3(kTC), 0, k.s, w.as<float>(),
                       absb1.as<float2>() + prev * N, N);
    AV_LAUNCH_CHECK();
    // the unused coil overlapping most with the previous one
    const std::vector<double> ov = coil_abs_sums(k, crec, crec + prev * N, k.C);
    int best = -1;
    for (int c = 0; c < k.C; ++c) {
      if (std::find(inds.begin(), inds.end(), c) != inds.end()) continue;
      if (best < 0 || ov[c] > ov[best]) best = c;
    }
    inds.push_back(best);
    hipLaunchKernelGGL(k_weighted_inputs, dim3(nblocks(N)), dim3(kTC), 0, k.s,
                       absb1.as<float2>() + best * N, u + (cnt - 1) * N, crec + best * N,
                       w.as<float>(), bm.as<float2>(), cm.as<float2>(), N);
    AV_LAUNCH_CHECK();
    coil_b1_recon(k, bm.as<float2>(), cm.as<float2>(), 1, p.b1NrIt, p.b1Reg, p, x1.as<float2>());
    hipLaunchKernelGGL(k_apply_phase, dim3(nblocks(N)), dim3(kTC), 0, k.s,
                       absb1.as<float2>() + best * N, x1.as<float2>(), b1 + best * N, N);
    AV_LAUNCH_CHECK();
    AV_HIP(hipMemcpyAsync(umax.p, u + (cnt - 1) * N, sizeof(float2) * N, hipMemcpyDeviceToDevice,
                          k.s));
    coil_utgv2(k, b1, crec, inds, p, umax.as<float2>());
    AV_HIP(hipMemcpyAsync(u + cnt * N, umax.p, sizeof(float2) * N, hipMemcpyDeviceToDevice, k.s));
  }
  coil_b1_recon(k, umax.as<float2>(), crec, k.C, p.b1FinalNrIt, p.b1FinalReg, p, b1);
  AV_HIP(hipStreamSynchronize(k.s));
  if (order) *order = inds;
}

}  // namespace avionic
