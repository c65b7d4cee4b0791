// Shared parts of the Kaiser-Bessel gridding passes (noncart.hpp): block sizes,
// grid-length plans.
#pragma once

#include <algorithm>

#include "fft_device.hpp"
#include "noncart.hpp"

namespace avionic {

namespace {

#ifndef AVIONIC_NC_COLF_THREADS
#define AVIONIC_NC_COLF_THREADS 256
#endif
#ifndef AVIONIC_NC_COLA_THREADS
#define AVIONIC_NC_COLA_THREADS 512
#endif
constexpr int NCF = AVIONIC_NC_COLF_THREADS;  // threads of a forward column-pass block
constexpr int NCC = AVIONIC_NC_COLA_THREADS;  // threads of an adjoint column-pass block
constexpr int NCR = 256;   // threads of a row-pass / sample-pass block
constexpr int NCE = 4096;  // complex elements of an LDS transform tile
// Twiddle-table entries and per-lane outputs of the narrow / wide kernel
// variants (plan_is_wide: a grid longer than 512 or a radix-11 / -13 stage).
constexpr int nc_table_len(int kind) {
  return kind == kPlanTwo ? kMaxRadix * kMaxRadix : (kind == kPlanWide ? kMaxFftLen : kMaxFftLenNarrow);
}
constexpr int row_slots_nc(int kind) { return max_slots(NCE, NCR, kind); }

__device__ inline int wrap_up(int v, int G) { return v >= G ? v - G : v; }

// Grid transforms: on the geometry's runtime plans (NcPlanRt), or compiled
// for a grid length in both directions, with XB grid columns per column-pass
// block (pick_cols at that length): 384 (a 256 x 256 image at oversampling
// 1.5), 512 (256 x 256 at 2, the reference's default oversampling), 192 and 256
// (128 x 128 at 1.5 and 2).  nc_ct_len picks the compiled kernels; they run
// their stages with the index arithmetic folded into constants.
struct NcPlanRt {
  static constexpr int L = 0, XB = 0;
};
template <class F, int XB_>
struct NcCt : F {
  static constexpr int XB = XB_;
  static constexpr int RL = F::R2 > 1 ? F::R2 : F::R1;  // last radix
};
using NcPlan384 = NcCt<FftCt<384, 16, 8, 3>, 8>;
using NcPlan512 = NcCt<FftCt<512, 8, 8, 8>, 8>;
using NcPlan192 = NcCt<FftCt<192, 16, 4, 3>, 16>;
using NcPlan256 = NcCt<FftCt<256, 16, 16>, 16>;
// K's passes: radices of about equal size keep their lanes equally busy in every
// stage; K^H's column pass (512 lanes, its sums between) measured faster with
// the others above.  K at 256x256x30x12: 324 -> 312 us (osf 1.5, against 16, 8,
// 3), 424 -> 397 us (osf 2, 8, 8, 8 against 16, 16, 2; K^H 481 -> 459 us).
using NcFwd384 = NcCt<FftCt<384, 8, 8, 6>, 8>;
using NcFwd192 = NcCt<FftCt<192, 16, 12>, 16>;

// The compiled grid length that applies (0: none): both grid directions have
// that length and the tiles have the compiled sizes.
template <class PL>
bool nc_is(const NcGeom &g) {
  return g.px.L == PL::L && g.py.L == PL::L && g.XBf == PL::XB && g.XBa == PL::XB &&
         g.RBf <= NCE / PL::L && g.RBa <= NCE / PL::L;
}
int nc_ct_len(const NcGeom &g) {
  if (g.wide == kPlanWide) return 0;
  if (nc_is<NcPlan384>(g)) return 384;
  if (nc_is<NcPlan512>(g)) return 512;
  if (nc_is<NcPlan192>(g)) return 192;
  if (nc_is<NcPlan256>(g)) return 256;
  return 0;
}

}  // namespace

}  // namespace avionic
