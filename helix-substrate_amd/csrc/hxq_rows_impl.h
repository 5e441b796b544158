// Instantiations of the few-row GEMM for one activation type (included by
// hxq_rows_bf16.hip, hxq_rows_f16.hip and hxq_rows_f32.hip, which build in parallel).
#pragma once
#include <type_traits>

#include "hxq_rows.h"

namespace hxq {
namespace rw {

template <int XT, int MT, int NS, int SP, int W>
static int launch_fmt(const Call &c, int format, bool aff, const Plan &p, hipStream_t stream) {
    const dim3 grid(p.bx, p.by);
#define HXQ_RW(AF_, F_, W_) \
    hipLaunchKernelGGL((rows_kernel<MT, NS, SP, XT, AF_, F_, W_>), grid, dim3(W_ * 64), 0, stream, c.idx, c.x, \
                       c.cb, c.ga, c.M, c.OUT, c.K, c.ngroups, c.gmul, c.a, 0)
    switch (format) {
        case HXQ_FMT_SCALAR:
            if (aff) HXQ_RW(true, HXQ_FMT_SCALAR, W); else HXQ_RW(false, HXQ_FMT_SCALAR, W);
            break;
        case HXQ_FMT_SCALAR_U16:
            if constexpr (NS <= kWideSubs) {
                // two index loads and the affine: 16 waves leave 128 registers, which
                // spill (36 and 44 bytes a lane at 1 x 1 x 4 and 2 x 3 x 1).  us with
                // 16 / 8 waves: 16 x 18944 x 3584 40.7 / 35.0, 17 x 18944 x 3584
                // 56.5 / 44.8, 16 x 3584 x 18944 48.3 / 40.2, 16 x 512 x 3584 10.0 /
                // 10.3; two row tiles of one subtile fit 16: 17 x 3584 x 18944 41.3 / 43.3
                constexpr int WA = MT == 2 && NS == 1 ? W : 8;
                if (aff) HXQ_RW(true, HXQ_FMT_SCALAR_U16, WA); else HXQ_RW(false, HXQ_FMT_SCALAR_U16, W);
            } else {
                HXQ_REQUIRE(false, "no such few-row plan");
            }
            break;
        case HXQ_FMT_VQ2_U16: HXQ_RW(false, HXQ_FMT_VQ2_U16, W); break;
        case HXQ_FMT_VQ2_P12: HXQ_RW(false, HXQ_FMT_VQ2_P12, W); break;
        default: HXQ_RW(true, HXQ_FMT_AF6, W); break;
    }
#undef HXQ_RW
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

// fp32 X takes twice the registers: eight waves, so that 256 are there for each
template <int XT>
int launch_rows(const Call &c, int format, bool aff, const Plan &p, hipStream_t stream) {
    constexpr int W = XT == 2 ? 8 : 16;
#define HXQ_RWS(MT_, NS_, SP_, W_) \
    if (p.mt == MT_ && p.ns == NS_ && p.sp == SP_) return launch_fmt<XT, MT_, NS_, SP_, W_>(c, format, aff, p, stream)
    HXQ_RWS(1, 1, 2, W);
    HXQ_RWS(1, 1, 4, W);
    HXQ_RWS(1, 2, 2, W);
    HXQ_RWS(1, 3, 1, W);
    HXQ_RWS(1, 5, 1, W);
    HXQ_RWS(2, 1, 2, W);
    HXQ_RWS(2, 2, 1, W);
    HXQ_RWS(2, 3, 1, W);
    HXQ_RWS(2, 5, 1, 8);
    if constexpr (XT != 2) {
        HXQ_RWS(3, 1, 2, 8);
        HXQ_RWS(3, 2, 1, 8);
        HXQ_RWS(3, 3, 1, 8);
        HXQ_RWS(3, 5, 1, 8);
        HXQ_RWS(4, 1, 2, 8);
        HXQ_RWS(4, 2, 1, 8);
        HXQ_RWS(4, 3, 1, 8);
        HXQ_RWS(4, 5, 1, 8);
    }
#undef HXQ_RWS
    HXQ_REQUIRE(false, "no such few-row plan");
}

// Two blocks per CU: 80 KB of LDS and 128 registers each.
template <int XT>
int launch_grouped(const Call &c, const Grouped &g, bool aff, int blocks, hipStream_t stream) {
#define HXQ_RWG(AF_)                                                                                          \
    hipLaunchKernelGGL((rows_kernel<1, kGroupedSubs, 1, XT, AF_, HXQ_FMT_SCALAR, 8, true>), dim3(blocks),      \
                       dim3(512), 0, stream, c.idx, c.x, c.cb, c.ga, c.M, c.OUT, c.K, c.ngroups, c.gmul, c.a, g)
    if (aff) HXQ_RWG(true); else HXQ_RWG(false);
#undef HXQ_RWG
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

}  // namespace rw
}  // namespace hxq
