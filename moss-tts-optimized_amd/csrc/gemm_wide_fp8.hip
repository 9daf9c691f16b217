// e4m3 instances of the wide GEMM tile (weights converted exactly to bf16, row scale in the epilogue).
#include "gemm_wide_kernel.h"

namespace moss {
namespace {

template <int R, int JT>
int launch_tile(WideEpilogue epi, const WidePlan& p, const WideArgs& a, hipStream_t st) {
    const dim3 grid((unsigned)(((a.M + 32 * JT - 1) / (32 * JT)) * ((a.N + 128 * R - 1) / (128 * R)) * p.split));
#define MOSS_WIDE(...)                                                                                               \
    hipLaunchKernelGGL((gemm_wide_kernel<kFp8E4M3, R, JT, __VA_ARGS__>), grid, dim3(256), 0, st, (const uint16_t*)a.x,        \
                       (const uint8_t*)a.qw, (const uint16_t*)nullptr, (const uint8_t*)nullptr, a.row_scale,          \
                       (uint16_t*)a.y, a.part, a.M, a.N, a.K, p.split, a.qr)
    if constexpr (R == 1 ? JT != 3 : JT == 4) {  // any_tile of gemm_wide_w4.hip
        if (p.any) {
            if (epi == kWideSplit) MOSS_WIDE(kWideSplit, true);
            else MOSS_WIDE(kWidePlain, true);
            return moss_launch_status();
        }
    }
    if (epi == kWideSplit) MOSS_WIDE(kWideSplit);
    else MOSS_WIDE(kWidePlain);
#undef MOSS_WIDE
    return moss_launch_status();
}

}  // namespace

int wide_launch_fp8(WideEpilogue epi, const WidePlan& p, const WideArgs& a, hipStream_t st) {
    switch (10 * p.r + p.jt) {
        case 11: return launch_tile<1, 1>(epi, p, a, st);
        case 12: return launch_tile<1, 2>(epi, p, a, st);
        case 13: return launch_tile<1, 3>(epi, p, a, st);
        case 14: return launch_tile<1, 4>(epi, p, a, st);
        case 15: return launch_tile<1, 5>(epi, p, a, st);
        case 23: return launch_tile<2, 3>(epi, p, a, st);
        case 24: return launch_tile<2, 4>(epi, p, a, st);
        case 25: return launch_tile<2, 5>(epi, p, a, st);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace moss
