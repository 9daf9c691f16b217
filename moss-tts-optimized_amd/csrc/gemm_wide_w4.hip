// INT4 group-32 instances of the wide GEMM tile, and the choice of tile and split for both formats.
#include "gemm_wide_kernel.h"

#include <algorithm>

namespace moss {
namespace {

// Nanoseconds a workgroup takes per K step of 64, by tile (columns JT = 1 .. 5): `alone`, with a CU to
// itself, and `shared`, per workgroup with two on the CU.  From timings of every tile and split at 45
// shapes (M = 5 .. 2048 on the four projections of the 4096 / 12288 model), taken where most CUs have work:
// fewer busy CUs hold a higher clock and a step takes down to 0.75 of this.  By these costs the chosen
// tile and split, with the partial sums' cost, was the best measured one at 34 of the 45 shapes, within 6%
// of it at 41 and within 17% at all.  0: no such instance (R = 2 below 3 token tiles was nowhere the best,
// and INT4 at 2 x 5 spills; e4m3 at 2 x 5 keeps two registers in scratch, outside its loop).
struct StepCost {
    int alone[5], shared[5];
};
constexpr StepCost kStepCost[2][2] = {
    {{{345, 390, 430, 540, 620}, {262, 345, 400, 530, 580}}, {{0, 0, 760, 1000, 0}, {0, 0, 720, 940, 0}}},
    {{{330, 370, 400, 470, 560}, {275, 320, 385, 520, 555}}, {{0, 0, 740, 900, 1056}, {0, 0, 680, 880, 1100}}},
};

// Tiles of the any-shape form: a subset, to keep the library small.
constexpr bool any_tile(int r, int jt) { return r == 1 ? jt != 3 : jt == 4; }

template <int R, int JT>
int launch_tile(WideEpilogue epi, const WidePlan& p, const WideArgs& a, hipStream_t st) {
    const int bn = (epi == kWideSilu ? 64 : 128) * R;
    const dim3 grid((unsigned)(((a.M + 32 * JT - 1) / (32 * JT)) * ((a.N + bn - 1) / bn) * p.split));
#define MOSS_WIDE(...)                                                                                               \
    hipLaunchKernelGGL((gemm_wide_kernel<kInt4G32, R, JT, __VA_ARGS__>), grid, dim3(256), 0, st, (const uint16_t*)a.x,        \
                       (const uint8_t*)a.qw, (const uint16_t*)a.sc, (const uint8_t*)a.zp, a.row_scale, (uint16_t*)a.y, \
                       a.part, a.M, a.N, a.K, p.split, a.qr)
    if constexpr (any_tile(R, JT)) {
        if (p.any) {
            if (epi == kWideSplit) MOSS_WIDE(kWideSplit, true);
            else MOSS_WIDE(kWidePlain, true);
            return moss_launch_status();
        }
    }
    if (epi == kWideSplit) MOSS_WIDE(kWideSplit);
    else if (epi == kWideSilu) MOSS_WIDE(kWideSilu);
    else if (epi == kWideQkRope) MOSS_WIDE(kWideQkRope);
    else MOSS_WIDE(kWidePlain);
#undef MOSS_WIDE
    return moss_launch_status();
}

}  // namespace

// A workgroup's own weight rows (256 of K bytes) and activation rows (160 of 2 K) lie within the 32-bit offsets of
// the buffer instructions.
bool wide_any_shape(int K) { return K % kStep == 0 && 320ll * K < 1ll << 32; }

// Whole blocks of four K steps and 4-output stores; INT4: the 8 zero bytes of every block on one
// nibble side of their 128-group chunk (the last chunk a multiple of 16 groups long, as K / 32 is then).
bool wide_shape(int fmt, int K, int nw) {
    if (nw % 4 || K % (4 * kStep) || !wide_any_shape(K)) return false;
    return fmt == kFp8E4M3 || K / 32 % 16 == 0;
}

// A SiLU workgroup reaches from its gate rows to the up rows, N of K / 2 bytes further on.
bool wide_silu_shape(int K, int N) { return wide_shape(kInt4G32, K, 2 * N) && (long long)N * K < 1ll << 31; }

// The expected time of a plan from timings of 15000 random shapes (2 to 1024 tokens, K = 256 .. 12288, N = 64 ..
// 16384, weights from memory): microseconds to start and to end (base) and per step and round of 256
// workgroups, the partial sums and their reduction, the output and the weights.  Within 4 to 6% of half of the
// times and 15% of nine in ten.
struct FitCost {
    double base[2][5], step[2][5];         // [r - 1][jt - 1]; step 0: no such instance
    double split, part, out, weights;      // part: per 8 bytes at 8 TB/s; out at 4 TB/s; weights at 4.5 TB/s
};
constexpr FitCost kFitAny[2] = {
    {{{2.1, 3.2, 0, 3.6, 3.2}, {0, 0, 0, 5.6, 0}}, {{0.374, 0.430, 0, 0.564, 0.657}, {0, 0, 0, 1.045, 0}}, 2.5, 2.3, 1.4, 0.68},
    {{{2.3, 3.0, 0, 3.2, 3.0}, {0, 0, 0, 4.3, 0}}, {{0.231, 0.264, 0, 0.417, 0.468}, {0, 0, 0, 0.791, 0}}, 2.4, 2.0, 2.4, 0.51},
};
constexpr FitCost kFitFp8 = {{{2.2, 2.5, 2.2, 1.5, 2.0}, {0, 0, 2.9, 3.8, 3.4}},
                             {{0.267, 0.300, 0.383, 0.461, 0.481}, {0, 0, 0.625, 0.721, 0.858}}, 2.0, 1.6, 2.6, 0.51};

double wide_us(int fmt, int M, int K, int nw, const WidePlan& p) {
    const FitCost& c = p.any ? kFitAny[fmt] : kFitFp8;
    const int total = K / kStep;
    const int steps = p.any ? ((total + p.split - 1) / p.split + 3) & ~3 : total / p.split;
    const long wgs = (long)((M + 32 * p.jt - 1) / (32 * p.jt)) * ((nw + 128 * p.r - 1) / (128 * p.r)) * p.split;
    const double mn = (double)M * nw;
    double us = c.base[p.r - 1][p.jt - 1] + (double)((wgs + 255) / 256) * steps * c.step[p.r - 1][p.jt - 1] +
                c.out * mn * 2 / 4e6 + c.weights * nw * K * (fmt == kInt4G32 ? 0.5625 : 1.0) / 4.5e6;
    if (p.split > 1) us += c.split + c.part * p.split * mn * 8 / 8e6;
    return us;
}

// The regular form: the expected time of each tile and split is what the step costs above give for the workgroups per CU,
// not less than the weights' bytes at 4.5 TB/s, and for a split the partial sums written and read back
// (8 bytes each at 8 TB/s: they mostly stay in the last-level cache) and the launch that adds them, 6 us for
// two of 512 x 4096.  A split leaves a share two blocks of K and its partials fit 32 MiB.  The any-shape form, a
// few percent slower a step, is also weighed where the regular one fits: it splits a K of any number of steps
// (e4m3 K = 6400 = 100 steps, M = 10, N = 3000: 31.8 us whole, 11.4 split).  Its shares are whole blocks, so the
// last ones can lie past K and add zeros (65 steps split by 8: shares of 12 steps, the last two empty).
static WidePlan plan(int fmt, int M, int K, int nw, int min_split, int max_split, bool regular) {
    WidePlan best{1, 1, 1, !regular, 1e30};
    const double wbytes = (double)nw * K * (fmt == kInt4G32 ? 0.5625 : 1.0);
    const int total = K / kStep;
    for (int r = 1; r <= 2; ++r)
        for (int jt = 1; jt <= 5; ++jt) {
            const StepCost& c = kStepCost[fmt][r - 1];
            if (!c.alone[jt - 1] || (jt > 1 && 32 * (jt - 1) >= M)) continue;
            const long tiles = (long)((M + 32 * jt - 1) / (32 * jt)) * ((nw + 128 * r - 1) / (128 * r));
            for (int split = min_split; split <= max_split; split *= 2) {
                const bool any = !regular || total % (4 * split);  // the regular form: whole blocks of four steps
                if (any && !any_tile(r, jt)) break;
                const int steps = any ? ((total + split - 1) / split + 3) & ~3 : total / split;
                if (split > 1 && (steps < 8 || (long long)split * M * nw * 4 > 32ll << 20)) break;
                const long per_cu = (tiles * split + 255) / 256;
                if (!regular) {
                    const WidePlan p{r, jt, split, true, 0};
                    const double us = wide_us(fmt, M, K, nw, p);
                    if (us < best.us) best = {r, jt, split, true, us};
                    continue;
                }
                const double ns = (any ? 1.06 : 1.0) * (per_cu == 1 ? c.alone[jt - 1] : (double)per_cu * c.shared[jt - 1]);
                double us = 3.5 + std::max(steps * ns / 1000, wbytes / 4.5e6);
                if (split > 1) us += 2.0 + (double)split * M * nw * 8 / 8e6;
                if (us < best.us) best = {r, jt, split, any, us};
            }
        }
    return best;
}

WidePlan wide_plan(int fmt, int M, int K, int nw, int min_split, int max_split) {
    return plan(fmt, M, K, nw, min_split, max_split, wide_shape(fmt, K, nw));
}

WidePlan wide_plan_any(int fmt, int M, int K, int nw, int max_split) { return plan(fmt, M, K, nw, 1, max_split, false); }

int wide_launch_w4(WideEpilogue epi, const WidePlan& p, const WideArgs& a, hipStream_t st) {
    switch (10 * p.r + p.jt) {
        case 11: return launch_tile<1, 1>(epi, p, a, st);
        case 12: return launch_tile<1, 2>(epi, p, a, st);
        case 13: return launch_tile<1, 3>(epi, p, a, st);
        case 14: return launch_tile<1, 4>(epi, p, a, st);
        case 15: return launch_tile<1, 5>(epi, p, a, st);
        case 23: return launch_tile<2, 3>(epi, p, a, st);
        case 24: return launch_tile<2, 4>(epi, p, a, st);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace moss
