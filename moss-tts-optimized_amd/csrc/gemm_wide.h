// The prompt GEMM tile whose waves own 32 or 64 weight rows over 32 JT tokens (gemm_wide_kernel.h).
#pragma once

#include "common.h"

namespace moss {

enum WeightFormat { kInt4G32 = 0, kFp8E4M3 = 1 };

// The q/k head RMSNorm + RoPE and K/V write that end the prompt pass's QKV projection.
struct QkRope {
    const uint16_t* q_weight;  // [128] head RMSNorm weights
    const uint16_t* k_weight;
    const uint16_t* cos_t;  // [L, 128], row = position
    const uint16_t* sin_t;
    uint16_t* k_cache;  // [8, L, 128]
    uint16_t* v_cache;
    const int64_t* positions;  // [M], clamped into 0 .. L - 1
    int L;
    float eps;
};

enum WideEpilogue { kWidePlain = 0, kWideSplit = 1, kWideSilu = 2, kWideQkRope = 3 };

// Tile and K split of one call: 128 r weight rows x 32 jt tokens per workgroup, split workgroups per tile.
struct WidePlan {
    int r, jt, split;
    bool any;   // the form for any K % 64 == 0 and any N
    double us;  // expected time
};

struct WideArgs {
    const void *x, *qw, *sc, *zp;  // sc, zp: INT4 only
    const float* row_scale;        // e4m3 only, may be null
    void* y;                       // bf16 [M, N] (kWideQkRope: the query heads)
    float* part;                   // kWideSplit: fp32 [split, M, N]
    int M, K, N;                   // kWideSilu: outputs N, weight rows 2 N
    QkRope qr;
};

// Shapes the tile takes: whole blocks of K and 4-output stores (the fused epilogues need them), or any
// K % 64 == 0 and any N; nw: weight rows.
bool wide_shape(int fmt, int K, int nw);
bool wide_any_shape(int K);
bool wide_silu_shape(int K, int N);  // the SiLU form, 2 N weight rows
// The tile and split with the least expected time, min_split <= split <= max_split (powers of two; 1 and 1: K
// whole).
WidePlan wide_plan(int fmt, int M, int K, int nw, int min_split, int max_split);
// The form for any K % 64 == 0 and any N of the plan above, for operands without the regular one's alignment.
WidePlan wide_plan_any(int fmt, int M, int K, int nw, int max_split);
// The expected time of a plan on the scale of the LDS tiles' (lds_us in w4g32_gemm.hip): e4m3, and INT4 in the
// any-shape form.
double wide_us(int fmt, int M, int K, int nw, const WidePlan& p);
int wide_launch_w4(WideEpilogue epi, const WidePlan& p, const WideArgs& a, hipStream_t st);
int wide_launch_fp8(WideEpilogue epi, const WidePlan& p, const WideArgs& a, hipStream_t st);

}  // namespace moss
