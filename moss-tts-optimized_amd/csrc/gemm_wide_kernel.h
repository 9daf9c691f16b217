// Y[M, N] = X[M, K] . W[N, K]^T on the matrix cores, bf16 activations and outputs, fp32 sums, for
// INT4 group-32 weights and e4m3 weights: the kernel behind gemm_wide_w4.hip and gemm_wide_fp8.hip.
//
// A workgroup of 4 waves takes 128 R weight rows (R = 1, 2) and 32 JT tokens.  The dequantized
// weights are the MFMA's A operand, formed in the registers of the lane that feeds them: wave w owns
// 32-row tiles 128 r + 32 w (r < R) and every token, so a weight is dequantized once per 32 JT tokens
// and an activation read from LDS feeds R MFMAs.  In a K step of 64, lane l takes row l & 31 of a tile
// and the 32-wide half l >> 5 of the step (one INT4 group), 8 weights per MFMA.
//
// Activations go from global memory to LDS without registers (buffer_load_dwordx4 ... lds: lane i
// of an instruction writes bytes 16 i .. + 15 of a 1 KiB span) into a ring of four steps.  Buffer
// instructions, not global_load_lds: the compiler counts the latter as an access of both memories and
// then waits for every load in flight (vmcnt(0)) wherever a code register is first used, which exposed
// the copies' latency in every step.  The same accesses read rows past the end as zero.
// LDS layout: 128 bytes per token row and step, 16-byte chunk c of row r at c ^ (r & 7) ^ ((r >> 3) & 1):
// the 16 lanes that read one chunk of 16 consecutive rows in one LDS cycle hit 16 different bank groups.
//
// What bounds it: the matrix pipe with a full chip (M = 2048, K = 4096, N = 24576, INT4: 357 us, 1150
// TFLOP/s, the pipe busy 74% of the cycles at the 1.5 GHz the chip holds under this load; the tile of
// w4g32_gemm_tdma_kernel 503 us), and with one workgroup per CU the issue of the dequantization (about
// 100 VALU instructions per row tile and step at 5 cycles each for a single wave, 0.3 us per step).
// Three things made it: a step is a chain of R JT MFMAs with the next quarter step's dequantization and
// LDS reads placed between them, about 5 VALU instructions to an MFMA, which hides them (an MFMA alone
// takes 33 cycles, with 6 fma_mix 38); the dequantization avoids v_dot2_f32_bf16, which does not run
// beside an MFMA (one MFMA and 4 of them: 65 cycles, and 4 fma_mix: 36; 402 us against 357); and R = 2
// halves the LDS reads, which at R = 1 take as long as the MFMAs they feed (8 LDS cycles per wave and
// KiB, four waves, against 32).
#pragma once

#include "gemm_wide.h"

#include <type_traits>

namespace moss {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kXcds = 8;
constexpr int kStep = 64;   // K of one step
constexpr int kRing = 4;    // activation buffers; steps per block of scales

__device__ __forceinline__ void pin() { __builtin_amdgcn_sched_barrier(0); }
__device__ __forceinline__ void cbar() { asm volatile("" ::: "memory"); }

// s_waitcnt vmcnt(n)
#define MOSS_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))

template <bool HI>
__device__ __forceinline__ uint32_t fp8x2_to_bf16x2(uint32_t w) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, HI));
}

// 16 bytes per lane straight to lds + 16 lane
__device__ __forceinline__ void lds_copy16(const Span& s, uint16_t* lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(span_rsrc(s), lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ uint32_t load_u16(const Span& s, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b16(span_rsrc(s), voff, soff, 0);
}
__device__ __forceinline__ uint32_t load_u8(const Span& s, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b8(span_rsrc(s), voff, soff, 0);
}
__device__ __forceinline__ uint2 load8(const Span& s, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(span_rsrc(s), voff, soff, 0));
}

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

struct Group {
    float s, bias;  // the group's scale, -(64 + z) s
};
__device__ __forceinline__ Group make_group(uint32_t s_bits, uint32_t z) {
    Group g;
    g.s = __uint_as_float(s_bits << 16);
    g.bias = -(float)(z | 64u) * g.s;
    return g;
}

// bf16 pair u of a code word, bit-exact (the results of dequant_word_mixed): the pair's nibbles are
// moved to bits 4..7 of its halves, where they are the fp16 numbers 64 + q, and
// (64 + q) s - (64 + z) s is exact in fp32.  v_dot2_f32_bf16 would save a shift, but on gfx950 it does
// not run beside an MFMA (one MFMA and four of them take 65 cycles, one MFMA and four fma_mix 36).
template <int U>
__device__ __forceinline__ uint32_t dequant_pair(uint32_t w, uint32_t mask, uint32_t base, const Group& g) {
    const uint32_t v = U == 0 ? w << 4 : w >> (4 * (U - 1));
    const f16x2_t d = __builtin_bit_cast(f16x2_t, (v & mask) | base);
    return pack_bf16x2(__builtin_fmaf((float)d.x, g.s, g.bias), __builtin_fmaf((float)d.y, g.s, g.bias));
}


template <int FMT, int R, int JT, int EPI, bool ANY = false>
__global__ __launch_bounds__(256, 2) void gemm_wide_kernel(
    const uint16_t* __restrict__ X, const uint8_t* qw, const uint16_t* sc, const uint8_t* zp,
    const float* __restrict__ row_scale, uint16_t* __restrict__ Y, float* __restrict__ part, int M, int N, int K,
    int split, QkRope qr) {
    static_assert(!ANY || EPI == kWidePlain || EPI == kWideSplit, "epilogues of whole heads and pairs");
    constexpr bool INT4 = FMT == kInt4G32, SZ = INT4 && ANY;  // SZ: scale and zero loaded with each step's codes
    constexpr int BM = 32 * JT, BN = (EPI == kWideSilu ? 64 : 128) * R;
    constexpr int W = 2;                   // steps the codes travel ahead (divides kRing)
    constexpr int CW = INT4 ? 1 : 2;        // code loads per row tile and step
    constexpr int CL = SZ ? 3 : CW;         // weight loads per row tile and step
    constexpr int kTile = 2048 * JT;    // bf16 values of one step's activations
    __shared__ __attribute__((aligned(1024))) uint16_t X0[kTile];
    __shared__ __attribute__((aligned(1024))) uint16_t X1[kTile];
    __shared__ __attribute__((aligned(1024))) uint16_t X2[kTile];
    __shared__ __attribute__((aligned(1024))) uint16_t X3[kTile];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mt = (M + BM - 1) / BM, wgs = gridDim.x;
    const int xcd = blockIdx.x % kXcds;
    int t = xcd * (wgs / kXcds) + min(xcd, wgs % kXcds) + blockIdx.x / kXcds;
    const int m0 = (t % mt) * BM;
    t /= mt;
    const int z = EPI == kWideSplit ? t % split : 0;
    const int n0 = (EPI == kWideSplit ? t / split : t) * BN;
    const int G = K >> 5, total = K / kStep;
    const int share = EPI == kWideSplit ? (ANY ? (total + split - 1) / split : total / split) : total;
    const int steps = ANY ? (share + kRing - 1) & ~(kRing - 1) : share;
    const int kbase = z * steps * kStep;
    // ANY: steps past the end of K read zeros, through empty spans (their uniform offset is 0 then, so
    // that no range check can wrap around)
    auto live = [&](int step) { return !ANY || z * steps + step < total; };
    auto within = [&](const Span& s, int step) { return Span{s.base, live(step) ? s.bytes : 0u}; };
    auto at = [&](uint32_t soff, int step) { return live(step) ? soff : 0u; };

    const int half = lane >> 5;
    // activations: rows of the tile past M read as zero
    const Span xspan{X + (size_t)m0 * K, (uint32_t)min(BM, M - m0) * (uint32_t)K * 2u};
    uint32_t xoff[JT];
#pragma unroll
    for (int c = 0; c < JT; ++c) {
        const int r8 = JT * wave + c, r = 8 * r8 + (lane >> 3);
        xoff[c] = 2u * (uint32_t)(r * K) + 16u * (uint32_t)((lane & 7) ^ ((lane >> 3) & 7) ^ (r8 & 1));
    }
    auto copy_x = [&](uint16_t* buf, int step) {
#pragma unroll
        for (int c = 0; c < JT; ++c)
            lds_copy16(within(xspan, step), buf + 512 * (JT * wave + c), xoff[c],
                       at(2 * (kbase + kStep * step), step));
    };
    const int swz = (lane & 7) ^ ((lane >> 3) & 1);
    uint32_t roff[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        roff[kk] = 128u * (uint32_t)(lane & 31) + 16u * (uint32_t)((4 * half + kk) ^ swz);
    auto read_b = [&](const uint16_t* buf, int kk, int j) {
        return *reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const char*>(buf) + roff[kk] + 4096 * j);
    };

    // weights: row tile r of this wave is rows n0 + 128 r + 32 wave .. + 31; with the SiLU epilogue
    // gate rows n0 + 64 r + 16 wave .. + 15 and the up rows of the same outputs, N further on, so
    // that a lane's accumulators e and e + 8 are the gate and the up sum of one output.  Rows past the
    // weight's last one read as zero.
    const uint32_t rowb = INT4 ? (uint32_t)G * 16u : (uint32_t)K;
    const uint32_t rows = EPI == kWideSilu ? (uint32_t)(2 * N - n0) : (uint32_t)min(BN, N - n0);
    const Span wspan{qw + (size_t)n0 * rowb, rows * rowb};
    const Span sspan{sc + (INT4 ? (size_t)n0 * G : 0), rows * (uint32_t)G * 2u};
    const Span zspan{zp + (INT4 ? (size_t)n0 * (G >> 1) : 0), rows * (uint32_t)(G >> 1)};
    const uint32_t wlane = EPI == kWideSilu ? (uint32_t)(16 * wave + (lane & 15) + ((lane >> 4) & 1) * N)
                                            : (uint32_t)(32 * wave + (lane & 31));
    // A row tile that starts past the last row reads tile 0's rows again and stores none of them: a uniform
    // offset at or past the end of a span would wrap the range check (offset >= bytes - uniform offset).
    auto tile_row = [&](int r) {
        const uint32_t row = (EPI == kWideSilu ? 64u : 128u) * r;
        return row < rows ? row : 0u;
    };
    const uint32_t woff = wlane * rowb + (INT4 ? 16u : 32u) * half;
    u32x4_t cw[W][R][CW];
    uint32_t cs[W][R], cz[W][R];  // SZ: the scale, the byte that holds the zero point
    u32x4_t ts[R], tsn[R];
    uint2 tz[R], tzn[R];
    uint32_t zsh = 0, zshn = 0;
    // SZ: where this lane's zero point lies (group g of the row), and its nibble's shift
    auto zero_at = [&](int step, uint32_t& sh) {
        int zb;
        zero_loc(min((kbase >> 5) + 2 * step + half, G - 1), G, zb, sh);
        return (uint32_t)zb;
    };
    auto load_w = [&](int slot, int step) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int c = 0; c < CW; ++c)
                cw[slot][r][c] = load16(within(wspan, step), woff + 16 * c,
                                        at(tile_row(r) * rowb + (INT4 ? kbase / 2 + 32 * step : kbase + 64 * step), step));
            if constexpr (SZ) {
                uint32_t sh;
                cs[slot][r] = load_u16(within(sspan, step), wlane * (uint32_t)(2 * G) + 2 * half,
                                       at(tile_row(r) * (uint32_t)(2 * G) + kbase / 16 + 4 * step, step));
                cz[slot][r] = load_u8(within(zspan, step), wlane * (uint32_t)(G >> 1) + zero_at(step, sh),
                                      at(tile_row(r) * (uint32_t)(G >> 1), step));
            }
        }
    };
    auto load_blk = [&](u32x4_t (&s)[R], uint2 (&zz)[R], uint32_t& sh, int blk) {
        if constexpr (INT4 && !SZ) {
            int zb;
            zero_loc((kbase >> 5) + 8 * blk, G, zb, sh);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                s[r] = load16(sspan, wlane * (uint32_t)(2 * G), tile_row(r) * (uint32_t)(2 * G) + kbase / 16 + 16 * blk);
                zz[r] = load8(zspan, wlane * (uint32_t)(G >> 1), tile_row(r) * (uint32_t)(G >> 1) + zb);
            }
        }
    };
    f32x16_t acc[R][JT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[r][j][e] = 0.f;

    const int blocks = steps / kRing;
    load_blk(ts, tz, zsh, 0);
    // the loads in the order the steps before step 0 would issue them, so that the steps' wait counts
    // hold from the start
    uint16_t* const ring[3] = {X0, X1, X2};
#pragma unroll
    for (int v = -kRing; v < 0; ++v) {
        if (v >= 1 - kRing) copy_x(ring[(v + kRing - 1) % 3], v + kRing - 1);
        cbar();
        if (v + W >= 0) load_w(v + W, v + W);
        cbar();
    }
    MOSS_WAIT_VM(JT + 2 * R * CL);  // steps 0 and 1 have landed
    __builtin_amdgcn_s_barrier();
    cbar();
    const MixedUnpack mu = make_mixed_unpack();

    Group gd[R];
    auto group = [&](auto ic, const u32x4_t (&s)[R], const uint2 (&zz)[R], uint32_t sh, int step) {
        constexpr int i = decltype(ic)::value;
        if constexpr (SZ) {
            uint32_t lsh;
            zero_at(step, lsh);
#pragma unroll
            for (int r = 0; r < R; ++r) gd[r] = make_group(cs[i % W][r], (cz[i % W][r] >> lsh) & 15u);
        } else if constexpr (INT4) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t zw = i < 2 ? zz[r].x : zz[r].y;
                gd[r] = make_group(s[r][i] >> (16 * half), (zw >> (8 * (2 * (i & 1) + half) + sh)) & 15u);
            }
        }
    };
    // pair u of the A operand for word kk of this lane's group
    auto pair = [&](auto uc, const u32x4_t (&w)[R][CW], int kk, int r) -> uint32_t {
        constexpr int u = decltype(uc)::value;
        if constexpr (INT4) return dequant_pair<u>(w[r][0][kk], mu.mask_hi, mu.f16_bias, gd[r]);
        else return fp8x2_to_bf16x2<u % 2 == 1>(w[r][kk >> 1][2 * (kk & 1) + u / 2]);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    using No = std::false_type;
    using Yes = std::true_type;
    u32x4_t a[R];
    bf16x8_t b[JT];
    group(S0{}, ts, tz, zsh, 0);
#pragma unroll
    for (int j = 0; j < JT; ++j) b[j] = read_b(X0, 0, j);
#pragma unroll
    for (int r = 0; r < R; ++r)
        a[r] = u32x4_t{pair(S0{}, cw[0], 0, r), pair(S1{}, cw[0], 0, r), pair(S2{}, cw[0], 0, r), pair(S3{}, cw[0], 0, r)};

    auto step = [&](auto ic, auto lc, int blk, const uint16_t* rd, const uint16_t* rdn, uint16_t* wr) {
        constexpr int i = decltype(ic)::value;
        constexpr bool LAST = decltype(lc)::value;
        const int s = blk * kRing + i;
        constexpr bool copies = !LAST || i == 0;
        constexpr bool codes = !LAST || i + W < kRing;
        if constexpr (copies) copy_x(wr, s + kRing - 1);
        cbar();
        auto quarter = [&](auto kc) {
            constexpr int kk = decltype(kc)::value;
            constexpr bool more = !(LAST && i == kRing - 1 && kk == 3);  // another quarter follows
            constexpr int nk = (kk + 1) & 3;
            if constexpr (kk == 3 && more) {
                if constexpr (INT4 && !SZ && i == kRing - 1) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        ts[r] = tsn[r];
                        tz[r] = tzn[r];
                    }
                    zsh = zshn;
                }
                group(std::integral_constant<int, (i + 1) % kRing>{}, ts, tz, zsh, s + 1);
            }
            const auto& w = cw[(kk == 3 ? i + 1 : i) % W];
            u32x4_t an[R];
            auto piece = [&](int n) {  // one of 4 R pairs
                const int r = n >> 2, u = n & 3;
                an[r][u] = u == 0 ? pair(S0{}, w, nk, r) : u == 1 ? pair(S1{}, w, nk, r)
                         : u == 2 ? pair(S2{}, w, nk, r) : pair(S3{}, w, nk, r);
            };
            int n = 0;
#pragma unroll
            for (int j = 0; j < JT; ++j) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[r]), b[j],
                                                                       acc[r][j], 0, 0, 0);
                    if (r == R - 1 && more) b[j] = read_b(kk == 3 ? rdn : rd, nk, j);
                    const int upto = 4 * R * (j * R + r + 1) / (R * JT);
#pragma unroll
                    for (; n < upto; ++n)
                        if (more) piece(n);
                    pin();
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (more) a[r] = an[r];
            if constexpr (kk == 2) {
                // the step's codes have all been taken
                if constexpr (codes) load_w(i % W, s + W);
                if constexpr (INT4 && !SZ && !LAST && i == 0) load_blk(tsn, tzn, zshn, blk + 1);
                cbar();
                pin();
            }
        };
        quarter(S0{});
        quarter(S1{});
        quarter(S2{});
        quarter(S3{});
        // the copies of step s + 2, issued in step s - 1, have landed: this many loads follow them
        if constexpr (!LAST || i < 2) {
            constexpr int C = R * CL;
            constexpr int n = !LAST ? JT + 2 * C : i == 0 ? JT + (1 + (W < 4)) * C : ((W < 4) + (W < 3)) * C;
            MOSS_WAIT_VM(n);
            __builtin_amdgcn_s_barrier();
        }
        cbar();
    };
    int blk = 0;
    for (; blk < blocks - 1; ++blk) {
        step(S0{}, No{}, blk, X0, X1, X3);
        step(S1{}, No{}, blk, X1, X2, X0);
        step(S2{}, No{}, blk, X2, X3, X1);
        step(S3{}, No{}, blk, X3, X0, X2);
    }
    step(S0{}, Yes{}, blk, X0, X1, X3);
    step(S1{}, Yes{}, blk, X1, X2, X0);
    step(S2{}, Yes{}, blk, X2, X3, X1);
    step(S3{}, Yes{}, blk, X3, X0, X2);

    if constexpr (EPI == kWideQkRope) {
        // One head per 128-row tile.  The bf16 products are staged token-major (token t of tile j in
        // buffer (t / 8) % 4, 8-byte chunk c at c ^ (t & 31)), then each token row goes through
        // head4_norm_rope on 16 lanes.
        constexpr int QH = 32, KH = 8, D = 128, RP = 16, PASSES = BM / RP;
        const int head0 = n0 / D, jl = tid & 15;
        auto chunk = [&](int r, int row, int c) {
            const int a = (row >> 3) & 3;
            uint16_t* b = a == 0 ? X0 : a == 1 ? X1 : a == 2 ? X2 : X3;
            return reinterpret_cast<uint2*>(b + ((r * JT + (row >> 5)) * 8 + (row & 7)) * 128 + 4 * (c ^ (row & 31)));
        };
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int j = 0; j < JT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint2 o;
                    o.x = pack_bf16x2(acc[r][j][4 * q], acc[r][j][4 * q + 1]);
                    o.y = pack_bf16x2(acc[r][j][4 * q + 2], acc[r][j][4 * q + 3]);
                    *chunk(r, 32 * j + (lane & 31), 8 * wave + 2 * q + half) = o;
                }
        __syncthreads();
        auto ld4 = [](const uint16_t* p) { return *reinterpret_cast<const uint2*>(p); };
#pragma unroll
        for (int pass = 0; pass < PASSES; ++pass) {
            const int row = RP * pass + (tid >> 4), m = m0 + row;
            if (m >= M) continue;  // whole 16-lane groups
            const int64_t pos = min(max(qr.positions[m], (int64_t)0), (int64_t)(qr.L - 1));
            if (head0 >= QH + KH) {  // value heads: the rounded products as they are
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    uint16_t* vd = qr.v_cache + ((size_t)(head0 + r - QH - KH) * qr.L + pos) * D;
                    *reinterpret_cast<uint2*>(vd + 4 * jl) = *chunk(r, row, jl);
                    *reinterpret_cast<uint2*>(vd + 64 + 4 * jl) = *chunk(r, row, 16 + jl);
                }
                continue;
            }
            const uint16_t* wt = head0 < QH ? qr.q_weight : qr.k_weight;
            const uint2 wa = ld4(wt + 4 * jl), wb = ld4(wt + 64 + 4 * jl);
            const uint16_t* cr = qr.cos_t + (size_t)pos * D;
            const uint16_t* sr = qr.sin_t + (size_t)pos * D;
            const uint2 ca = ld4(cr + 4 * jl), cb = ld4(cr + 64 + 4 * jl);
            const uint2 sa = ld4(sr + 4 * jl), sb = ld4(sr + 64 + 4 * jl);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                uint2 lo, hi;
                head4_norm_rope(*chunk(r, row, jl), *chunk(r, row, 16 + jl), wa, wb, ca, cb, sa, sb, qr.eps, lo, hi);
                const int head = head0 + r;
                uint16_t* dst = head < QH ? Y + ((size_t)m * QH + head) * D
                                          : qr.k_cache + ((size_t)(head - QH) * qr.L + pos) * D;
                *reinterpret_cast<uint2*>(dst + 4 * jl) = lo;
                *reinterpret_cast<uint2*>(dst + 64 + 4 * jl) = hi;
            }
        }
        return;
    }
    // C[n][m] of a 32 x 32 tile: lane l, element e -> n row 8 (e / 4) + 4 (l / 32) + e % 4, m column
    // l % 32; the four e of a quad are consecutive n
    if constexpr (ANY) {
        if (N % 4 || (EPI == kWidePlain && reinterpret_cast<uintptr_t>(Y) % 8)) {
            // No quads: a store of one value per lane would touch a row per lane, so each 128-row half of the tile
            // goes through the LDS of the ring, fp32 by token row (row t in buffer (t / 8) % 4, 16-byte chunk c at
            // c ^ (t & 31)), and leaves row by row (M = 595, K = 320, N = 12317: 32.2 -> 21.4 us; M = 150, K = 4160,
            // N = 1001: 17.0 -> 14.0).
            auto chunk = [&](int row, int c) {
                const int b = (row >> 3) & 3;
                uint16_t* x = b == 0 ? X0 : b == 1 ? X1 : b == 2 ? X2 : X3;
                return reinterpret_cast<float*>(x) + ((row >> 5) * 8 + (row & 7)) * 128 + 4 * (c ^ (row & 31));
            };
#pragma unroll
            for (int r = 0; r < R; ++r) {
                __syncthreads();
#pragma unroll
                for (int j = 0; j < JT; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<float4*>(chunk(32 * j + (lane & 31), 8 * wave + 2 * q + half)) = make_float4(
                            acc[r][j][4 * q], acc[r][j][4 * q + 1], acc[r][j][4 * q + 2], acc[r][j][4 * q + 3]);
                __syncthreads();
                const int nr = n0 + 128 * r, nn = min(128, N - nr), rows = min(BM, M - m0);
                if (nn <= 0) break;
                const bool v0 = lane < nn, v1 = lane + 64 < nn;
                float s0 = 1.f, s1 = 1.f;
                if (!INT4 && EPI == kWidePlain && row_scale) {
                    if (v0) s0 = row_scale[nr + lane];
                    if (v1) s1 = row_scale[nr + 64 + lane];
                }
                for (int row = wave; row < rows; row += 4) {
                    const float c0 = chunk(row, lane >> 2)[lane & 3], c1 = chunk(row, 16 + (lane >> 2))[lane & 3];
                    const size_t o = (size_t)(m0 + row) * N + nr + lane;
                    if constexpr (EPI == kWideSplit) {
                        float* out = part + (size_t)z * M * N + o;
                        if (v0) out[0] = c0;
                        if (v1) out[64] = c1;
                    } else {
                        if (v0) Y[o] = f32_to_bf16(c0 * s0);
                        if (v1) Y[o + 64] = f32_to_bf16(c1 * s1);
                    }
                }
            }
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < JT; ++j) {
        const int m = m0 + 32 * j + (lane & 31);
        if (m >= M) continue;
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int q = 0; q < (EPI == kWideSilu ? 2 : 4); ++q) {
                const int n = n0 + (EPI == kWideSilu ? 64 * r + 16 * wave : 128 * r + 32 * wave) + 8 * q + 4 * half;
                if (n >= N) continue;  // N % 4 == 0: a quad is all in range or all out
                const f32x16_t& c = acc[r][j];
                const float v0 = c[4 * q], v1 = c[4 * q + 1], v2 = c[4 * q + 2], v3 = c[4 * q + 3];
                if constexpr (EPI == kWideSplit) {
                    *reinterpret_cast<float4*>(part + ((size_t)z * M + m) * N + n) = make_float4(v0, v1, v2, v3);
                } else {
                    uint2 o;
                    if constexpr (EPI == kWideSilu) {
                        const int u = 4 * q + 8;
                        o.x = silu_mul_rounded_bits(v0, c[u]) | ((uint32_t)silu_mul_rounded_bits(v1, c[u + 1]) << 16);
                        o.y = silu_mul_rounded_bits(v2, c[u + 2]) | ((uint32_t)silu_mul_rounded_bits(v3, c[u + 3]) << 16);
                    } else {
                        float4 s = make_float4(1.f, 1.f, 1.f, 1.f);
                        if (!INT4 && row_scale)
                            s = make_float4(row_scale[n], row_scale[n + 1], row_scale[n + 2], row_scale[n + 3]);
                        o.x = INT4 ? pack_bf16x2(v0, v1) : pack_bf16x2(v0 * s.x, v1 * s.y);
                        o.y = INT4 ? pack_bf16x2(v2, v3) : pack_bf16x2(v2 * s.z, v3 * s.w);
                    }
                    *reinterpret_cast<uint2*>(Y + (size_t)m * N + n) = o;
                }
            }
        }
    }
}

}  // namespace
}  // namespace moss
