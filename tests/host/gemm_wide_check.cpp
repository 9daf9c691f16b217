// Host checks of the wide GEMM tile, compiled against hip_on_host.h.
//   bounds          every instance, over remainders of M, N and K: addresses of every read, and stores
//   plan            reads "format M K N" lines (0 INT4, 1 e4m3, 2 INT4 gate||up + SiLU of N outputs, 3 INT4 q||k||v +
//                   RoPE), prints what the dispatch picks for each: r, jt, split, any, workspace
//                   (the LDS tiles: -rows, columns, split; neither: 0)
#include "w4g32_gemm.hip"

namespace moss {
int qk_rope_from_parts(const float*, int, const void*, const void*, const void*, const void*, void*, void*, void*,
                       const void*, int, int, float, hipStream_t) { return 0; }
int addnorm_from_parts(const float*, int, const void*, const void*, void*, void*, int, int, float, hipStream_t) { return 0; }
int add_rmsnorm_inplace(void*, const void*, const void*, void*, int, int, float, hipStream_t) { return 0; }
bool w4g32_gemv_tokens_shape(int M, int K) { return M >= 2 && M <= 4 && K <= 16384; }
int w4g32_gemv_tokens_launch(const void*, const void*, const void*, const void*, void*, int, int, int, hipStream_t) { return 0; }
}  // namespace moss
extern "C" int moss_silu_mul(const void*, void*, int, int, void*) { return 0; }
extern "C" int moss_rmsnorm(const void*, const void*, const void*, void*, void*, int, int, float, void*) { return 0; }
extern "C" int moss_qk_norm_rope_kv(const void*, const void*, const void*, const void*, const void*, void*, void*, void*,
                                    const void*, int, int, float, int, void*) { return 0; }

// An array whose neighbours on both sides are watched.
template <class T>
struct Watched {
    static constexpr size_t kGuard = 4096;
    std::vector<T> all;
    size_t n;
    Watched(size_t n_) : all(n_ + 2 * kGuard, (T)77), n(n_) {}
    T* data() { return all.data() + kGuard; }
    bool intact() const {
        for (size_t i = 0; i < kGuard; ++i)
            if (all[i] != (T)77 || all[kGuard + n + i] != (T)77) return false;
        return true;
    }
};

// Never touched, so a large one costs no memory.
struct Untouched {
    char* p;
    explicit Untouched(size_t bytes) : p((char*)malloc(std::max<size_t>(bytes, 1))) { operands.push_back({p, bytes}); }
    ~Untouched() { free(p); }
    Untouched(const Untouched&) = delete;
    const char* data() const { return p; }
};

static int runs;
static bool check(int fmt, int r, int jt, int split, bool any, WideEpilogue epi, int M, int N, int K) {
    const WidePlan p{r, jt, split, any, 0};
    const int nw = epi == kWideSilu ? 2 * N : N, G = K / 32, L = 64, before = (int)violations;
    const bool int4 = fmt == kInt4G32;
    operands.clear();
    const Untouched x((size_t)M * K * 2), qw((size_t)nw * K / (int4 ? 2 : 1)), sc(int4 ? (size_t)nw * G * 2 : 0),
        zp(int4 ? (size_t)nw * G / 2 : 0);
    Watched<uint16_t> y((size_t)M * (epi == kWideQkRope ? 4096 : N)), kc(8 * L * 128), vc(8 * L * 128);
    Watched<float> part(epi == kWideSplit ? (size_t)p.split * M * N : 1);
    std::vector<float> scale(int4 ? 1 : N);
    std::vector<uint16_t> row(128), table(L * 128);
    std::vector<int64_t> pos(M, L - 1);
    const QkRope qr{row.data(), row.data(), table.data(), table.data(), kc.data(), vc.data(), pos.data(), L, 1e-6f};
    const WideArgs a{x.data(), qw.data(), sc.data(), zp.data(), int4 ? nullptr : scale.data(), y.data(), part.data(), M, K, N, qr};
    const int rc = int4 ? wide_launch_w4(epi, p, a, nullptr) : wide_launch_fp8(epi, p, a, nullptr);
    ++runs;
    const bool ok = rc == 0 && violations == before && y.intact() && part.intact() && kc.intact() && vc.intact();
    if (!ok)
        printf("FAIL format %d tile %d x %d any %d split %d epilogue %d M %d N %d K %d: rc %d\n", fmt, p.r, p.jt, p.any,
               p.split, epi, M, N, K, rc);
    return ok;
}

static bool bounds() {
    static const int tiles[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 5}, {2, 3}, {2, 4}, {2, 5}};
    bool ok = true;
    for (int fmt : {(int)kInt4G32, (int)kFp8E4M3})
        for (auto& t : tiles) {
            const int r = t[0], jt = t[1], bn = 128 * r;
            if (fmt == kInt4G32 && r == 2 && jt == 5) continue;
            // one row past a tile, rows that end in its first and in its second row tile, one short of it
            for (int n : {4, 124, 128, 132, 252, 256, bn + 4, bn + 128, bn + 132, 2 * bn - 4}) {
                const int m = 32 * jt + 1;
                ok &= check(fmt, r, jt, 1, false, kWidePlain, m, n, 512);
                ok &= check(fmt, r, jt, 2, false, kWideSplit, m, n, 512);
                if (fmt == kInt4G32) ok &= check(fmt, r, jt, 1, false, kWideSilu, m, n, 512);
            }
            if (fmt == kInt4G32) ok &= check(fmt, r, jt, 1, false, kWideQkRope, 32 * jt - 1, 6144, 512);
            if (r == 1 ? jt == 3 : jt != 4) continue;  // no any-shape instance
            for (int n : {1, 127, 128, 129, 255, bn + 1, bn + 128, 2 * bn - 1})
                for (int k : {64, 576}) {
                    ok &= check(fmt, r, jt, 1, true, kWidePlain, 32 * jt - 1, n, k);
                    // shares of K past its end among them
                    for (int split : {2, 4}) ok &= check(fmt, r, jt, split, true, kWideSplit, 33, n, k);
                }
        }
    // weights past 4 GiB: the last workgroups' rows
    last_blocks = 3;
    for (int fmt : {(int)kInt4G32, (int)kFp8E4M3})
        for (int r : {1, 2}) {
            const int n = (1 << (fmt == kInt4G32 ? 21 : 20)) + 132;
            ok &= check(fmt, r, 4, 1, false, kWidePlain, 3, n, 4096);
            ok &= check(fmt, r, 4, 2, true, kWideSplit, 3, n + 1, 4096);
        }
    printf("%d launches\n", runs);
    return ok;
}

int main(int argc, char** argv) {
    if (argc > 1 && !strcmp(argv[1], "bounds")) return bounds() ? 0 : 1;
    run_launches = false;
    int fmt, M, K, N;
    const void* p = (const void*)4096;  // aligned for everything, never read
    while (scanf("%d %d %d %d", &fmt, &M, &K, &N) == 4) {
        WidePlan w{};
        const long long ws = gemm_workspace_bytes(M, K, fmt == 2 ? 2 * N : N);
        if (fmt == 2) {  // gate||up with the SiLU epilogue, N outputs
            const bool fused = silu_fusable_shape(M, K, N);
            if (fused && wide_silu_shape(K, N)) w = wide_plan(kInt4G32, M, K, 2 * N, 1, 1);
            else if (fused || tokens_gemv(M, K, p, p) || !wide_silu_shape(K, N) ||
                     !choose_wide(kInt4G32, M, K, 2 * N, p, p, p, p, p, p, ws, w) || w.split > 1 || w.any) w = WidePlan{};
        } else if (fmt == 3) {  // q||k||v with the q/k norm + RoPE epilogue
            if (qk_rope_fusable_shape(M, K) && wide_shape(kInt4G32, K, kQkvN)) w = wide_plan(kInt4G32, M, K, kQkvN, 1, 1);
        } else if (!(fmt == kInt4G32 && tokens_gemv(M, K, p, p))) {
            if (!choose_wide(fmt, M, K, N, p, p, p, p, p, p, ws, w)) {
                w = WidePlan{};
                if (!stream_shape(fmt, M, K, N, p, p, p, p, p)) {
                    const Plan t = plan_gemm(M, K, N, fmt == kInt4G32);
                    w = WidePlan{t.reg ? 0 : -t.bm, t.bn, t.split, false, 0};
                }
            }
        }
        printf("%d %d %d %d %lld\n", w.r, w.jt, w.split, (int)w.any, ws);
    }
    return 0;
}
