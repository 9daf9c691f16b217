"""The wide GEMM tile against the float32 product of the dequantized weights: one token short of and past a
tile, rows past the last tile, K of one block and K splits; every instance of it that the dispatch picks
(INSTANCES), its SiLU and q/k-norm epilogues among them; weights past 2 GiB; and the LDS tiles that other
calls stay in (TILES_IN_LDS).

Tolerance: the output is one bf16 rounding (at most 2^-9 of its value) of a float32 sum whose order
differs from the reference's (K 2^-24 of the sum of magnitudes at most, here 1e-3 of an output of
typical size)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _packed(n, k, seed, dev):
    from moss_tts._runtime import w4g32

    g = torch.Generator(device=dev).manual_seed(seed)
    return w4g32.quantize_minmax(torch.randn((n, k), device=dev, generator=g) * 0.02), g


def _close(y, ref):
    rms = ref.square().mean().sqrt()
    assert ((y.float() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-3 * rms).all()


SHAPES = [(1, 512, 128), (31, 512, 132), (33, 1024, 260), (65, 512, 516), (96, 4096, 1028), (97, 4096, 2052),
          (129, 4096, 4096), (161, 12288, 2052), (320, 4096, 6144), (301, 4608, 4100), (1000, 1024, 8200),
          (513, 4096, 12292), (6, 12288, 4096)]
# the any-shape form: K of one step to many with and without a rest, any N, a K split with a rest
ANY = [(5, 64, 5), (33, 192, 130), (16, 320, 64), (65, 4160, 1001), (150, 4032, 515), (301, 12224, 258), (700, 1088, 4099)]


# One call of every instance: (0 INT4, 1 e4m3, 2 INT4 gate||up + SiLU, 3 INT4 q||k||v + RoPE; 128-row tiles, 32-token
# tiles, any-shape form, K split): (M, K, N).  test_gemm_wide_bounds.py holds the list against the dispatch.
INSTANCES = {
    (0, 1, 1, 0, 0): (7, 512, 100), (0, 1, 1, 0, 1): (20, 2048, 24), (0, 1, 1, 1, 0): (19, 256, 59),
    (0, 1, 1, 1, 1): (6, 3584, 59), (0, 1, 2, 0, 0): (170, 512, 5508), (0, 1, 2, 0, 1): (70, 2048, 3292),
    (0, 1, 2, 1, 0): (74, 256, 13121), (0, 1, 2, 1, 1): (1042, 4224, 41), (0, 1, 3, 0, 0): (72, 512, 25856),
    (0, 1, 3, 0, 1): (261, 1024, 3812), (0, 1, 4, 0, 0): (871, 512, 3236), (0, 1, 4, 0, 1): (211, 4096, 1716),
    (0, 1, 4, 1, 0): (126, 256, 23257), (0, 1, 4, 1, 1): (354, 7488, 271), (0, 1, 5, 0, 0): (464, 512, 8344),
    (0, 1, 5, 0, 1): (132, 9216, 5708), (0, 1, 5, 1, 0): (577, 256, 3473), (0, 1, 5, 1, 1): (659, 11776, 263),
    (0, 2, 3, 0, 0): (694, 512, 6624), (0, 2, 4, 0, 0): (607, 512, 10272), (0, 2, 4, 1, 0): (215, 2240, 22581),
    (0, 2, 4, 1, 1): (171, 13824, 2720), (1, 1, 1, 0, 0): (60, 256, 16), (1, 1, 1, 0, 1): (3, 8192, 120),
    (1, 1, 1, 1, 0): (5, 320, 49), (1, 1, 1, 1, 1): (4, 3008, 53), (1, 1, 2, 0, 0): (87, 256, 11088),
    (1, 1, 2, 0, 1): (193, 4096, 516), (1, 1, 2, 1, 0): (198, 64, 6877), (1, 1, 2, 1, 1): (783, 14848, 19),
    (1, 1, 3, 0, 0): (79, 256, 21804), (1, 1, 3, 0, 1): (73, 6144, 2092), (1, 1, 4, 0, 0): (193, 256, 13652),
    (1, 1, 4, 0, 1): (193, 2048, 3468), (1, 1, 4, 1, 0): (992, 64, 2793), (1, 1, 4, 1, 1): (1299, 12032, 27),
    (1, 1, 5, 0, 0): (259, 256, 14024), (1, 1, 5, 0, 1): (134, 4096, 2928), (1, 1, 5, 1, 0): (536, 64, 14337),
    (1, 1, 5, 1, 1): (1089, 11264, 209), (1, 2, 3, 0, 0): (169, 256, 26004), (1, 2, 3, 0, 1): (89, 7168, 9360),
    (1, 2, 4, 0, 0): (682, 256, 8724), (1, 2, 4, 1, 0): (1122, 384, 28875), (1, 2, 4, 1, 1): (127, 16128, 9520),
    (1, 2, 5, 0, 0): (266, 256, 27764), (1, 2, 5, 0, 1): (157, 11264, 8932), (2, 1, 1, 0, 0): (36, 512, 20),
    (2, 1, 2, 0, 0): (229, 512, 2120), (2, 1, 3, 0, 0): (285, 512, 3412), (2, 1, 4, 0, 0): (122, 512, 11572),
    (2, 1, 5, 0, 0): (142, 1024, 11692), (2, 2, 3, 0, 0): (677, 512, 3756), (2, 2, 4, 0, 0): (249, 512, 12312),
    (3, 1, 1, 0, 0): (69, 512, 6144), (3, 1, 2, 0, 0): (185, 512, 6144), (3, 1, 3, 0, 0): (369, 512, 6144),
    (3, 1, 4, 0, 0): (523, 512, 6144), (3, 1, 5, 0, 0): (690, 512, 6144), (3, 2, 3, 0, 0): (855, 512, 6144),
    (3, 2, 4, 0, 0): (1025, 512, 6144),
}


# Calls that stay in the LDS tiles: (0 INT4, 1 e4m3; rows, columns of the tile, K split, a K that leaves a rest):
# (M, K, N).
TILES_IN_LDS = {
    (0, 64, 64, 1, 0): (12, 1024, 12413), (0, 64, 64, 1, 1): (17, 128, 189), (0, 64, 64, 2, 1): (29, 896, 56),
    (0, 64, 64, 4, 1): (14, 1792, 144), (0, 64, 128, 1, 0): (35, 5632, 32655),
    (0, 64, 128, 1, 1): (40, 64, 32670), (0, 128, 64, 1, 0): (70, 5888, 32475),
    (0, 128, 64, 1, 1): (245, 64, 7572), (0, 128, 64, 2, 1): (80, 3968, 6080),
    (0, 128, 64, 4, 1): (111, 2816, 2312), (0, 128, 128, 1, 0): (170, 256, 28828),
    (0, 128, 128, 1, 1): (323, 64, 23748), (1, 64, 64, 1, 0): (25, 1280, 15601),
    (1, 64, 64, 1, 1): (32, 832, 6499), (1, 64, 64, 2, 0): (52, 4096, 15828),
    (1, 64, 64, 2, 1): (49, 1152, 3148), (1, 64, 64, 4, 0): (9, 1024, 132), (1, 64, 64, 4, 1): (5, 1280, 3004),
    (1, 64, 64, 8, 0): (21, 2048, 48), (1, 64, 64, 8, 1): (64, 2560, 108), (1, 64, 128, 1, 0): (5, 9472, 32714),
    (1, 64, 128, 1, 1): (11, 12352, 32678), (1, 128, 64, 1, 0): (68, 11776, 29573),
    (1, 128, 64, 1, 1): (75, 6592, 32556), (1, 128, 64, 2, 1): (454, 2304, 1600),
    (1, 128, 64, 4, 1): (111, 3328, 3912), (1, 128, 64, 8, 1): (197, 9216, 1004),
    (1, 128, 128, 1, 1): (433, 64, 22552),
}


@pytest.mark.parametrize("m,k,n", SHAPES + ANY + [c for i, c in [*INSTANCES.items(), *TILES_IN_LDS.items()] if i[0] == 0])
def test_int4_matches_float32(dev, m, k, n):
    from moss_tts._runtime import w4g32

    print(f"wide int4 M={m} K={k} N={n}", flush=True)
    pw, g = _packed(n, k, m + k + n, dev)
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    _close(w4g32.gemm(x, pw), x.float() @ w4g32.dequantize(pw).float().T)


@pytest.mark.parametrize("m,k,n", [(2, 256, 132)] + SHAPES[1:] + ANY
                         + [c for i, c in [*INSTANCES.items(), *TILES_IN_LDS.items()] if i[0] == 1])
def test_fp8_matches_float32(dev, m, k, n):
    from moss_tts._runtime import fp8

    print(f"wide fp8 M={m} K={k} N={n}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + k + n)
    w = torch.randn((n, k), device=dev, generator=g)
    s = w.abs().amax(1) / 448.0
    codes = (w / s[:, None]).to(torch.float8_e4m3fn)
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    _close(fp8.linear(x, codes, s), x.float() @ (codes.float() * s[:, None]).T)


@pytest.mark.parametrize("m,k,n", [(m, 4096, n) for m, n in ((5, 2048), (24, 12288), (33, 1028), (64, 12288), (96, 12288),
                                                             (150, 12288), (437, 12288))]
                         + [c for i, c in INSTANCES.items() if i[0] == 2])
def test_silu_equals_gemm_then_silu(dev, m, k, n):
    from moss_tts._runtime import pointwise, w4g32

    print(f"wide silu M={m} K={k} N={n}", flush=True)
    pw, g = _packed(2 * n, k, m + n, dev)
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    want = pointwise.silu_mul(w4g32.gemm(x, pw))
    assert torch.equal(w4g32.gemm_silu(x, pw).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,k", [(m, 4096) for m in (270, 437, 1500)] + [c[:2] for i, c in INSTANCES.items() if i[0] == 3])
def test_qk_rope_equals_gemm_then_qk_rope(dev, m, k):
    from moss_tts._runtime import pointwise, w4g32

    print(f"wide qk rope M={m} K={k}", flush=True)
    L = 2048
    w, g = _packed(6144, k, m, dev)
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    qn, kn = ((1 + 0.1 * torch.randn(128, device=dev, generator=g)).bfloat16() for _ in range(2))
    cos, sin = (torch.randn((L, 128), device=dev, generator=g).bfloat16() for _ in range(2))
    pos = torch.randperm(L, device=dev, generator=g)[:m].to(torch.int64)
    kv = [torch.randn((1, 8, L, 128), device=dev, generator=g).bfloat16() for _ in range(2)]
    k1, v1, k2, v2 = (t.clone() for t in kv + kv)
    q1 = w4g32.gemm_qk_rope(x, w, qn, kn, cos, sin, k1, v1, pos, 1e-6)
    q2 = pointwise.qk_rope(w4g32.gemm(x, w), qn, kn, cos, sin, k2, v2, pos, 1e-6, cos_by_position=True)
    for a, b in ((q1.contiguous(), q2.contiguous()), (k1, k2), (v1, v2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("m", [5, 40, 130])
def test_weight_past_2_gib(dev, m):
    """Rows at both ends of a weight whose codes pass 2 GiB, against the same rows as weights of their own: one
    sum order, so bit for bit (32772 rows fill the card as the whole does, so neither splits K)."""
    from moss_tts._runtime import w4g32

    k, n = 1024, 2 ** 22 + 132
    print(f"wide large weight M={m}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m)
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), device=dev, generator=g, dtype=torch.int32)
    scales = (0.01 + 0.01 * torch.rand((n, k // 32), device=dev, generator=g)).bfloat16()
    zeros = torch.randint(0, 256, (n, k // 64), device=dev, generator=g, dtype=torch.uint8)
    assert qw.numel() * 4 > 2 ** 31
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    y = w4g32.gemm(x, w4g32.PackedW4G32(qw, scales, zeros))
    for lo in (0, n - 32772):
        part = w4g32.PackedW4G32(qw[lo:lo + 32772], scales[lo:lo + 32772], zeros[lo:lo + 32772])
        assert torch.equal(y[:, lo:lo + 32772], w4g32.gemm(x, part))
