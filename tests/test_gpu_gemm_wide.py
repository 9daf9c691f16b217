"""The wide GEMM tile against the float32 product of the dequantized weights: every tile of it (32 to
160 tokens, 128 and 256 weight rows), one token short of and past a tile, rows past the last tile, K of
one block and K splits, and its SiLU and q/k-norm epilogues at sizes that pick different tiles.

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


@pytest.mark.parametrize("m,k,n", SHAPES + ANY)
def test_int4_matches_float32(dev, m, k, n):
    from moss_tts._runtime import w4g32

    print(f"wide int4 M={m} K={k} N={n}", flush=True)
    pw, g = _packed(n, k, m + k + n, dev)
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    _close(w4g32.gemm(x, pw), x.float() @ w4g32.dequantize(pw).float().T)


@pytest.mark.parametrize("m,k,n", [(2, 256, 132)] + SHAPES[1:] + ANY)
def test_fp8_matches_float32(dev, m, k, n):
    from moss_tts._runtime import fp8

    print(f"wide fp8 M={m} K={k} N={n}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + k + n)
    w = torch.randn((n, k), device=dev, generator=g)
    s = w.abs().amax(1) / 448.0
    codes = (w / s[:, None]).to(torch.float8_e4m3fn)
    x = torch.randn((m, k), device=dev, generator=g).bfloat16()
    _close(fp8.linear(x, codes, s), x.float() @ (codes.float() * s[:, None]).T)


@pytest.mark.parametrize("m,n", [(5, 2048), (24, 12288), (33, 1028), (64, 12288), (96, 12288), (150, 12288), (437, 12288)])
def test_silu_equals_gemm_then_silu(dev, m, n):
    from moss_tts._runtime import pointwise, w4g32

    print(f"wide silu M={m} N={n}", flush=True)
    pw, g = _packed(2 * n, 4096, m + n, dev)
    x = torch.randn((m, 4096), device=dev, generator=g).bfloat16()
    want = pointwise.silu_mul(w4g32.gemm(x, pw))
    assert torch.equal(w4g32.gemm_silu(x, pw).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m", [270, 437, 1500])
def test_qk_rope_equals_gemm_then_qk_rope(dev, m):
    from moss_tts._runtime import pointwise, w4g32

    print(f"wide qk rope M={m}", flush=True)
    L = 2048
    w, g = _packed(6144, 4096, m, dev)
    x = torch.randn((m, 4096), device=dev, generator=g).bfloat16()
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
