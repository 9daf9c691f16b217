"""Prompt attention where the softmax's running reference has to move: scores that grow along the keys, in
large steps and in many small ones, value by value against float32 attention; and its error in norm, which is
what a reference that lags the maximum shows.

Tolerance of the values: P and the output are rounded to bf16 (2^-9 of a value each), P's roundings average
out in the weighted sum; 2^-7 of the output's magnitude plus 2^-8 of the largest |V| covers both."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,start", [(33, 0), (512, 95), (513, 0), (600, 130), (1025, 0)])
@pytest.mark.parametrize("growth", [0.0, 0.05, 3.0])
def test_growing_scores(dev, n, start, growth):
    from moss_tts._runtime import attention

    print(f"prompt attention n={n} start={start} growth={growth}", flush=True)
    L = -(-(n + start) // 64) * 64
    g = torch.Generator(device=dev).manual_seed(n + start)
    q = torch.randn((n, 32, 128), device=dev, generator=g).bfloat16()
    k = torch.randn((1, 8, L, 128), device=dev, generator=g)
    k = (k * (1 + growth * torch.arange(L, device=dev)[:, None] / 64)).bfloat16()
    v = torch.randn((1, 8, L, 128), device=dev, generator=g).bfloat16()
    out = attention.prefill_attention(q, k, v, torch.full((1,), start, device=dev)).view(n, 32, 128).float()
    hidden = torch.arange(start + n, device=dev)[None, :] > torch.arange(start, start + n, device=dev)[:, None]
    for h in range(0, 32, 5):
        s = q[:, h].float() @ k[0, h // 4, :start + n].float().T / math.sqrt(128)
        ref = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[0, h // 4, :start + n].float()
        bound = ref.abs() * 2.0 ** -7 + v.float().abs().max() * 2.0 ** -8
        assert ((out[:, h] - ref).abs() <= bound).all(), f"head {h}"


@pytest.mark.parametrize("n,start", [(150, 600), (437, 0), (513, 1000), (1100, 0)])
@pytest.mark.parametrize("sharpness", [1.0, 4.0])
def test_error_of_one_rounding_of_p(dev, n, start, sharpness):
    """No more error than P rounded once to bf16 relative to its row's maximum gives, with the denominator of
    the rounded P and a bf16 output, all else in 64 bits: the kernel has further maxima (one per 32-key tile
    and wave) that are exact too, which lowers its error by 3 to 6%.  A reference up to 2^8 below the maximum
    gives 1.00 to 1.16 times the error of one rounding."""
    from moss_tts._runtime import attention

    print(f"prompt attention n={n} start={start} sharpness={sharpness}", flush=True)
    L = -(-(n + start) // 64) * 64
    g = torch.Generator(device=dev).manual_seed(n + start)
    q = (sharpness * torch.randn((n, 32, 128), device=dev, generator=g)).bfloat16()
    k, v = (torch.randn((1, 8, L, 128), device=dev, generator=g).bfloat16() for _ in range(2))
    out = attention.prefill_attention(q, k, v, torch.full((1,), start, device=dev)).view(n, 32, 128).double()
    hidden = torch.arange(start + n, device=dev)[None, :] > torch.arange(start, start + n, device=dev)[:, None]
    error = once = 0.0
    for h in range(32):
        kh, vh = (t[0, h // 4, :start + n].double() for t in (k, v))
        s = (q[:, h].double() @ kh.T / math.sqrt(128)).masked_fill(hidden, -math.inf)
        p = (s - s.amax(-1, keepdim=True)).exp()
        exact = p @ vh / p.sum(-1, keepdim=True)
        p = p.bfloat16().double()
        rounded = (p @ vh / p.sum(-1, keepdim=True)).bfloat16().double()
        error += float((out[:, h] - exact).square().sum())
        once += float((rounded - exact).square().sum())
    print(f"error {math.sqrt(error / once):.4f} of one rounding's", flush=True)
    assert error <= once
