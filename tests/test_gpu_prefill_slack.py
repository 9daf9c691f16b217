"""Prompt attention where the softmax's running reference has to move: scores that grow along the keys,
in one step far past the reference and in many steps just below its slack, against float32 attention.

Tolerance: P and the output are rounded to bf16 (2^-9 of a value each), P's roundings average out in
the weighted sum; 2^-7 of the output's magnitude plus 2^-8 of the largest |V| covers both."""
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
