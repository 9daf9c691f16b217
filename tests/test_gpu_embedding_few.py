"""The embedding sum on both sides of its few-token form: token by token equal to the sum of all tokens
at once, bit for bit (the rounded additions of a value have one order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,h", [(1, 4096), (4, 4096), (5, 4096), (3, 264), (40, 1028)])
def test_few_tokens_equal_many(dev, tokens, h):
    from moss_tts._runtime import attention

    g = torch.Generator(device=dev).manual_seed(tokens + h)
    text = torch.randn((50, h), device=dev, generator=g).bfloat16()
    audio = torch.randn((32, 30, h), device=dev, generator=g).bfloat16()
    ids = torch.randint(0, 30, (tokens, 33), device=dev, generator=g)
    want = text[ids[:, 0]]
    for b in range(32):
        want = (want.float() + audio[b][ids[:, 1 + b]].float()).bfloat16()
    assert torch.equal(attention.embedding_sum(ids, text, audio).view(tokens, h), want)
    many = ids.repeat(-(-20 * 4096 // (tokens * h)), 1)
    assert torch.equal(attention.embedding_sum(many, text, audio).view(-1, h)[-tokens:], want)
