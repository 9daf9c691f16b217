"""The range check of the quantizers' scales: one group just inside and just outside 2^120, infinities and
NaN, at the first and the last group of a weight, for both quantizers."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("n,k,group", [(1, 64, 0), (5, 4672, 0), (5, 4672, 5 * 146 - 1)])
def test_scale_range(dev, symmetric, n, k, group):
    from moss_tts._runtime import w4g32

    print(f"quantize range N={n} K={k} group={group} symmetric={symmetric}", flush=True)
    quantize = w4g32.quantize_symmetric if symmetric else w4g32.quantize_minmax
    levels = 7 if symmetric else 15
    base = torch.randn((n, k), device=dev)
    for value, fits in ((levels * 2.0 ** 119, True), (levels * 2.0 ** 120, False), (float("inf"), False)):
        w = base.clone()
        w.view(-1, 32)[group] = 0
        w.view(-1, 32)[group, 7] = value
        if fits:
            assert quantize(w).scales.float().abs().max() == 2.0 ** 119
        else:
            with pytest.raises(ValueError, match="2\\^120"):
                quantize(w)
    assert quantize(base).scales.isfinite().all()
