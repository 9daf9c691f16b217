"""The range check of the quantizers' scales: one group's scale the last bf16 below 2^120 and 2^120 itself,
infinities of both signs, at the first and the last group of a weight, for both quantizers; a NaN is no
extreme of its group, so it is not refused and changes no other group."""
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
    largest = 2.0 ** 120 - 2.0 ** 112  # 8 significant bits; times the levels it is exact in float32
    base = torch.randn((n, k), device=dev)
    for value, fits in ((levels * largest, True), (levels * 2.0 ** 120, False), (float("inf"), False), (float("-inf"), False)):
        w = base.clone()
        w.view(-1, 32)[group] = 0
        w.view(-1, 32)[group, 7] = value
        if fits:
            assert quantize(w).scales.float().abs().max() == largest
        else:
            with pytest.raises(ValueError, match="2\\^120"):
                quantize(w)
    plain = quantize(base)
    assert plain.scales.isfinite().all()
    for lanes in (slice(7, 8), slice(0, 1), slice(0, 32)):
        w = base.clone()
        w.view(-1, 32)[group, lanes] = float("nan")
        scales = quantize(w).scales.view(-1)
        others = torch.arange(scales.numel(), device=dev) != group
        assert scales.isfinite().all() and torch.equal(scales[others], plain.scales.view(-1)[others])


@pytest.mark.parametrize("symmetric", [False, True])
def test_under_a_default_device(dev, symmetric):
    """A module made where a program has set the device for its new tensors."""
    from moss_tts._runtime.modules import QuantLinearG32

    w = torch.randn((8, 64), device=dev)
    with torch.device(dev):
        inside = QuantLinearG32.from_float(w, symmetric=symmetric)
    outside = QuantLinearG32.from_float(w, symmetric=symmetric)
    assert torch.equal(inside.qw, outside.qw) and torch.equal(inside.scales, outside.scales)
