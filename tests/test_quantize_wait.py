"""``QuantLinearG32.from_float`` waits for the quantizer on every path: its kernel writes a flag in pinned host
memory that nothing else keeps alive, so that memory may not be given back while the kernel can still run."""
import pytest
import torch

from moss_tts._runtime import modules, w4g32


class _DeviceWeight:
    is_cuda, ndim = True, 2

    def detach(self):
        return self

    float = contiguous = detach


class _Packed:
    K, N = 64, 8
    qw = scales = zeros = torch.zeros(1)


@pytest.mark.parametrize("kw", [{}, {"no_such_option": 1}])
def test_from_float_waits(monkeypatch, kw):
    waits = []
    monkeypatch.setattr(w4g32, "quantize_launch", lambda w, symmetric: (_Packed(), lambda: waits.append(1)))
    if kw:
        with pytest.raises(TypeError):
            modules.QuantLinearG32.from_float(_DeviceWeight(), **kw)
    else:
        assert modules.QuantLinearG32.from_float(_DeviceWeight()).in_features == 64
    assert waits == [1]
