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


@pytest.mark.parametrize("symmetric", [None, "", "yes", 2])
def test_symmetric_is_a_truth_value(monkeypatch, symmetric):
    """The C entry takes an int; any truth value chooses the quantizer, as it always has."""
    sent = []
    monkeypatch.setattr(w4g32, "_cuda_contig", lambda *a: None)
    monkeypatch.setattr(w4g32.PackedW4G32, "empty", lambda *a: _Packed())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: type("Stream", (), {"cuda_stream": 0}))
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    monkeypatch.setattr(w4g32.native, "call", lambda name, *args: sent.append(args[-2]))
    w4g32.quantize_launch(torch.zeros(8, 64), symmetric)
    assert sent == [int(bool(symmetric))]
