"""The work a program has this framework do, as cases that can be timed and compared.

Every case goes through the public entry points: the decode step and the prompt pass of
``DecodeStepG32``, the operators of one layer of the prompt pass, the quantized projection modules,
the FP8 linear, and the weight quantizer.  Weights, activations, caches and embeddings are synthetic
with the Qwen3-8B shapes of the MOSS-TTS backbone (hidden 4096, 32 query / 8 KV heads of 128, MLP
12288, q||k||v 6144) and made from the seed alone.
"""
from __future__ import annotations

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "moss-tts-optimized_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from moss_tts._runtime import attention, fp8, w4g32  # noqa: E402
from moss_tts._runtime.decode import DecodeStepG32, DecoderLayerG32, rope_tables  # noqa: E402
from moss_tts._runtime.modules import Bf16Linear, QuantGateUpG32, QuantLinearG32  # noqa: E402
from moss_tts._runtime.w4g32 import PackedW4G32  # noqa: E402

HIDDEN, INTER, QH, KH, HD, QKV = 4096, 12288, 32, 8, 128, 6144
BOOKS, CODES, TEXT_VOCAB = 32, 1024, 151936
EPS, THETA = 1e-6, 1e6
PROJECTIONS = ((HIDDEN, QKV, False), (HIDDEN, HIDDEN, False), (HIDDEN, 2 * INTER, True), (INTER, HIDDEN, False))


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one audio frame of a running request, bf16 activations: the serving loop's unit of work
        # (4 of the 36 layers, 446 MB of packed weights, and the 32 audio heads in bf16)
        dict(name="decode_frame", kind="decode", layers=4, length=2048, position=1500, w4a8=False, text=False),
        # the same with the reference's int8 serving arithmetic, earlier in the request
        dict(name="decode_frame_w4a8", kind="decode", layers=4, length=1024, position=700, w4a8=True, text=False),
        # a voice-cloning prompt: replays the 512-token bucket, text logits and audio logits
        dict(name="prompt_437", kind="prompt", layers=3, tokens=437, start=0, length=1024),
        # one layer of a prompt beyond the buckets, the longest: runs eagerly
        dict(name="layer_2048", kind="layer", tokens=2048, start=0, length=2048),
        # one layer of a short prompt that continues a cached prefix
        dict(name="layer_150_after_600", kind="layer", tokens=150, start=600, length=1024),
        # the swapped output projection on one token: the smallest call, launch and host latency
        dict(name="linear_o_1", kind="linear", rows=1, k=HIDDEN, n=HIDDEN, paired=False),
        # the swapped gate||up module on a handful of tokens
        dict(name="linear_gateup_24", kind="linear", rows=24, k=HIDDEN, n=2 * INTER, paired=True),
        # the swapped down projection on a medium prompt of odd length
        dict(name="linear_down_301", kind="linear", rows=301, k=INTER, n=HIDDEN, paired=False),
        # FP8 weight-only linears: the fused gate||up of one token
        dict(name="fp8_gateup_1", kind="fp8", rows=1, k=HIDDEN, n=2 * INTER, paired=True, scaled=True),
        # a small batch
        dict(name="fp8_64", kind="fp8", rows=64, k=HIDDEN, n=INTER, paired=False, scaled=True),
        # a long prompt of odd length
        dict(name="fp8_777", kind="fp8", rows=777, k=HIDDEN, n=INTER, paired=False, scaled=True),
        # loading: a float projection quantized on the device (QuantLinearG32.from_float)
        dict(name="quantize_mlp", kind="quantize", k=HIDDEN, n=INTER, symmetric=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "prompt", "layer", "linear", "linear", "linear", "fp8", "fp8", "quantize"))
    if kind == "decode":
        length = rng.choice((512, 1024, 2048, 4096))
        return dict(kind=kind, layers=4, length=length, position=rng.randrange(length), w4a8=rng.random() < 0.5,
                    text=rng.random() < 0.25)
    if kind == "prompt":
        length = rng.choice((1024, 2048))
        return dict(kind=kind, layers=3, tokens=rng.randint(2, 512), length=length,
                    start=0 if rng.random() < 0.6 else rng.randint(1, length - 512))
    if kind == "layer":
        tokens = _log_int(rng, 33, 1800)
        start = 0 if rng.random() < 0.6 else _log_int(rng, 16, 1800)
        return dict(kind=kind, tokens=tokens, start=start, length=-(-(start + tokens) // 128) * 128)
    if kind == "linear":
        rows = _log_int(rng, 1, 1024)
        if rng.random() < 0.7:
            k, n, paired = rng.choice(PROJECTIONS)
        else:
            k, n, paired = 64 * _log_int(rng, 4, 192), _log_int(rng, 64, 16384), False
        return dict(kind=kind, rows=rows, k=k, n=n, paired=paired)
    if kind == "fp8":
        rows = _log_int(rng, 1, 1024)
        if rng.random() < 0.7:
            k, n = rng.choice(((HIDDEN, HIDDEN), (HIDDEN, INTER), (INTER, HIDDEN), (HIDDEN, 2 * INTER)))
        else:
            k, n = 64 * _log_int(rng, 4, 192), 2 * _log_int(rng, 32, 8192)
        return dict(kind=kind, rows=rows, k=k, n=n, paired=rows == 1 and rng.random() < 0.5, scaled=rng.random() < 0.8)
    k, n = 64 * _log_int(rng, 16, 192), _log_int(rng, 256, 4096)
    return dict(kind="quantize", k=k, n=n, symmetric=rng.random() < 0.5)


# ------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape, scale=1.0):
    return torch.randn(shape, generator=gen, device="cuda").mul_(scale)


def _norm(gen, n):
    return (1 + 0.01 * _randn(gen, n)).bfloat16()


def _weight(gen, n, k):
    """N(0, 0.02) quantized min-max per (row, 32 inputs): codes uint8 [N, K], zeros uint8 [N, K/32],
    scales bf16 [N, K/32]."""
    w = _randn(gen, n, k, scale=0.02).view(n, k // 32, 32)
    lo, hi = w.amin(-1), w.amax(-1)
    s = ((hi - lo) / 15.0).clamp_min(1e-8).bfloat16()
    z = torch.round(-lo / s.float()).clamp_(0, 15)
    q = torch.round(w / s.float()[..., None]).add_(z[..., None]).clamp_(0, 15)
    return q.view(n, k).to(torch.uint8), z.to(torch.uint8), s


def _pack(weight):
    """The row-packed layout of include/moss_hip.h."""
    q, z, s = weight
    n, k = q.shape
    t = q.view(n, k // 8, 8).to(torch.int32)
    word = torch.zeros((n, k // 8), dtype=torch.int32, device=q.device)
    for i in range(4):
        word |= t[..., 2 * i] << (4 * i)
        word |= t[..., 2 * i + 1] << (16 + 4 * i)
    groups = k // 32
    zp = torch.empty((n, groups // 2), dtype=torch.uint8, device=q.device)
    for c in range(0, groups, 128):
        r = min(128, groups - c)
        zp[:, c // 2: c // 2 + r // 2] = z[:, c: c + r // 2] | (z[:, c + r // 2: c + r] << 4)
    return PackedW4G32(word, s.contiguous(), zp)


def _dequant(weight):
    """float64 [N, K] of the bf16 weights bf16((q - z) s) that the packed codes stand for."""
    q, z, s = weight
    n, k = q.shape
    d = (q.view(n, k // 32, 32).float() - z.float()[..., None]) * s.float()[..., None]
    return d.bfloat16().double().view(n, k)


def _layer_weights(gen):
    return dict(qkv=_weight(gen, QKV, HIDDEN), o=_weight(gen, HIDDEN, HIDDEN), gate_up=_weight(gen, 2 * INTER, HIDDEN),
                down=_weight(gen, HIDDEN, INTER), input_norm=_norm(gen, HIDDEN), post_norm=_norm(gen, HIDDEN),
                q_norm=_norm(gen, HD), k_norm=_norm(gen, HD))


def _token_ids(gen, n):
    return torch.cat([torch.randint(0, TEXT_VOCAB, (n, 1), generator=gen, device="cuda"),
                      torch.randint(0, CODES + 1, (n, BOOKS), generator=gen, device="cuda")], 1)


def _model_inputs(case, gen):
    """The parts of a model that are not projections, the caches it starts from, and the token ids."""
    text_head = case["kind"] == "prompt" or case["text"]
    shape = (1, KH, case["length"], HD)
    return dict(final_norm=_norm(gen, HIDDEN),
                heads=_randn(gen, BOOKS * CODES + 2, HIDDEN, scale=0.02).bfloat16(),
                text_head=_randn(gen, TEXT_VOCAB, HIDDEN, scale=0.02).bfloat16() if text_head else None,
                text=_randn(gen, TEXT_VOCAB, HIDDEN, scale=0.2).bfloat16(),
                audio=_randn(gen, BOOKS, CODES + 1, HIDDEN, scale=0.2).bfloat16(),
                keys=[_randn(gen, *shape).bfloat16() for _ in range(case["layers"])],
                values=[_randn(gen, *shape).bfloat16() for _ in range(case["layers"])],
                ids=_token_ids(gen, case["tokens"] if case["kind"] == "prompt" else 1))


def _layer_inputs(case, gen):
    shape = (1, KH, case["length"], HD)
    n = case["tokens"]
    return dict(residual=_randn(gen, n, HIDDEN).bfloat16(), state=_randn(gen, n, HIDDEN).bfloat16(),
                next_norm=_norm(gen, HIDDEN), keys=_randn(gen, *shape).bfloat16(),
                values=_randn(gen, *shape).bfloat16())


def _fp8_inputs(case, gen):
    """e4m3 weights with the per-row scale that maps the row's largest magnitude onto 448."""
    w = _randn(gen, case["n"], case["k"], scale=0.02)
    scale = w.abs().amax(1) / 448.0 if case["scaled"] else None
    codes = (w / scale[:, None] if case["scaled"] else w).to(torch.float8_e4m3fn)
    return codes, scale, _randn(gen, case["rows"], case["k"]).bfloat16()


def _rope_tables(length):
    """The bf16 cos / sin tables that the path is given, as the model defines them."""
    inv = 1.0 / (THETA ** (torch.arange(0, HD, 2, dtype=torch.float32) / HD))
    emb = (torch.arange(length, dtype=torch.float32)[:, None] @ inv[None, :]).repeat(1, 2)
    return emb.cos().bfloat16().cuda(), emb.sin().bfloat16().cuda()


def _decoder_layer(w):
    return DecoderLayerG32(QuantLinearG32(_pack(w["qkv"])), QuantLinearG32(_pack(w["o"])),
                           QuantGateUpG32(_pack(w["gate_up"])), QuantLinearG32(_pack(w["down"])),
                           w["input_norm"], w["post_norm"], w["q_norm"], w["k_norm"])


@torch.inference_mode()
def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind in ("decode", "prompt"):
        layers = [_decoder_layer(_layer_weights(gen)) for _ in range(case["layers"])]
        m = _model_inputs(case, gen)
        text_head = Bf16Linear(m["text_head"]) if m["text_head"] is not None else None
        step = DecodeStepG32(layers, m["final_norm"], Bf16Linear(m["heads"]), m["text"], m["audio"],
                             max_length=case["length"], eps=EPS, theta=THETA, w4a8=case.get("w4a8", False),
                             audio_stride=CODES, text_head=text_head)
        if kind == "prompt":
            step.capture_prefill()
        elif case["text"]:
            step.capture_text()
        else:
            step.capture()
        for mine, given in zip(step.keys + step.values, m["keys"] + m["values"]):
            mine.copy_(given)  # after the captures, whose warm-up passes write cache rows
        return dict(case=case, step=step, ids=m["ids"])
    if kind == "layer":
        w, m = _layer_weights(gen), _layer_inputs(case, gen)
        cos, sin = rope_tables(case["length"], THETA, "cuda")
        packed = {name: _pack(w[name]) for name in ("qkv", "o", "gate_up", "down")}
        positions = torch.arange(case["start"], case["start"] + case["tokens"], device="cuda")
        return dict(case=case, w={**w, **packed}, cos=cos, sin=sin, positions=positions, start=positions[:1].clone(), **m)
    if kind == "linear":
        module = QuantGateUpG32 if case["paired"] else QuantLinearG32
        linear = module(_pack(_weight(gen, case["n"], case["k"])))
        return dict(case=case, linear=linear, x=_randn(gen, case["rows"], case["k"]).bfloat16())
    if kind == "fp8":
        codes, scale, x = _fp8_inputs(case, gen)
        return dict(case=case, codes=codes, scale=scale, x=x)
    return dict(case=case, w=_randn(gen, case["n"], case["k"], scale=0.02))


# ------------------------------------------------------------------------------------ one pass
@torch.inference_mode()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        step = state["step"]
        logits = (step.full_step if case["text"] else step.step)(state["ids"], case["position"])
        return dict(logits=logits, keys=step.keys, values=step.values)
    if kind == "prompt":
        step, rows = state["step"], slice(case["start"], case["start"] + case["tokens"])
        text, audio = step.prefill_logits(state["ids"], case["start"])
        # the prompt's cache rows; rows after it are padding that later steps overwrite
        return dict(text=text, audio=audio, keys=[k[:, :, rows] for k in step.keys],
                    values=[v[:, :, rows] for v in step.values])
    if kind == "layer":
        w = state["w"]
        q = w4g32.gemm_qk_rope(state["state"], w["qkv"], w["q_norm"], w["k_norm"], state["cos"], state["sin"],
                               state["keys"], state["values"], state["positions"], EPS)
        attn = attention.prefill_attention(q.transpose(1, 2), state["keys"], state["values"], state["start"])
        residual, hidden = w4g32.gemm_add_rmsnorm(attn, w["o"], state["residual"], w["post_norm"], EPS)
        act = w4g32.gemm_silu(hidden, w["gate_up"])
        residual, hidden = w4g32.gemm_add_rmsnorm(act, w["down"], residual, state["next_norm"], EPS)
        return dict(attn=attn, residual=residual, hidden=hidden, keys=state["keys"], values=state["values"])
    if kind == "linear":
        return state["linear"](state["x"])
    if kind == "fp8":
        if case["paired"]:
            return fp8.fp8_silu_decode(state["x"], state["codes"], state["scale"])
        return fp8.linear(state["x"], state["codes"], state["scale"])
    linear = QuantLinearG32.from_float(state["w"], symmetric=case["symmetric"])
    return dict(qw=linear.qw, scales=linear.scales, zeros=linear.zeros)


# ------------------------------------------------------------------------------------ floors
def _int4_bytes(n, k):
    return n * k // 2 + n * (k // 32) * 2 + n * (k // 64)


_LAYER_WEIGHTS = sum(_int4_bytes(n, k) for k, n, _ in PROJECTIONS)
_LAYER_MACS = sum(n * k for k, n, _ in PROJECTIONS)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        p, rows = case["position"] + 1, TEXT_VOCAB if case["text"] else BOOKS * CODES + 2
        kv = 2 * KH * p * HD * 2
        return dict(bytes=case["layers"] * (_LAYER_WEIGHTS + kv) + rows * HIDDEN * 2 + (BOOKS + 1) * HIDDEN * 2,
                    flops=2.0 * (case["layers"] * (_LAYER_MACS + 2 * QH * HD * p) + rows * HIDDEN))
    if kind in ("prompt", "layer"):
        n, s = case["tokens"], case["start"]
        pairs = n * s + n * (n + 1) // 2                  # (query, key) pairs of causal attention
        kv = 2 * KH * (s + n) * HD * 2
        layer = dict(bytes=_LAYER_WEIGHTS + kv + 2 * n * HIDDEN * 2, flops=2.0 * (_LAYER_MACS * n + 2 * QH * HD * pairs))
        if kind == "layer":
            return layer
        rows = TEXT_VOCAB + BOOKS * CODES + 2
        # after the last layer's K/V rows only the last token goes on
        last = 2.0 * (QKV * HIDDEN * n + (_LAYER_MACS - QKV * HIDDEN) + 2 * QH * HD * (s + n))
        return dict(bytes=case["layers"] * (_LAYER_WEIGHTS + kv) + rows * HIDDEN * 2 + n * (BOOKS + 1) * HIDDEN * 2,
                    flops=(case["layers"] - 1) * layer["flops"] + last + 2.0 * rows * HIDDEN)
    k, n = case["k"], case["n"]
    if kind == "quantize":
        return dict(bytes=4 * n * k + _int4_bytes(n, k), flops=0)
    rows = case["rows"]
    out = n // 2 if case["paired"] else n
    weights = _int4_bytes(n, k) if kind == "linear" else n * k + (4 * n if case["scaled"] else 0)
    return dict(bytes=weights + 2 * rows * (k + out), flops=2.0 * rows * k * n)


def tolerance(case):
    """About four times what the path shows against 64 bits: a bf16 output rounded once is 0.0017 off
    in norm, the SiLU product of two of them 0.0035, a layer's outputs 0.006; over the layers of a
    whole model the bf16 roundings add up to 0.02 in the logits, which two correct implementations
    share but for the values where a sum in another order rounds the other way."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind in ("decode", "prompt"):
        return dict(rel=0.03)
    if kind == "layer":
        return dict(rel=0.02)
    return dict(rel=0.014 if case["paired"] else 0.007)


# ------------------------------------------------------------------------------------ in 64 bits
def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _int8(x):
    """x with every group of 32 rounded to int8 codes of its own scale max|x| / 127."""
    g = x.view(*x.shape[:-1], -1, 32)
    s = (g.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-8)
    return (torch.round(g / s) * s).view(x.shape)


def _project(x, weight, w4a8):
    if not w4a8:
        return x @ _dequant(weight).T
    q, z, s = weight  # W4A8: the unrounded (q - z) s meets the int8 codes
    n, k = q.shape
    w = ((q.view(n, k // 32, 32).double() - z.double()[..., None]) * s.double()[..., None]).view(n, k)
    return _int8(x) @ w.T


def _rope(x, cos, sin):
    half = torch.cat([-x[..., HD // 2:], x[..., :HD // 2]], -1)
    return x * cos + half * sin


def _silu_mul(x):
    gate, up = x.chunk(2, -1)
    return gate * torch.sigmoid(gate) * up


def _block(w, residual, state, keys, values, start, cos, sin, w4a8=False):
    """One layer in float64 over the tokens at start ..; writes their K/V rows into keys / values and
    returns the attention, the residual stream after it and the MLP's output."""
    n = state.shape[0]
    heads = _project(state, w["qkv"], w4a8).view(n, QH + 2 * KH, HD)
    rows = slice(start, start + n)
    c, s = cos[rows, None].double(), sin[rows, None].double()
    q = _rope(_rms(heads[:, :QH], w["q_norm"]), c, s)
    keys[0, :, rows] = _rope(_rms(heads[:, QH:QH + KH], w["k_norm"]), c, s).transpose(0, 1)
    values[0, :, rows] = heads[:, QH + KH:].transpose(0, 1)
    at = torch.arange(start, start + n, device=state.device)
    hidden = torch.arange(start + n, device=state.device)[None, :] > at[:, None]
    attn = torch.empty((n, QH, HD), dtype=torch.float64, device=state.device)
    for h in range(QH):
        kv = h // (QH // KH)
        scores = (q[:, h] @ keys[0, kv, :start + n].T) / math.sqrt(HD)
        attn[:, h] = torch.softmax(scores.masked_fill(hidden, -math.inf), -1) @ values[0, kv, :start + n]
    attn = attn.view(n, HIDDEN)
    residual = residual + _project(attn, w["o"], w4a8)
    act = _silu_mul(_project(_rms(residual, w["post_norm"]), w["gate_up"], w4a8))
    return attn, residual, _project(act, w["down"], w4a8)


@torch.inference_mode()
def exact(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind in ("decode", "prompt"):
        layers = [_layer_weights(gen) for _ in range(case["layers"])]
        m = _model_inputs(case, gen)
        start, n = (case["position"], 1) if kind == "decode" else (case["start"], case["tokens"])
        cos, sin = _rope_tables(case["length"])
        keys, values = [k.double() for k in m["keys"]], [v.double() for v in m["values"]]
        residual = m["text"][m["ids"][:, 0]].double()
        for b in range(BOOKS):
            residual = residual + m["audio"][b][m["ids"][:, 1 + b]].double()
        for i, w in enumerate(layers):
            _, residual, mlp = _block(w, residual, _rms(residual, w["input_norm"]), keys[i], values[i], start, cos, sin,
                                      case.get("w4a8", False))
            residual = residual + mlp
        state = _rms(residual[-1:], m["final_norm"])
        if kind == "prompt":
            rows = slice(start, start + n)
            audio = (state @ m["heads"][:BOOKS * CODES].double().T).view(BOOKS, CODES)
            return dict(text=state @ m["text_head"].double().T, audio=audio, keys=[k[:, :, rows] for k in keys],
                        values=[v[:, :, rows] for v in values])
        logits = state @ (m["text_head"] if case["text"] else m["heads"]).double().T
        return dict(logits=logits if case["text"] else logits.view(-1), keys=keys, values=values)
    if kind == "layer":
        w, m = _layer_weights(gen), _layer_inputs(case, gen)
        cos, sin = _rope_tables(case["length"])
        keys, values = m["keys"].double(), m["values"].double()
        attn, residual, mlp = _block(w, m["residual"].double(), m["state"].double(), keys, values, case["start"], cos, sin)
        residual = residual + mlp
        return dict(attn=attn, residual=residual, hidden=_rms(residual, m["next_norm"]), keys=keys, values=values)
    if kind == "linear":
        weight = _weight(gen, case["n"], case["k"])
        y = _randn(gen, case["rows"], case["k"]).bfloat16().double() @ _dequant(weight).T
        return _silu_mul(y) if case["paired"] else y
    if kind == "fp8":
        codes, scale, x = _fp8_inputs(case, gen)
        y = x.double() @ codes.double().T
        y = y * scale.double() if case["scaled"] else y
        return _silu_mul(y) if case["paired"] else y
    w = _randn(gen, case["n"], case["k"], scale=0.02).view(case["n"], case["k"] // 32, 32).double()
    scales = w.abs().amax(-1) / 7 if case["symmetric"] else (w.amax(-1) - w.amin(-1)) / 15
    return dict(qw=None, scales=scales, zeros=None)
