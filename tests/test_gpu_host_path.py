"""The native launch path (csrc/host.cpp) against the Python path it stands in for:
the same bits over layouts, strides, routing modes, block sizes and V formats, None for
the calls it does not serve (which the Python path then takes), the environment
switches, streams and graph capture."""
from __future__ import annotations

import types

import numpy as np
import pytest
import torch

from _helpers import packed_inputs, random_bitmask, to_dev
from tilemix_amd import _native
from tilemix_amd.attention.hip import tilemix as tmx
from tilemix_amd.attention.tilemix_varlen import tilemix_varlen_attention
from tilemix_amd.models import tilemix_llama as TL

pytestmark = pytest.mark.gpu

_NONE = types.SimpleNamespace(**{name: (lambda *a: None) for name in ("packed", "dense", "quantize", "rms_norm",
                                                                      "rotary", "silu_mul")})


class _Spy:
    """The real module; whether it served the entry point's own call (a dense call that it does not
    serve may come back as a packed one, after the Python path's copies)."""

    def __init__(self):
        self.served = None

    def __getattr__(self, name):
        def call(*a):
            out = getattr(_native.__dict__["_real_host"], name)(*a)
            if self.served is None:
                self.served = out is not None
            return out
        return call


@pytest.fixture
def both(monkeypatch):
    """both(fn, served=True): fn() through the native path and through the Python path, bitwise
    equal; checks whether the native path served the call."""
    monkeypatch.setattr(_native, "_real_host", _native.host(), raising=False)

    def run(fn, served=True):
        spy = _Spy()
        monkeypatch.setattr(_native, "host", lambda: spy)
        got = fn()
        assert spy.served in ((True,) if served else (False, None))
        monkeypatch.setattr(_native, "host", lambda: _NONE)
        want = fn()
        torch.cuda.synchronize()
        for a, b in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
            assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
            assert torch.equal(*(x.contiguous().view(torch.int16) if x.dtype == torch.float16 else x
                                 for x in (a, b)))
        return got

    return run


def _bitmask(hk, length, block_m, device, seed=1):
    return torch.from_numpy(random_bitmask(hk, -(-length // block_m), seed=seed)).to(device)


@pytest.mark.parametrize("mode", ["mixed", "fp16", "int8"])
@pytest.mark.parametrize("block_m", [64, 128, 256])
@pytest.mark.parametrize("fp16_v", [True, False])
@pytest.mark.parametrize("d", [64, 128])
def test_packed(device, both, mode, block_m, fp16_v, d):
    lengths = [130, 0, 1, 257]
    q, k, v, cu = packed_inputs(lengths, 4, 2, d, seed=3)
    dq, dk, dv, dcu = (to_dev(x, device) for x in (q, k, v, cu))
    bits = _bitmask(2, 257, block_m, device)
    both(lambda: tmx.tilemix_attention_with_quant(
        dq, dk, dv, dcu, dcu, 257, 257, bits, block_m=block_m, block_n=64, BLKQ=128, BLKK=64, causal=True,
        scalar_scales=block_m == 128, routing_mode=mode, int8_use_fp16_v=fp16_v)[0])


@pytest.mark.parametrize("form", ["head_major", "fused_qkv", "one_head_expanded", "one_token"])
@pytest.mark.parametrize("block_m", [64, 128])
def test_packed_layouts(device, both, form, block_m):
    """The output of a packed call has q's strides where q is dense (head-major q: head-major output)."""
    g = torch.Generator(device=device).manual_seed(block_m)
    n, hq, hk, d = 1 if form == "one_token" else 300, 4, 2, 64
    q, k, v = (torch.randn(n, h, d, generator=g, device=device).half() for h in (hq, hk, hk))
    if form in ("head_major", "one_token"):
        q, k, v = (t.transpose(0, 1).contiguous().transpose(0, 1) for t in (q, k, v))
    elif form == "fused_qkv":
        q, k, v = torch.cat((q, k, v), dim=1).split([hq, hk, hk], dim=1)
    else:
        q = q[:, :1].expand(-1, hq, -1)
    cu = torch.tensor([0, 1, n] if n > 1 else [0, n], dtype=torch.int32, device=device)
    bits = _bitmask(hk, n, block_m, device)
    out = both(lambda: tmx.tilemix_attention_with_quant(
        q, k, v, cu, cu, n, n, bits, block_m=block_m, block_n=64, BLKQ=128, BLKK=64, causal=True,
        scalar_scales=False, routing_mode="mixed", int8_use_fp16_v=True)[0])
    assert out.stride() == torch.empty_like(q).stride()


@pytest.mark.parametrize("form", ["token_major", "head_major_1", "fused_qkv", "wide_heads"])
@pytest.mark.parametrize("d,length", [(64, 256), (128, 193), (80, 64), (112, 1)])
def test_dense_layouts(device, both, form, d, length):
    """Layouts read where they lie: projections viewed [B, H, T, D], one sequence in head-major
    order, slices of one QKV buffer, heads padded to a wider stride."""
    b, hq, hk = (1 if form == "head_major_1" else 3), 6, 2
    g = torch.Generator(device=device).manual_seed(d + length)
    if form == "fused_qkv":
        x = torch.randn(b, length, (hq + 2 * hk) * d, generator=g, device=device).half()
        parts = x.split([hq * d, hk * d, hk * d], dim=-1)
        q, k, v = (p.view(b, length, -1, d).transpose(1, 2) for p in parts)
    elif form == "head_major_1":
        q, k, v = (torch.randn(b, h, length, d, generator=g, device=device).half() for h in (hq, hk, hk))
    else:
        width = d + 8 if form == "wide_heads" else d
        q, k, v = (torch.randn(b, length, h, width, generator=g, device=device).half()[..., :d].transpose(1, 2)
                   for h in (hq, hk, hk))
    bits = _bitmask(hk, length, 64, device)
    out = both(lambda: tilemix_varlen_attention(q, k, v, 64, 64, causal=True, scale=d ** -0.5, precision_map_all=bits,
                                                candidates=[(64, 64)], flat_lengths=[bits.numel()]))
    assert out.shape == (b, hq, length, d)


@pytest.mark.parametrize("form", ["expanded", "overlapping", "one_token"])
@pytest.mark.parametrize("operand", [0, 1, 2])
def test_tokens_closer_than_their_rows(device, form, operand):
    """One sequence whose tokens repeat, overlap, or (one token) have a stride that says nothing: the result of
    the dense tensors, through both entry points."""
    g = torch.Generator(device=device).manual_seed(operand)
    n, h, d = 1 if form == "one_token" else 150, 2, 64
    x = [torch.randn(1, n, h, d, generator=g, device=device).half().transpose(1, 2) for _ in range(3)]
    if form == "expanded":
        x[operand] = x[operand][:, :, :1].expand(-1, -1, n, -1)
    elif form == "overlapping":
        base = torch.randn(h, 8 * n + d, generator=g, device=device).half()
        x[operand] = base.as_strided((1, h, n, d), (0, 8 * n + d, 8, 1))
    else:
        x[operand] = x[operand].as_strided((1, h, 1, d), (0, d, 0, 1))
    dense = [t.clone(memory_format=torch.contiguous_format) for t in x]
    bits = _bitmask(h, n, 64, device)
    cu = torch.tensor([0, n], dtype=torch.int32, device=device)

    def call(q, k, v):
        return tilemix_varlen_attention(q, k, v, 64, 64, causal=True, scale=0.125, precision_map_all=bits,
                                        candidates=[], flat_lengths=[])

    def packed(*qkv):
        return tmx.tilemix_attention_with_quant(
            *(t[0].transpose(0, 1) for t in qkv), cu, cu, n, n, bits, block_m=64, block_n=64, causal=True,
            scalar_scales=False, routing_mode="mixed", int8_use_fp16_v=True)[0]

    assert torch.equal(call(*x), call(*dense))
    assert torch.equal(packed(*x), packed(*dense))


@pytest.mark.parametrize("form", ["head_major", "misaligned", "head_dim_72", "map_on_cpu", "int64_cu", "bias", "forced"])
def test_not_served(device, both, form, monkeypatch):
    """Calls that need a copy, a conversion, padding or a switch go through the Python path."""
    b, hq, hk, t = 2, 4, 2, 128
    d = 72 if form == "head_dim_72" else 64
    g = torch.Generator(device=device).manual_seed(5)
    q, k, v = (torch.randn(b, t, h, d, generator=g, device=device).half().transpose(1, 2) for h in (hq, hk, hk))
    bits, bias = _bitmask(hk, t, 64, device), None
    if form == "head_major":
        q = q.contiguous()
    elif form == "misaligned":
        q = torch.randn(b, t, hq, d + 4, generator=g, device=device).half()[..., 4:].transpose(1, 2)
    elif form == "map_on_cpu":
        bits = bits.cpu()
    elif form == "bias":
        bias = torch.randn(b, hq, t, t, generator=g, device=device).half()
    elif form == "forced":
        monkeypatch.setenv("TILEMIX_FORCE_CONFIG", "64,64")
    if form == "int64_cu":
        cu = torch.arange(0, (b + 1) * t, t, device=device, dtype=torch.int64)
        both(lambda: tmx.tilemix_attention_with_quant(
            *(x.transpose(1, 2).reshape(b * t, -1, d) for x in (q, k, v)), cu, cu, t, t, bits, block_m=64, block_n=64,
            causal=True, scalar_scales=False, routing_mode="mixed", int8_use_fp16_v=True)[0], served=False)
        return
    both(lambda: tilemix_varlen_attention(q, k, v, 64, 64, causal=True, scale=d ** -0.5, precision_map_all=bits,
                                          bias=bias, candidates=[], flat_lengths=[]), served=False)


@pytest.mark.parametrize("name,value,served", [("TILEMIX_BITMASK_ROUTING_MODE", "int8", True),
                                               ("TILEMIX_BITMASK_ROUTING_MODE", " FP16", False),
                                               ("TILEMIX_SCORE_ONLY_PV", "0", True),
                                               ("TILEMIX_SCORE_ONLY_PV", "no", False),
                                               ("TILEMIX_SCORE_ONLY_PV", "", True),
                                               ("TILEMIX_BITMASK_ROUTING_MODE", "", True),
                                               ("TILEMIX_FORCE_CONFIG", "", True),
                                               ("TILEMIX_HIP_FUSED_Q_QUANT", "", False),
                                               ("TILEMIX_HIP_FUSED_Q_QUANT", "0", False)])
def test_environment(device, both, monkeypatch, name, value, served):
    g = torch.Generator(device=device).manual_seed(6)
    q, k, v = (torch.randn(2, 96, h, 64, generator=g, device=device).half().transpose(1, 2) for h in (4, 2, 2))
    bits = _bitmask(2, 96, 64, device)
    monkeypatch.setenv(name, value)
    both(lambda: tilemix_varlen_attention(q, k, v, 64, 64, causal=True, scale=0.125, precision_map_all=bits,
                                          candidates=[], flat_lengths=[]), served=served)


def test_errors_are_the_python_path_s(device):
    x = torch.randn(64, 2, 64, device=device).half()
    cu = torch.tensor([0, 64], dtype=torch.int32, device=device)
    bits = _bitmask(2, 64, 64, device)
    kw = dict(block_m=64, block_n=64, causal=True, scalar_scales=False, routing_mode="mixed", int8_use_fp16_v=True)
    with pytest.raises(ValueError, match="rows, expected"):
        tmx.tilemix_attention_with_quant(x, x, x, cu, cu, 64, 64, bits[:1], **kw)
    with pytest.raises(ValueError, match="requires equal Q/K lengths"):
        tmx.tilemix_attention_with_quant(x, x, x, cu, cu, 64, 32, bits, **kw)
    with pytest.raises(ValueError, match="scalar_scales requires"):
        tmx.tilemix_attention_with_quant(x, x, x, cu, cu, 64, 64, bits, **{**kw, "scalar_scales": True})
    with pytest.raises(TypeError, match="float16"):
        tmx.tilemix_attention_with_quant(x.float(), x.float(), x.float(), cu, cu, 64, 64, bits, **kw)


@pytest.mark.parametrize("lengths", [[64], [130, 0, 1, 257], [0, 3]])
def test_quantize(device, both, lengths):
    q, k, v, cu = packed_inputs(lengths, 4, 2, 80, seed=9)
    dq, dk, dv, dcu = (to_dev(x, device) for x in (q, k, v, cu))
    longest = max(lengths)
    assert len(both(lambda: tmx.quantize_qkv_for_tilemix(dq, dk, dv, dcu, dcu, longest, longest))) == 9
    both(lambda: tmx.quantize_qk_for_tilemix(dq, dk, dcu, dcu, longest, longest, BLKQ=96, BLKK=32))
    both(lambda: tmx.quantize_qk_for_tilemix(dq, dk, dcu.cpu(), dcu, longest, longest), served=False)
    both(lambda: tmx.quantize_qk_for_tilemix(dq, dk[:, :, :72], dcu, dcu, longest, longest))


def test_helpers(device, both):
    g = torch.Generator(device=device).manual_seed(7)
    x = torch.randn(3, 5, 200, generator=g, device=device).half()
    w = torch.randn(200, generator=g, device=device).half()
    both(lambda: TL.rms_norm(x, w, 1e-6))
    both(lambda: TL.rms_norm(x[:, :, :104], w[:104], 1e-6), served=False)
    both(lambda: TL.silu_mul(x, x + 1))
    q, k = (torch.randn(2, 9, h, 64, generator=g, device=device).half().transpose(1, 2) for h in (5, 3))
    for batch in (1, 2):
        c, s = (torch.randn(batch, 9, 64, generator=g, device=device).half() for _ in range(2))
        both(lambda: TL.rotary_token_major(q, k, c, s))
        both(lambda: TL.rotary_token_major(q.contiguous(), k.contiguous(), c, s))


def test_stream_and_capture(device):
    """A call on another stream, and a captured call replayed between eager ones on new inputs."""
    g = torch.Generator(device=device).manual_seed(8)
    q, k, v = (torch.randn(2, 160, h, 128, generator=g, device=device).half().transpose(1, 2) for h in (4, 2, 2))
    bits = _bitmask(2, 160, 64, device)

    def call():
        return tilemix_varlen_attention(q, k, v, 64, 64, causal=True, scale=0.1, precision_map_all=bits,
                                        candidates=[], flat_lengths=[])

    want = call()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = call()
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for i in range(4):
        for t in (q, k, v):
            t.copy_(torch.randn(t.shape, generator=g, device=device).half())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, call()), i
