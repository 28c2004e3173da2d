"""Argument validation of the uniform-length and several-tensor C entry points (CPU: a
call that fails validation returns before any HIP call)."""
from __future__ import annotations

import ctypes

import pytest

from tilemix_amd import _native


@pytest.fixture(scope="module")
def lib():
    return _native.load_library()


def test_uniform_attention_validation(lib):
    assert lib.tilemix_attn_fwd_uniform(None, 64, None) == 1
    p = _native.AttnParams()
    assert lib.tilemix_attn_fwd_uniform(ctypes.byref(p), 0, None) == 1
    assert b"no tokens" in lib.tilemix_last_error()
    for f in ("q", "k", "v", "out"):
        setattr(p, f, ctypes.c_void_p(16))
    p.max_seqlen_q, p.max_seqlen_k = 64, 65
    assert lib.tilemix_attn_fwd_uniform(ctypes.byref(p), 64, None) == 1
    assert b"must equal the uniform length" in lib.tilemix_last_error()
    p.max_seqlen_k, p.batch = 64, 1 << 26
    assert lib.tilemix_attn_fwd_uniform(ctypes.byref(p), 64, None) == 1
    assert b"32-bit token index" in lib.tilemix_last_error()
    p.batch = 1
    assert lib.tilemix_attn_fwd(ctypes.byref(p), None) == 1  # without a uniform length: cu arrays needed
    assert b"cu_seqlens" in lib.tilemix_last_error()


def test_several_tensors_validation(lib):
    q = (_native.QuantParams * 3)()
    assert lib.tilemix_quant_per_block_int8_many(None, 1, 0, None) == 1
    for count, uniform in ((0, 0), (4, 0), (1, -1)):
        assert lib.tilemix_quant_per_block_int8_many(q, count, uniform, None) == 1
        assert b"1 to 3 tensors" in lib.tilemix_last_error()
    for s, batch in zip(q, (1, 1, 2)):
        s.input = s.output = s.scale = 16
        s.heads, s.head_dim, s.blk_tokens, s.batch = 1, 64, 64, batch
    assert lib.tilemix_quant_per_block_int8_many(q, 3, 64, None) == 1
    assert b"share the batch" in lib.tilemix_last_error()
    assert lib.tilemix_quant_per_block_int8_many(q, 1, 0, None) == 1  # no uniform length: cu_seqlens needed
    assert b"null tensor pointer" in lib.tilemix_last_error()


def test_uniform_quantisation_token_index(lib):
    """More tokens than a 32-bit index holds are refused before anything is launched."""
    p = (_native.QuantParams * 1)()
    p[0].input = p[0].output = p[0].scale = 16
    p[0].heads, p[0].head_dim, p[0].blk_tokens = 1, 8, 64
    for length, batch in ((1 << 16, 1 << 15), (64, 1 << 26), (2**31 - 1, 2)):
        p[0].batch = batch
        assert lib.tilemix_quant_per_block_int8_many(p, 1, length, None) == 1
        assert b"32-bit token index" in lib.tilemix_last_error()


def test_quantisation_block_limit(lib):
    """A sequence of 2^24 blocks or more is refused with the limit (HIP launches fewer than 2^32 threads
    along x); what lies between is launched in pieces."""
    p = (_native.QuantParams * 1)()
    p[0].input = p[0].output = p[0].scale = p[0].cu_seqlens = 16
    p[0].heads, p[0].head_dim, p[0].blk_tokens, p[0].batch, p[0].max_seqlen = 1, 8, 1, 1, 1 << 24
    assert lib.tilemix_quant_per_block_int8_many(p, 1, 0, None) == 1
    assert b"at most 16777215 blocks" in lib.tilemix_last_error()


def test_attention_token_stride(lib):
    """Tokens closer than their rows are long are refused (a sequence's reads are bounded by its length
    times the token stride, so the last rows would read zeros)."""
    p = _native.AttnParams()
    for f in ("q", "k", "v", "out", "precision_bitmask", "cu_seqlens_q", "cu_seqlens_k"):
        setattr(p, f, ctypes.c_void_p(1 << 12))
    p.heads_q = p.heads_k = p.batch = 1
    p.head_dim, p.max_seqlen_q, p.max_seqlen_k = 64, 128, 128
    p.block_m, p.block_n, p.block_n_mask, p.blkq, p.blkk, p.routing_mode = 128, 64, 64, 128, 64, 1
    strides = ("stride_q_token", "stride_k_token", "stride_v_token")
    for short in strides:
        for f in strides:
            setattr(p, f, 56 if f == short else 64)
        assert lib.tilemix_attn_fwd(ctypes.byref(p), None) == 1
        assert b"token strides must be at least head_dim" in lib.tilemix_last_error()
