"""Per-block int8 quantisation of varlen token-major tensors on the HIP library.

Same public functions, arguments and results as the reference module
attention/triton/quant_per_block_varlen.py:

* ``per_block_int8_single(x, cu_seqlens_x, max_seqlen_x, BLK=128, sm_scale=1.0)``
  (reference :48-75) -> ``(x_int8, x_scale fp32 [rows, H], cu_seqlens_x_scale int64 [B+1])``
* ``per_block_int8(q, k, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
  BLKQ=128, BLKK=64, sm_scale=None)`` (reference :78-106).

The device kernel computes the scale-row prefix itself, so the internal
``quantize_many`` used by the attention entry needs no device->host copy, and it
takes Q, K and V in one launch.
The public functions still return scale tensors with exactly
``cu_seqlens_x_scale[-1]`` rows, which needs the row counts on the host: they are
taken from ``cu_seqlens_x`` directly when that lives on the CPU, otherwise read
back in one copy per call (the reference reads them back too, :62-63).
"""
from __future__ import annotations

import torch

from ... import _native


def _scale_capacity(n_tokens: int, batch: int, blk: int) -> int:
    # sum_b ceil(L_b / blk) <= ceil(sum_b L_b / blk) + batch, with sum_b L_b <= n_tokens
    return (n_tokens + blk - 1) // blk + batch


def _prepare_input(x: torch.Tensor) -> torch.Tensor:
    if x.ndim != 3:
        raise ValueError("expected a flattened [tokens, heads, dim] tensor")
    if x.dtype != torch.float16:
        raise TypeError(f"TileMix HIP quantisation supports float16 input, got {x.dtype}")
    if not x.is_cuda:
        raise RuntimeError("TileMix quantisation runs on the GPU (HIP); got a CPU tensor")
    if x.stride(2) != 1 or x.stride(0) % 8 or x.stride(1) % 8 or x.data_ptr() % 16:
        x = x.contiguous()
    return x


def _outputs(p: _native.QuantParams, x: torch.Tensor, cu: torch.Tensor, max_seqlen, blk, sm_scale, half_scales: bool,
             cu_scale_ptr: int):
    """Allocate one tensor's codes and scales and describe its quantisation in ``p``."""
    device, heads, dim, batch = x.device, x.shape[1], x.shape[2], cu.numel() - 1
    if dim % 8:
        raise ValueError(f"head_dim must be a multiple of 8, got {dim}")
    cap = _scale_capacity(x.shape[0], batch, blk)
    codes = torch.empty(x.shape, dtype=torch.int8, device=device)
    scale = torch.empty((cap, heads), dtype=torch.float32, device=device)
    scale16 = torch.empty((cap, heads), dtype=torch.float16, device=device) if half_scales else None
    p.input = x.data_ptr()
    p.output = codes.data_ptr()
    p.scale = scale.data_ptr()
    p.scale_half = scale16.data_ptr() if scale16 is not None else None
    p.cu_seqlens = cu.data_ptr()
    p.cu_seqlens_scale = cu_scale_ptr
    p.stride_in_token, p.stride_in_head = x.stride(0), x.stride(1)
    p.stride_out_token, p.stride_out_head = codes.stride(0), codes.stride(1)
    p.scale_rows_capacity = cap
    p.sm_scale = float(sm_scale)
    p.heads, p.head_dim, p.blk_tokens = heads, dim, int(blk)
    p.batch, p.max_seqlen = batch, int(max_seqlen)
    return codes, scale, scale16


def quantize_blocks(x: torch.Tensor, cu_seqlens: torch.Tensor, max_seqlen: int, blk: int,
                    sm_scale: float = 1.0, *, half_scales: bool = False):
    """Quantise without any host synchronisation.

    Returns ``(codes int8 like x, scale fp32 [capacity, H], scale16 fp16 [capacity, H] | None,
    cu_scale int32 [B+1])``; rows of the scale tensors past ``cu_scale[-1]`` are
    unused.
    """
    x = _prepare_input(x)
    device = x.device
    cu = cu_seqlens.to(device=device, dtype=torch.int32).contiguous()
    batch = cu.numel() - 1
    cu_scale = torch.empty(batch + 1, dtype=torch.int32, device=device)
    p = _native.QuantParams()
    codes, scale, scale16 = _outputs(p, x, cu, max_seqlen, blk, sm_scale, half_scales, cu_scale.data_ptr())
    if batch > 0:
        _native.quant_per_block_int8(p, device)
    else:
        cu_scale.zero_()
    return codes, scale, scale16, cu_scale


def quantize_many(items, *, half_scales: bool = False):
    """``quantize_blocks`` of two or three tensors ``(x, cu_seqlens, max_seqlen, blk, sm_scale)``
    in one launch: the list of ``(codes, scale, scale16 | None)`` and the scale-row prefixes
    int32 [len(items), B+1] (a list of them where the batches or devices differ: one
    launch each then)."""
    prepared = []
    for x, cu_seqlens, *rest in items:
        x = _prepare_input(x)
        prepared.append((x, cu_seqlens.to(device=x.device, dtype=torch.int32).contiguous(), *rest))
    device, entries = prepared[0][0].device, prepared[0][1].numel()
    if any(x.device != device or cu.numel() != entries for x, cu, *_ in prepared[1:]):
        done = [quantize_blocks(*item, half_scales=half_scales) for item in prepared]
        return [r[:3] for r in done], [r[3] for r in done]
    cu_scales = torch.empty((len(prepared), entries), dtype=torch.int32, device=device)
    params = (_native.QuantParams * len(prepared))()
    results = [_outputs(p, *item, half_scales, cu_scales.data_ptr() + 4 * i * entries)
               for i, (p, item) in enumerate(zip(params, prepared))]
    if entries > 1:
        _native.quant_per_block_int8_many(params, device)
    else:
        cu_scales.zero_()
    return results, cu_scales


def scale_rows(items, cu_scales) -> list[int]:
    """Scale rows of each item of a ``quantize_many`` call: from its ``cu_seqlens`` where that
    lives on the CPU, else from the prefixes the launch wrote (one copy to the host for all of
    them; the reference reads each back, :62-63)."""
    rows = []
    for _, cu_seqlens, _, blk, _ in items:
        if cu_seqlens.device.type != "cpu":
            ends = cu_scales.cpu() if isinstance(cu_scales, torch.Tensor) else [c.cpu() for c in cu_scales]
            return [int(c[-1]) for c in ends]
        lens = (cu_seqlens[1:] - cu_seqlens[:-1]).to(torch.int64)
        rows.append(int(((lens + blk - 1) // blk).sum()))
    return rows


@torch.no_grad()
def per_block_int8_single(x, cu_seqlens_x, max_seqlen_x, BLK=128, sm_scale=1.0):
    """Reference attention/triton/quant_per_block_varlen.py:48-75."""
    codes, scale, _, cu_scale = quantize_blocks(x, cu_seqlens_x, max_seqlen_x, BLK, sm_scale)
    [rows] = scale_rows([(x, cu_seqlens_x, max_seqlen_x, BLK, sm_scale)], [cu_scale])
    return codes, scale[:rows], cu_scale.to(torch.int64)


@torch.no_grad()
def per_block_int8(q, k, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
                   BLKQ=128, BLKK=64, sm_scale=None):
    """Reference attention/triton/quant_per_block_varlen.py:78-106 (same Q sm_scale rule)."""
    head_dim = q.shape[-1]
    if sm_scale is None:
        sm_scale = head_dim ** -0.5
    if abs(sm_scale - 1.0) < 1e-6:
        q_sm_scale = 1.0
    else:
        q_sm_scale = sm_scale * 1.44269504
    items = [(q, cu_seqlens_q, max_seqlen_q, BLKQ, q_sm_scale), (k, cu_seqlens_k, max_seqlen_k, BLKK, 1.0)]
    [(q_int8, q_scale, _), (k_int8, k_scale, _)], cu_scales = quantize_many(items)
    rows_q, rows_k = scale_rows(items, cu_scales)
    return (q_int8, q_scale[:rows_q], k_int8, k_scale[:rows_k],
            cu_scales[0].to(torch.int64), cu_scales[1].to(torch.int64))
