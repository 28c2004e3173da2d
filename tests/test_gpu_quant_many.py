"""Quantisation launches of one to three tensors: widths whose 8-element chunks
divide the workgroup and widths that leave threads idle, blocks held in registers
and streamed ones, ragged and empty sequences, non-finite values, and uniform
lengths without cu_seqlens.  Codes, scales and prefixes are bit-exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import packed_inputs, to_dev
from oracle import tilemix_oracle as O
from tilemix_amd import _native
from tilemix_amd.attention.hip.quant_per_block_varlen import quantize_blocks, quantize_many

pytestmark = pytest.mark.gpu


def _check(codes, scale, scale16, cu_scale, x, cu, blk, sm=1.0):
    rc, rs, rcu = O.quant_per_block_int8(x, cu, blk, sm_scale=sm)
    rows, n = int(rcu[-1]), int(cu[-1])
    assert cu_scale.cpu().tolist() == rcu.tolist()
    np.testing.assert_array_equal(codes.cpu().numpy()[:n], rc[:n])
    np.testing.assert_array_equal(scale.cpu().numpy()[:rows].view(np.uint32), rs.view(np.uint32))
    if scale16 is not None:
        np.testing.assert_array_equal(scale16.cpu().numpy()[:rows].view(np.uint16),
                                      rs.astype(np.float16).view(np.uint16))


# head_dim: chunks per row that divide 256 threads (8, 64, 256) and that do not (24, 80, 120, 136);
# BLK: one row group, exactly the register path's last row group, one past it, streamed.
@pytest.mark.parametrize("dim,blk", [(8, 64), (24, 48), (64, 256), (80, 200), (80, 201), (120, 128), (128, 128),
                                     (128, 129), (136, 64), (256, 64), (256, 65)])
def test_three_tensors_in_one_launch(device, dim, blk):
    lengths = [blk, 0, 1, 2 * blk + 3, blk - 1]
    q, k, v, cu = packed_inputs(lengths, 3, 2, dim, seed=dim + blk)
    q[lengths[0]:lengths[0] + 1] = 0  # an all-zero block (sequence 2): scale 0, codes 0
    dcu = to_dev(cu, device)
    items = [(to_dev(q, device), dcu, max(lengths), blk, 1.0), (to_dev(k, device), dcu, max(lengths), 64, 1.0),
             (to_dev(v, device), dcu, max(lengths), blk, 0.7)]
    results, cu_scales = quantize_many(items, half_scales=True)
    torch.cuda.synchronize()
    for (codes, scale, scale16), cus, x, (_, _, _, b, sm) in zip(results, cu_scales, (q, k, v), items):
        _check(codes, scale, scale16, cus, x, cu, b, sm)


@pytest.mark.parametrize("bad", [0x7c00, 0xfc00, 0x7e00, 0x7c01, 0xfdff])  # +-inf, quiet and signalling NaNs
def test_block_maximum_ignores_nans(device, bad):
    """The block maximum ignores NaNs and their codes are 0; an infinity makes the scale infinite
    and every code of its block 0.  Other blocks are unaffected."""
    rng = np.random.default_rng(bad)
    x = rng.standard_normal((130, 2, 128)).astype(np.float16)
    x.view(np.uint16)[70, 1, 5] = bad
    cu = np.array([0, 130], dtype=np.int32)
    codes, scale, _, _ = quantize_blocks(to_dev(x, device), to_dev(cu, device), 130, 64)
    clean = x.copy()
    clean[70, 1, 5] = 0
    rc, rs, _ = O.quant_per_block_int8(clean, cu, 64)
    if bad in (0x7c00, 0xfc00):
        rc[64:128, 1] = 0
        rs[1, 1] = np.inf
    np.testing.assert_array_equal(codes.cpu().numpy(), rc)
    np.testing.assert_array_equal(scale.cpu().numpy()[:3].view(np.uint32), rs.view(np.uint32))


@pytest.mark.parametrize("length", [1, 64, 130])
def test_uniform_lengths_equal_cu_seqlens(device, length):
    batch, heads, dim, blk = 3, 2, 128, 64
    x = torch.randn(batch * length, heads, dim, device=device).half()
    cu = torch.arange(0, (batch + 1) * length, length, dtype=torch.int32, device=device)
    codes, scale, scale16, cu_scale = quantize_blocks(x, cu, length, blk, half_scales=True)
    got = [torch.full_like(t, 1) for t in (codes, scale, scale16, cu_scale)]
    params = (_native.QuantParams * 1)()
    p = params[0]
    p.input, p.output, p.scale, p.scale_half = x.data_ptr(), got[0].data_ptr(), got[1].data_ptr(), got[2].data_ptr()
    p.cu_seqlens_scale = got[3].data_ptr()
    p.stride_in_token, p.stride_in_head, p.stride_out_token, p.stride_out_head = heads * dim, dim, heads * dim, dim
    p.scale_rows_capacity, p.sm_scale = scale.shape[0], 1.0
    p.heads, p.head_dim, p.blk_tokens, p.batch = heads, dim, blk, batch
    _native.quant_per_block_int8_many(params, device, uniform_seqlen=length)
    torch.cuda.synchronize()
    rows = int(cu_scale[-1])
    for a, b, n in zip(got, (codes, scale, scale16, cu_scale), (len(codes), rows, rows, batch + 1)):
        assert torch.equal(a[:n], b[:n])


def test_more_blocks_than_one_launch_takes(device):
    """Blocks of one token: 9 + 17 heads of 2^20 + 3 tokens are more workgroups than a launch has
    (2^24 of 256 threads), and the 17 heads alone are, too."""
    n = (1 << 20) + 3
    cu = torch.tensor([0, n], dtype=torch.int32, device=device)
    g = torch.Generator(device=device).manual_seed(11)
    xs = [torch.randn(n, heads, 8, generator=g, device=device).half() for heads in (9, 17)]
    results, cu_scales = quantize_many([(x, cu, n, 1, 1.0) for x in xs], half_scales=True)
    torch.cuda.synchronize()
    assert cu_scales.tolist() == [[0, n], [0, n]]
    for x, (codes, scale, scale16) in zip(xs, results):
        amax = x.abs().amax(-1).float()
        want = amax / torch.full_like(amax, 127.0)  # IEEE quotients: by a Python number torch multiplies by 1/127
        assert torch.equal(scale[:n], want) and torch.equal(scale16[:n], want.half())
        t = x.float() / want[..., None]
        assert torch.equal(codes, torch.trunc(t + torch.where(t >= 0, 0.5, -0.5)).to(torch.int8))


@pytest.mark.parametrize("heads,dim,blk", [(1, 8, 1), (3, 24, 1), (5, 64, 3), (24, 128, 4), (7, 256, 16), (2, 136, 17)])
def test_one_tensor_small_blocks(device, heads, dim, blk):
    """Many workgroups of few rows, most of the grid empty: one long sequence among short and empty ones."""
    lengths = [2, 0, 301, 1, blk, 0]
    x, _, _, cu = packed_inputs(lengths, heads, heads, dim, seed=heads + blk)
    codes, scale, scale16, cu_scale = quantize_blocks(to_dev(x, device), to_dev(cu, device), 301, blk, half_scales=True)
    torch.cuda.synchronize()
    _check(codes, scale, scale16, cu_scale, x, cu, blk)


@pytest.mark.parametrize("batch", [1, 64, 65, 257, 1100])
def test_scale_rows_of_many_sequences(device, batch):
    """The scale-row base is summed by four waves, 64 earlier sequences each at a time."""
    rng = np.random.default_rng(batch)
    lengths = rng.integers(0, 9, batch).tolist()
    lengths[-1] = 5
    x, _, _, cu = packed_inputs(lengths, 2, 2, 8, seed=batch)
    codes, scale, scale16, cu_scale = quantize_blocks(to_dev(x, device), to_dev(cu, device), 8, 3, half_scales=True)
    torch.cuda.synchronize()
    _check(codes, scale, scale16, cu_scale, x, cu, 3)
