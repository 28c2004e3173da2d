"""Prefill helper kernels at the edges of their dispatch: RMSNorm widths on both sides
of every per-lane chunk count, rotary head dims around the workgroup shapes (head slots,
tokens per workgroup, the element-wise limit) with ragged token and head counts, and
SiLU * up on every fp16 gate.  Bars as in test_gpu_prefill_helpers.py."""
from __future__ import annotations

import pytest
import torch

from oracle import prefill_oracle as PO
from test_gpu_prefill_helpers import _rope_inputs, _within_ulps
from tilemix_amd.models import tilemix_llama as TL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [8, 512, 1024, 1032, 2048, 2056, 3072, 3075, 3080, 4096, 4104, 8184, 8192, 8200])
@pytest.mark.parametrize("rows", [1, 6])
def test_rms_norm_chunk_counts(device, cols, rows):
    g = torch.Generator().manual_seed(cols + rows)
    x = torch.randn(rows, cols, generator=g).half()
    w = (torch.randn(cols, generator=g) * 0.3 + 1.0).half()
    ok, frac = _within_ulps(TL.rms_norm(x.to(device), w.to(device), 1e-5), PO.rms_norm(x, w, 1e-5), 2)
    assert ok and frac <= max(0.01, 1.5 / (rows * cols)), frac


def test_rms_norm_row_stride_aligned_and_not(device):
    """Rows of 3072 columns inside wider buffers: a stride that keeps 16-byte alignment and one that does not."""
    g = torch.Generator().manual_seed(5)
    w = (torch.randn(3072, generator=g) * 0.3 + 1.0).half()
    for width in (3088, 3076):
        base = torch.randn(9, width, generator=g).half()
        got = TL.rms_norm(base.to(device)[:, :3072], w.to(device), 1e-5)
        ok, frac = _within_ulps(got, PO.rms_norm(base[:, :3072], w, 1e-5), 2)
        assert ok and frac <= 0.01, (width, frac)


@pytest.mark.parametrize("cols,width", [(3072, 3076), (3072, 3075), (512, 516), (8192, 8196), (2056, 2060),
                                        (4096, 4100), (4104, 4108), (6400, 6402), (8184, 8196)])
def test_rms_norm_aligned_rows_of_an_odd_stride(device, cols, width):
    """Alignment is each row's own: the 16-byte aligned rows among unaligned ones have the bits of an aligned
    tensor's (the order of the sum is the vector path's)."""
    g = torch.Generator().manual_seed(cols + width)
    base = torch.randn(256, width, generator=g).half().to(device)
    w = (torch.randn(cols, generator=g) * 0.3 + 1.0).half().to(device)
    rows = [r for r in range(256) if r * width % 8 == 0]
    got, want = TL.rms_norm(base[:, :cols], w, 1e-5), TL.rms_norm(base[:, :cols].contiguous(), w, 1e-5)
    assert torch.equal(got[rows], want[rows])
    ok, frac = _within_ulps(got, PO.rms_norm(base[:, :cols].cpu(), w.cpu(), 1e-5), 2)
    assert ok and frac <= 0.01, frac


@pytest.mark.parametrize("b,hq,hk,t,d", [
    (1, 17, 1, 1, 16),      # one chunk pair per row, one head past the 16 slots
    (2, 33, 16, 5, 64),     # three passes over the head slots
    (3, 5, 5, 7, 80),       # pairs that do not divide the workgroup
    (1, 16, 15, 3, 256),    # one token per workgroup
    (1, 20, 2, 3, 272),     # fewer than 16 head slots
    (1, 2, 1, 2, 4096),     # one head slot, one token
    (1, 2, 1, 2, 4112),     # past the vector path
    (1, 1, 1, 1, 128),      # fewer rows than a workgroup takes
    (3, 4, 1, 13, 64),      # rows that end within a workgroup
    (1, 20, 4, 11, 80),     # whole tokens per workgroup: 48 of its 51 rows
    (2, 1, 1, 33, 128),     # two heads; the last workgroup a fraction of a token
])
def test_rotary_shapes_bitexact(device, b, hq, hk, t, d):
    q, k, cos, sin = _rope_inputs(b, hq, hk, t, d, b, seed=d + t, device=device)
    wq, wk = PO.rotary_token_major(q, k, cos, sin)
    gq, gk = TL.rotary_token_major(q.to(device), k.to(device), cos.to(device), sin.to(device))
    assert torch.equal(gq.cpu(), wq) and torch.equal(gk.cpu(), wk)
    hm_q, hm_k = (x.contiguous().to(device) for x in (q, k))  # head-major inputs
    gq, gk = TL.rotary_token_major(hm_q, hm_k, cos.to(device), sin.to(device))
    assert torch.equal(gq.cpu(), wq) and torch.equal(gk.cpu(), wk)


@pytest.mark.parametrize("up", [1.0, -0.37])
def test_silu_mul_every_gate(device, up):
    """All 65536 fp16 gates: infinities and NaNs as in the formula, finite results within one ulp."""
    gate = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.float16)
    ups = torch.full_like(gate, up)
    got, want = TL.silu_mul(gate.to(device), ups.to(device)).cpu(), PO.silu_mul(gate, ups)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]) and torch.isfinite(got[finite]).all()
    ok, frac = _within_ulps(got[finite], want[finite], 1)
    assert ok and frac <= 1e-3, frac


def test_silu_mul_smallest_gates(device):
    """The gates up to 2^-20, exactly: there exp(-g) and the denominators are the nearest fp32 values, and a
    quotient one ulp off (the denominator 2 - 2^-23) would show in no other gate."""
    gate = torch.arange(0, 17, dtype=torch.int16).view(torch.float16)
    gate = torch.cat((gate, -gate))
    ones = torch.ones_like(gate)
    got, want = TL.silu_mul(gate.to(device), ones.to(device)).cpu(), PO.silu_mul(gate, ones)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
