"""The attention modules' rotary embedding: transformers' apply_rotary_pos_emb bit for bit
where one kernel serves it, and apply_rotary_pos_emb itself where a graph is recorded."""
from __future__ import annotations

import pytest
import torch
from transformers.models.llama.modeling_llama import apply_rotary_pos_emb

from tilemix_amd import _native
from tilemix_amd.models._common import apply_rotary

pytestmark = pytest.mark.gpu


def _operands(device, b, hq, hk, t, d, layout, cos_batch, dtype=torch.float16):
    g = torch.Generator(device=device).manual_seed(t + d)
    q, k = (torch.randn(b, t, h, d, generator=g, device=device).mul_(3).to(dtype).transpose(1, 2) for h in (hq, hk))
    if layout == "head_major":
        q, k = q.contiguous(), k.contiguous()
    angle = torch.randn(cos_batch, t, d // 2, generator=g, device=device)
    angle = torch.cat((angle, angle), -1)
    return q, k, angle.cos().to(dtype), angle.sin().to(dtype)


@pytest.mark.parametrize("b,hq,hk,t,d,cos_batch", [(1, 28, 4, 37, 128, 1), (2, 14, 2, 5, 64, 2), (2, 3, 1, 4, 72, 1),
                                                   (1, 4, 4, 1, 16, 1)])
@pytest.mark.parametrize("layout", ["token_major", "head_major"])
def test_equals_transformers(device, b, hq, hk, t, d, cos_batch, layout):
    args = _operands(device, b, hq, hk, t, d, layout, cos_batch)
    with torch.no_grad():
        got, want = apply_rotary(*args), apply_rotary_pos_emb(*args)
        assert _native.host().rotary(*args) is not None
    for a, w in zip(got, want):
        assert a.shape == w.shape and torch.equal(a.contiguous().view(torch.int16), w.contiguous().view(torch.int16))


def test_recorded_graphs_take_the_torch_ops(device):
    q, k, cos, sin = _operands(device, 1, 2, 1, 8, 64, "token_major", 1)
    q.requires_grad_(True)
    out, _ = apply_rotary(q, k, cos, sin)
    assert out.grad_fn is not None
    out.float().sum().backward()
    assert q.grad is not None
    traced = torch.jit.trace(lambda *a: apply_rotary(*a), (q.detach(), k, cos, sin), check_trace=False)
    other = _operands(device, 1, 2, 1, 8, 64, "head_major", 1)
    q2 = other[0] + 1
    assert torch.equal(traced(q2, k, cos, sin)[0], apply_rotary_pos_emb(q2, k, cos, sin)[0])
    batched = torch.vmap(lambda x: apply_rotary(x, k, cos, sin)[0])(torch.stack([q.detach(), q2]))
    assert torch.equal(batched[1], apply_rotary_pos_emb(q2, k, cos, sin)[0])
    from torch.autograd import forward_ad as fwd
    with fwd.dual_level():
        dual = fwd.make_dual(q.detach(), q2)
        assert fwd.unpack_dual(apply_rotary(dual, k, cos, sin)[0]).tangent is not None
    f32 = _operands(device, 1, 2, 1, 8, 64, "token_major", 1, torch.float32)
    assert torch.equal(apply_rotary(*f32)[0], apply_rotary_pos_emb(*f32)[0])
