"""Performance cases of the framework: the calls a program makes when it prefills
with TileMix, through the public entry points, and the plain 64-bit evaluation of
each (``exact``).

The framework has one direction, the prefill forward (it has no backward, and a
decode step below 16 tokens runs the model's own attention), so the cases span its
entry points instead: the dense attention call of the model glue, the packed
cu_seqlens call, the int8 quantisation API, the prefill helper kernels, an attention
module and a whole (short) model.
"""
from __future__ import annotations

import functools
import math
import random

import torch
from torch import nn

from tilemix_amd.attention import precision_maps
from tilemix_amd.attention.hip.tilemix import quantize_qkv_for_tilemix, tilemix_attention_with_quant
from tilemix_amd.attention.tilemix_varlen import tilemix_varlen_attention
from tilemix_amd.models import tilemix_llama, tilemix_qwen
from tilemix_amd.models._common import pick_mask_block_n

DEVICE = "cuda"
OUTLIER_CHANNELS = (7, 33, 70, 101)  # the benchmark's x8 channels of Q and K
SPTRANS = {"stride": 128, "c": 32}


def _attn(**kw) -> dict:
    """An attention call.  entry: "dense" ([B, H, T, D], the model glue's call) or
    "packed" (cu_seqlens).  seqs sequences of `length` tokens, or, with shortest < length,
    of shortest..length tokens drawn from `pick`."""
    case = {"kind": "attention", "entry": "packed", "seqs": 1, "length": 1024, "shortest": 0, "pick": 0,
            "heads": 24, "kv_heads": 8, "dim": 128, "block_m": 128, "layout": "sptrans", "int8_share": 0.5,
            "mode": "auto", "int8_v": False, "causal": True, "outliers": False}
    case.update(kw)
    return case


def listed() -> list[dict]:
    return [
        # The smallest call: one short prompt of a small model (the repository's 256-token
        # configuration); latency of the host path and of the launches.
        _attn(name="attn_256", entry="dense", length=256, heads=4, kv_heads=1, dim=64, block_m=64, layout="band",
              mode="mixed"),
        # One chat prompt of about a thousand tokens, not a multiple of any tile.
        _attn(name="attn_prompt_1000", entry="dense", length=1000, block_m=64, mode="mixed"),
        # A batch of prompts at the block size the model glue takes below 4096 tokens.
        _attn(name="attn_8x2048", entry="dense", seqs=8, length=2048, block_m=64, mode="mixed"),
        # The benchmark's workload: 8 x 4096, outlier channels, packed entry.
        _attn(name="attn_8x4096", seqs=8, length=4096, outliers=True),
        # A serving batch: 24 packed prompts of mixed odd lengths.
        _attn(name="attn_packed_24", seqs=24, length=8192, shortest=512, pick=4, heads=32, layout="align_sparse"),
        # The longest context: one 32768-token document, mask groups of 8 tiles, GQA 7.
        _attn(name="attn_32768", length=32768, heads=28, kv_heads=4, layout="bigbird"),
        # head_dim 64 models.
        _attn(name="attn_8x2048_d64", entry="dense", seqs=8, length=2048, heads=32, dim=64, block_m=64, mode="mixed"),
        # PV on int8 V codes for the INT8 tiles (the option of the packed entry that
        # TILEMIX_SCORE_ONLY_PV=0 selects in the dense one), ragged prompts.
        _attn(name="attn_int8v_packed_8", seqs=8, length=3000, shortest=300, pick=8, heads=32, mode="mixed",
              int8_v=True),
        # The quantisation API alone (a program that quantises once and launches several maps).
        {"name": "quantize_16384", "kind": "quantize", "tokens": 16384, "heads": 24, "kv_heads": 8, "dim": 128},
        # One decoder layer's elementwise kernels at the end-to-end benchmark's 32768 tokens.
        {"name": "helpers_32768", "kind": "helpers", "tokens": 32768, "hidden": 3072, "inner": 8192, "heads": 24,
         "kv_heads": 8, "dim": 128},
        # An attention module of a Qwen2 model on one odd-length prompt.
        {"name": "qwen_attention_1537", "kind": "qwen", "seqs": 1, "length": 1537, "heads": 28, "kv_heads": 4,
         "dim": 128},
        # Model prefill into a cache: the end-to-end benchmark's layers (two of them) and helpers.
        {"name": "llama_prefill_2x1024", "kind": "llama", "seqs": 2, "length": 1024, "layers": 2, "heads": 24,
         "kv_heads": 8, "dim": 128, "inner": 8192, "vocab": 8192},
    ]


def _spread(rng: random.Random, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random) -> dict:
    u = rng.random()
    if u < 0.10:
        heads, kv_heads = rng.choice([(24, 8), (32, 8), (28, 4), (4, 1)])
        return {"kind": "quantize", "tokens": _spread(rng, 17, 32768), "heads": heads, "kv_heads": kv_heads,
                "dim": rng.choice([64, 128])}
    if u < 0.30:
        heads, kv_heads, dim = rng.choice([(24, 8, 128), (32, 8, 64), (32, 8, 128)])
        hidden = heads * dim
        return {"kind": "helpers", "tokens": _spread(rng, 16, 32768), "hidden": hidden,
                "inner": rng.choice([hidden * 8 // 3 // 8 * 8, 4 * hidden, 8192]), "heads": heads,
                "kv_heads": kv_heads, "dim": dim}
    if u < 0.38:
        heads, kv_heads = rng.choice([(28, 4), (14, 2)])
        return {"kind": "qwen", "seqs": rng.choice([1, 2, 4]), "length": _spread(rng, 33, 4200), "heads": heads,
                "kv_heads": kv_heads, "dim": rng.choice([64, 128])}
    if u < 0.44:
        return {"kind": "llama", "seqs": rng.choice([1, 2, 4]), "length": _spread(rng, 17, 4200), "layers": 2,
                "heads": 24, "kv_heads": 8, "dim": 128, "inner": 8192, "vocab": 8192}
    length = _spread(rng, 16, 32768)
    seqs = max(1, min(24, _spread(rng, 1, 32), 65536 // length))
    heads, kv_heads = rng.choice([(4, 1), (14, 2), (24, 8), (24, 8), (28, 4), (32, 8)])
    while heads * seqs * length * length > 28 * 32768 * 32768:
        seqs = max(1, seqs // 2)
        heads, kv_heads = 24, 8
        if seqs == 1:
            break
    dense = rng.random() < 0.5
    ragged = not dense and seqs > 1 and rng.random() < 0.7
    return _attn(entry="dense" if dense else "packed", seqs=seqs, length=length,
                 shortest=max(1, length // 16) if ragged else 0, pick=rng.randrange(1 << 16), heads=heads,
                 kv_heads=kv_heads, dim=rng.choice([64, 64, 80, 128, 128, 128]),
                 block_m=64 if dense and length < 4096 else rng.choice([64, 128]) if not dense else 128,
                 layout=rng.choice(["band", "sptrans", "sptrans", "row_rand", "align_sparse", "bigbird", "global"]),
                 int8_share=rng.choice([0.25, 0.5, 0.5, 0.75]),
                 mode=rng.choice(["mixed", "mixed", "mixed", "fp16", "int8"] if dense else
                                 ["auto", "mixed", "mixed", "fp16", "int8"]),
                 int8_v=not dense and rng.random() < 0.25, causal=dense or length > 4096 or rng.random() < 0.7,
                 outliers=rng.random() < 0.3)


# ---- inputs -------------------------------------------------------------------


def _lengths(case: dict) -> list[int]:
    if not case["shortest"]:
        return [case["length"]] * case["seqs"]
    rng = random.Random(case["pick"])
    return [rng.randint(case["shortest"], case["length"]) for _ in range(case["seqs"])]


@functools.lru_cache(maxsize=32)
def _map_row(length: int, block_m: int, mask_n: int, layout: str, share: float) -> torch.Tensor:
    return precision_maps.make_precision_bitmask(
        length, block_m, mask_n, None, percentage=share, pattern_type=layout,
        pattern_params=dict(SPTRANS) if layout == "sptrans" else {}, COMPUTE_BLOCK_N=64)


def _routing(case: dict):
    """(longest sequence, mask-group width, routing rows of every KV head) of an attention case."""
    longest = max(_lengths(case))
    mask_n = pick_mask_block_n(longest, 64)
    return longest, mask_n, _map_row(longest, case["block_m"], mask_n, case["layout"], case["int8_share"]).repeat(
        case["kv_heads"])


def _randn(gen, *shape, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).mul_(scale)


def _attention_inputs(case: dict, seed: int):
    """Token-major q, k, v in fp16: N(0, 1), with the benchmark's x8 channels if asked."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    n = sum(_lengths(case))
    q, k, v = (_randn(gen, n, h, case["dim"]) for h in (case["heads"], case["kv_heads"], case["kv_heads"]))
    if case["outliers"]:
        for c in OUTLIER_CHANNELS:
            q[:, :, c % case["dim"]] *= 8.0
            k[:, :, c % case["dim"]] *= 8.0
    return q.half(), k.half(), v.half()


def _cu_seqlens(lengths: list[int]) -> torch.Tensor:
    ends = [0]
    for n in lengths:
        ends.append(ends[-1] + n)
    return torch.tensor(ends, dtype=torch.int32, device=DEVICE)


def _helper_inputs(case: dict, seed: int) -> dict:
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    t, d = case["tokens"], case["dim"]
    angle = torch.arange(t, device=DEVICE)[:, None] / 500000.0 ** (torch.arange(0, d, 2, device=DEVICE) / d)
    angle = torch.cat((angle, angle), dim=-1)[None]
    return {
        "x": _randn(gen, 1, t, case["hidden"]).half(),
        "weight": (1.0 + _randn(gen, case["hidden"], scale=0.1)).half(),
        "q": _randn(gen, 1, t, case["heads"], d).half().transpose(1, 2),
        "k": _randn(gen, 1, t, case["kv_heads"], d).half().transpose(1, 2),
        "cos": angle.cos().half(), "sin": angle.sin().half(),
        "gate": _randn(gen, 1, t, case["inner"], scale=2.0).half(),
        "up": _randn(gen, 1, t, case["inner"]).half(),
    }


def _seeded_weights(module: nn.Module, seed: int, std: float) -> nn.Module:
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    for name, p in module.named_parameters():
        if p.ndim > 1:
            p.data.copy_(_randn(gen, *p.shape, scale=std))
        elif "norm" in name:
            p.data.copy_(1.0 + _randn(gen, *p.shape, scale=0.1))
        else:
            p.data.copy_(_randn(gen, *p.shape, scale=0.1))
    return module.eval()


def _qwen_module(case: dict, seed: int):
    from transformers import Qwen2Config
    from transformers.models.qwen2.modeling_qwen2 import Qwen2RotaryEmbedding
    hidden = case["heads"] * case["dim"]
    cfg = Qwen2Config(hidden_size=hidden, intermediate_size=2 * hidden, num_hidden_layers=1,
                      num_attention_heads=case["heads"], num_key_value_heads=case["kv_heads"],
                      max_position_embeddings=32768, rope_theta=1000000.0)
    with torch.device(DEVICE):
        module = tilemix_qwen.TileMixqwenAttention(cfg, layer_idx=0).half()
        rotary = Qwen2RotaryEmbedding(cfg)
    module.set_attention_pattern("sptrans", percentage=0.5, **SPTRANS)
    return _seeded_weights(module, seed, hidden ** -0.5), rotary


def _llama_model(case: dict, seed: int):
    from transformers import LlamaConfig, LlamaForCausalLM
    hidden = case["heads"] * case["dim"]
    cfg = LlamaConfig(vocab_size=case["vocab"], hidden_size=hidden, intermediate_size=case["inner"],
                      num_hidden_layers=case["layers"], num_attention_heads=case["heads"],
                      num_key_value_heads=case["kv_heads"], head_dim=case["dim"], rope_theta=500000.0,
                      max_position_embeddings=131072, rms_norm_eps=1e-5, hidden_act="silu",
                      tie_word_embeddings=True)
    with torch.device(DEVICE):
        model = LlamaForCausalLM._from_config(cfg, dtype=torch.float16).eval()
        tilemix_llama.inject_tilemix_into_llama(model)
    tilemix_llama.configure_tilemix_attention_pattern(model, "sptrans", percentage=0.5, **SPTRANS)
    tilemix_llama.prepare_llama_prefill(model)
    return _seeded_weights(model, seed, 0.02)


def _token_ids(case: dict, seed: int) -> torch.Tensor:
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    return torch.randint(case["vocab"], (case["seqs"], case["length"]), generator=gen, device=DEVICE)


def _qwen_hidden(case: dict, seed: int) -> torch.Tensor:
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    return _randn(gen, case["seqs"], case["length"], case["heads"] * case["dim"]).half()


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state = {"case": case}
    if kind == "attention":
        lengths = _lengths(case)
        q, k, v = _attention_inputs(case, seed)
        longest, mask_n, rows = _routing(case)
        state.update(longest=longest, mask_n=mask_n, map=rows.to(DEVICE))
        if case["entry"] == "dense":  # what the model's projections hand over: [B, H, T, D] views
            q, k, v = (t.view(case["seqs"], case["length"], *t.shape[1:]).transpose(1, 2) for t in (q, k, v))
        else:
            state["cu"] = _cu_seqlens(lengths)
        state.update(q=q, k=k, v=v)
    elif kind == "quantize":
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        t, d = case["tokens"], case["dim"]
        state.update(q=_randn(gen, t, case["heads"], d).half(), k=_randn(gen, t, case["kv_heads"], d).half(),
                     v=_randn(gen, t, case["kv_heads"], d).half(), cu=_cu_seqlens([t]))
    elif kind == "helpers":
        state.update(_helper_inputs(case, seed))
    elif kind == "qwen":
        module, rotary = _qwen_module(case, seed)
        hidden = _qwen_hidden(case, seed)
        position = torch.arange(case["length"], device=DEVICE)[None]
        state.update(module=module, hidden=hidden, position_embeddings=rotary(hidden, position))
    else:
        state.update(model=_llama_model(case, seed), ids=_token_ids(case, seed))
    return state


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "attention" and case["entry"] == "dense":
        # the model glue's call (its routing mode comes from the environment there)
        if case["mode"] == "mixed":
            return tilemix_varlen_attention(
                state["q"], state["k"], state["v"], case["block_m"], 64, block_n_mask=state["mask_n"],
                causal=case["causal"], scale=case["dim"] ** -0.5, precision_map_all=state["map"],
                candidates=[(case["block_m"], 64)], flat_lengths=[state["map"].numel()])
        b, _, t, d = state["q"].shape
        q, k, v = (x.transpose(1, 2).reshape(b * t, -1, d) for x in (state["q"], state["k"], state["v"]))
        cu = torch.arange(0, (b + 1) * t, t, device=q.device, dtype=torch.int32)
    elif kind == "attention":
        q, k, v, cu = state["q"], state["k"], state["v"], state["cu"]
    if kind == "attention":
        return tilemix_attention_with_quant(
            q, k, v, cu, cu, state["longest"], state["longest"], state["map"], block_m=case["block_m"], block_n=64,
            block_n_mask=state["mask_n"], BLKQ=128, BLKK=64, causal=case["causal"],
            scalar_scales=case["block_m"] == 128, routing_mode=case["mode"], int8_use_fp16_v=not case["int8_v"])[0]
    if kind == "quantize":
        names = ("q8", "q_scale", "cu_q", "k8", "k_scale", "cu_k", "v8", "v_scale", "cu_v")
        return dict(zip(names, quantize_qkv_for_tilemix(state["q"], state["k"], state["v"], state["cu"], state["cu"],
                                                        case["tokens"], case["tokens"])))
    if kind == "helpers":
        q, k = tilemix_llama.rotary_token_major(state["q"], state["k"], state["cos"], state["sin"])
        return {"norm": tilemix_llama.rms_norm(state["x"], state["weight"], 1e-5), "q": q, "k": k,
                "act": tilemix_llama.silu_mul(state["gate"], state["up"])}
    with torch.no_grad():
        if kind == "qwen":
            return state["module"](state["hidden"], position_embeddings=state["position_embeddings"])[0]
        cache = tilemix_llama.PrefillCache()
        out = state["model"](state["ids"], past_key_values=cache, use_cache=True, logits_to_keep=1)
        return {"logits": out.logits, "keys": [layer.keys for layer in cache.layers],
                "values": [layer.values for layer in cache.layers]}


# ---- what a pass cannot do without ---------------------------------------------


def _pairs(lengths, causal: bool) -> int:
    return sum(n * (n + 1) // 2 if causal else n * n for n in lengths)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "attention":
        lengths = _lengths(case)
        return {"bytes": 2 * sum(lengths) * case["dim"] * (2 * case["heads"] + 2 * case["kv_heads"]),
                "flops": 4 * case["dim"] * case["heads"] * _pairs(lengths, case["causal"])}
    if kind == "quantize":
        return {"bytes": 3 * case["tokens"] * case["dim"] * (case["heads"] + 2 * case["kv_heads"]),
                "flops": 4 * case["tokens"] * case["dim"] * (case["heads"] + 2 * case["kv_heads"])}
    if kind == "helpers":
        rope = (case["heads"] + case["kv_heads"]) * case["dim"]
        values = 2 * case["hidden"] + 2 * rope + 2 * case["dim"] + 3 * case["inner"]
        return {"bytes": 2 * case["tokens"] * values,
                "flops": case["tokens"] * (4 * case["hidden"] + 3 * rope + 6 * case["inner"])}
    hidden, kv = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
    tokens = case["seqs"] * case["length"]
    weights = hidden * (2 * hidden + 2 * kv)
    attention = 4 * hidden * _pairs([case["length"]] * case["seqs"], True)
    if kind == "qwen":
        return {"bytes": 2 * (weights + 2 * tokens * hidden), "flops": 2 * tokens * weights + attention}
    weights += 3 * hidden * case["inner"]
    head = case["vocab"] * hidden
    return {"bytes": 2 * (case["layers"] * (weights + 2 * tokens * kv) + head),
            "flops": case["layers"] * (2 * tokens * weights + attention) + 2 * case["seqs"] * head}


def tolerance(case: dict):
    # About four times the measured distance from the 64-bit results: fp16 scores,
    # probabilities and outputs (5e-4 to 6e-4; 3.5e-3 to 3.9e-3 with the outlier channels, whose
    # peaked softmax magnifies the rounding of a score), fp16 scales and elementwise outputs
    # (3e-4), an attention module (1.6e-3 to 2.6e-3), two layers of a model (8e-3).  Codes and
    # cu_seqlens are whole numbers and stay the same.
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 1.5e-2 if case["outliers"] else 2.5e-3}
    return {"rel": {"quantize": 1e-3, "helpers": 1.2e-3, "qwen": 1e-2, "llama": 3e-2}[kind]}


# ---- the same results in 64 bits -------------------------------------------------


def _int8_codes(x: torch.Tensor, block: int):
    """One sequence [tokens, heads, dim]: per-block symmetric codes and fp16 scales, as 64-bit values
    [tokens, heads, dim] and [tokens, heads, 1].  The codes and scales are part of what the call
    computes (the fp32 formula decides them); everything after them is evaluated in 64 bits."""
    n = x.shape[0]
    pad = -n % block
    x32 = nn.functional.pad(x.float(), (0, 0, 0, 0, 0, pad)).unflatten(0, (-1, block))
    scale = x32.abs().amax(dim=(1, 3), keepdim=True) / 127.0
    t = x32 / scale
    codes = torch.trunc(t + torch.where(t >= 0, 0.5, -0.5)).nan_to_num_(0.0)
    scale = scale.half().double().expand(-1, block, -1, 1)
    return codes.double().flatten(0, 1)[:n], scale.flatten(0, 1)[:n]


def _exact_sequence(q, k, v, rows: torch.Tensor, *, block_m, mask_n, causal, mode, int8_v) -> torch.Tensor:
    """One sequence, token-major [tokens, heads, dim] in any float type; rows: its routing rows,
    KV head by KV head.  Returns 64-bit outputs."""
    n, heads, dim = q.shape
    kv_heads = k.shape[1]
    group, m_blocks = heads // kv_heads, -(-n // block_m)
    groups = -(-n // mask_n)
    bits = torch.tensor([[(int(r) >> g) & 1 for g in range(groups)] for r in rows[:kv_heads * m_blocks].tolist()],
                        dtype=torch.bool, device=DEVICE).view(kv_heads, m_blocks, groups)
    if mode in ("fp16", "int8"):
        bits = torch.full_like(bits, mode == "int8")
    (qc, qs), (kc, ks), (vc, vs) = _int8_codes(q, 128), _int8_codes(k, 64), _int8_codes(v, 64)
    q, k, v = q.double(), k.double(), v.double()
    qq, kq, vq = qc * qs, kc * ks, vc * vs if int8_v else v
    out = torch.empty_like(q)
    keys = torch.arange(n, device=DEVICE)
    step = max(128, min(n, (1 << 27) // n // 128 * 128))
    for h in range(heads):
        g = h // group
        for r0 in range(0, n, step):
            r1 = min(n, r0 + step)
            m1 = r1 if causal else n
            routed = bits[g][torch.arange(r0, r1, device=DEVICE) // block_m][:, keys[:m1] // mask_n]
            score = torch.where(routed, qq[r0:r1, h] @ kq[:m1, g].T, q[r0:r1, h] @ k[:m1, g].T) * dim ** -0.5
            if causal:
                score.masked_fill_(keys[None, :m1] > keys[r0:r1, None], -math.inf)
            p = torch.softmax(score, dim=-1)
            del score
            if int8_v:
                out[r0:r1, h] = p.masked_fill(~routed, 0.0) @ vq[:m1, g] + p.masked_fill(routed, 0.0) @ v[:m1, g]
            else:
                out[r0:r1, h] = p @ v[:m1, g]
    return out


def _exact_attention(q, k, v, lengths, rows, **kw) -> torch.Tensor:
    out, at = [], 0
    for n in lengths:
        out.append(_exact_sequence(q[at:at + n], k[at:at + n], v[at:at + n], rows, **kw))
        at += n
    return torch.cat(out)


def _rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """[..., tokens, heads, dim] with [tokens, dim] tables."""
    half = x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos[:, None] + turned * sin[:, None]


def _rms(x, weight, eps: float):
    return weight * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _exact_module(x, module, cos, sin, case: dict):
    """A TileMix attention module on 64-bit hidden states [seqs, tokens, hidden]: (output, k, v)."""
    b, t, _ = x.shape

    def project(layer):
        y = x @ layer.weight.double().T
        return (y if layer.bias is None else y + layer.bias.double()).view(b, t, -1, case["dim"])

    q, k, v = project(module.q_proj), project(module.k_proj), project(module.v_proj)
    q, k = _rope(q, cos, sin), _rope(k, cos, sin)
    block = module._get_block_config(t)
    mask_n = pick_mask_block_n(t, block.block_n)
    rows = _map_row(t, block.block_m, mask_n, "sptrans", 0.5).repeat(case["kv_heads"])
    out = _exact_attention(q.flatten(0, 1), k.flatten(0, 1), v.flatten(0, 1), [t] * b, rows, block_m=block.block_m,
                           mask_n=mask_n, causal=True, mode="mixed", int8_v=False)
    return out.reshape(b, t, -1) @ module.o_proj.weight.double().T, k.transpose(1, 2), v.transpose(1, 2)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "attention":
        _, mask_n, rows = _routing(case)
        lengths = _lengths(case)
        out = _exact_attention(*_attention_inputs(case, seed), lengths, rows, block_m=case["block_m"], mask_n=mask_n,
                               causal=case["causal"], mode=case["mode"], int8_v=case["int8_v"])
        if case["entry"] == "dense" and case["mode"] == "mixed":
            return out.view(case["seqs"], case["length"], case["heads"], case["dim"]).transpose(1, 2)
        return out
    if kind == "quantize":
        state = prepare(case, seed)
        scales = {}
        for name, block in (("q", 128), ("k", 64), ("v", 64)):
            x = nn.functional.pad(state[name].double(), (0, 0, 0, 0, 0, -case["tokens"] % block))
            scales[name] = x.unflatten(0, (-1, block)).abs().amax(dim=(1, 3)) / 127.0
        return {"q8": None, "q_scale": scales["q"], "cu_q": None, "k8": None, "k_scale": scales["k"], "cu_k": None,
                "v8": None, "v_scale": scales["v"], "cu_v": None}
    if kind == "helpers":
        s = {name: t.double() for name, t in _helper_inputs(case, seed).items()}
        q, k = (_rope(s[n].transpose(1, 2), s["cos"][0], s["sin"][0]).transpose(1, 2) for n in ("q", "k"))
        return {"norm": _rms(s["x"], s["weight"], 1e-5), "q": q, "k": k,
                "act": nn.functional.silu(s["gate"]) * s["up"]}
    if kind == "qwen":
        state = prepare(case, seed)
        cos, sin = (t[0].double() for t in state["position_embeddings"])
        return _exact_module(state["hidden"].double(), state["module"], cos, sin, case)[0]
    model, ids = _llama_model(case, seed), _token_ids(case, seed)
    table = model.model.embed_tokens.weight.double()
    x = table[ids]
    cos, sin = (t[0].double() for t in model.model.rotary_emb(x[:1].half(), torch.arange(ids.shape[1],
                                                                                         device=DEVICE)[None]))
    keys, values = [], []
    for layer in model.model.layers:
        out, k, v = _exact_module(_rms(x, layer.input_layernorm.weight.double(), 1e-5), layer.self_attn, cos, sin,
                                  case)
        x = x + out
        y = _rms(x, layer.post_attention_layernorm.weight.double(), 1e-5)
        gate, up = y @ layer.mlp.gate_proj.weight.double().T, y @ layer.mlp.up_proj.weight.double().T
        x = x + (nn.functional.silu(gate) * up) @ layer.mlp.down_proj.weight.double().T
        keys.append(k)
        values.append(v)
    return {"logits": _rms(x[:, -1:], model.model.norm.weight.double(), 1e-5) @ table.T, "keys": keys,
            "values": values}
