"""The work a serving program has this framework do, layer by layer, as cases that can be timed and checked.

Families, each through the entry point that a layer of the hybrid model calls:

* ``decode``          one token per sequence of a full-attention layer over its paged K/V
* ``prefill``         a prompt, or a chunk of one, of a full-attention layer, with the output gate
* ``prologue``        the step before either: q/k RMSNorm, partial rotary embedding, K/V append
* ``linear_step``     one token per sequence of a linear-attention layer (conv, recurrence, output norm)
* ``linear_prefill``  a prompt, or a chunk of one, of a linear-attention layer, with its output norm
* ``projection``      the fp8 block-scaled projections around all of them

Shapes are those of ``bench.py`` and of the tests: 16 query heads on 2 KV heads of 256 (or heads of 128), 16-token
blocks, 16 key heads and 32 value heads of 128, a hidden size of 2048.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qwen3.6-2080ti_amd"))

import attention_runtime
import hip_ops
from decode_state import LinearStatePool

DEVICE = "cuda:0"
BLOCK = 16
EPS = 1e-6
THETA = 10_000_000.0
ROTARY = 0.25


def listed() -> list[dict]:
    return [
        # The smallest call of a chat server: four short conversations, one token each.
        _decode("decode_few", batch=4, lo=512, hi=512),
        # A full decode batch under continuous batching: 64 conversations of 1k to 32k tokens.
        _decode("decode_batch", batch=64, lo=1024, hi=32768),
        # Fresh prompts of a few words up to a page, packed into one ragged step with nothing cached.
        _prefill("prefill_prompts", batch=5, new_lo=37, new_hi=700, prefix_lo=0, prefix_hi=0),
        # Chunked prefill in steady state: eight requests, 512 new tokens each, behind up to 8k cached ones.
        _prefill("prefill_chunk", batch=8, new_lo=512, new_hi=512, prefix_lo=0, prefix_hi=8192),
        # The norm, rotary and append launch of that same chunk.
        _prologue("prologue_chunk", batch=8, new_lo=512, new_hi=512, prefix_lo=0, prefix_hi=8192),
        # The linear-attention layers' token of the small chat server ...
        _linear_step("linear_step_few", batch=3),
        # ... and of a full decode batch.
        _linear_step("linear_step_batch", batch=128),
        # One long prompt alone on the GPU, continuing a carried state; its length is not a whole number of chunks.
        _linear_prefill("linear_prefill_one", batch=1, seq=6001, carried=True),
        # Four 8k prompts in one step, from empty states.
        _linear_prefill("linear_prefill_batch", batch=4, seq=8192, carried=False),
        # out_proj for a handful of decoding sequences, the weight packed once at load.
        _projection("projection_few", rows=5, out_features=2048, in_features=4096, packed=True),
        # q_proj with its gate half for a full decode batch, the weight as the checkpoint holds it.
        _projection("projection_batch", rows=128, out_features=8192, in_features=2048, packed=False),
        # in_proj_qkv over the 4096 new tokens of a prefill chunk.
        _projection("projection_chunk", rows=4096, out_features=8192, in_features=2048, packed=True),
    ]


def draw(rng: random.Random) -> dict:
    family = rng.choice(("decode", "prefill", "prologue", "linear_step", "linear_prefill", "projection"))
    if family == "decode":
        heads, kv_heads, dim = rng.choice(((16, 2, 256), (16, 2, 256), (8, 2, 128), (16, 1, 128)))
        batch = _log_int(rng, 1, 64)
        hi = _log_int(rng, 17, 32768)
        return _decode(None, batch=batch, lo=_log_int(rng, 1, hi), hi=hi, heads=heads, kv_heads=kv_heads, dim=dim,
                       index=rng.choice(("int32", "int64")))
    if family in ("prefill", "prologue"):
        heads, kv_heads, dim = rng.choice(((16, 2, 256), (16, 2, 256), (8, 2, 128), (4, 4, 256)))
        tokens = _log_int(rng, 24, 4096)  # new tokens of the step
        batch = rng.randint(1, max(1, min(8, tokens // 24)))
        new_hi = max(1, tokens // batch)
        prefix_hi = rng.choice((0, _log_int(rng, 16, 8192)))
        make = _prefill if family == "prefill" else _prologue
        return make(None, batch=batch, new_lo=rng.randint(max(1, new_hi // 4), new_hi), new_hi=new_hi, prefix_lo=prefix_hi // 3, prefix_hi=prefix_hi,
                    heads=heads, kv_heads=kv_heads, dim=dim, index=rng.choice(("int32", "int64")))
    if family == "linear_step":
        key_heads, value_heads = rng.choice(((16, 32), (16, 32), (16, 16), (8, 32)))
        return _linear_step(None, batch=_log_int(rng, 1, 128), key_heads=key_heads, value_heads=value_heads, normed=rng.random() < 0.8)
    if family == "linear_prefill":
        key_heads, value_heads = rng.choice(((16, 32), (16, 32), (16, 16), (8, 32)))
        batch = rng.choice((1, 1, 2, 3, 4))
        return _linear_prefill(None, batch=batch, seq=_log_int(rng, 40, 8192), carried=rng.random() < 0.5, key_heads=key_heads, value_heads=value_heads)
    out_features, in_features = rng.choice(((8192, 2048), (4096, 2048), (2048, 4096), (512, 2048)))
    return _projection(None, rows=_log_int(rng, 1, 4096), out_features=out_features, in_features=in_features, packed=rng.random() < 0.6,
                       dtype=rng.choice(("float32", "float32", "bfloat16")))


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _case(name, family, **values) -> dict:
    case = {"family": family, **values}
    if name is not None:
        case["name"] = name
    return case


def _decode(name, *, batch, lo, hi, heads=16, kv_heads=2, dim=256, index="int32"):
    return _case(name, "decode", batch=batch, lo=lo, hi=hi, heads=heads, kv_heads=kv_heads, dim=dim, index=index)


def _prefill(name, *, batch, new_lo, new_hi, prefix_lo, prefix_hi, heads=16, kv_heads=2, dim=256, index="int32"):
    return _case(name, "prefill", batch=batch, new_lo=new_lo, new_hi=new_hi, prefix_lo=prefix_lo, prefix_hi=prefix_hi, heads=heads,
                 kv_heads=kv_heads, dim=dim, index=index)


def _prologue(name, **values):
    return {**_prefill(name, **values), "family": "prologue"}


def _linear_step(name, *, batch, key_heads=16, value_heads=32, normed=True):
    return _case(name, "linear_step", batch=batch, key_heads=key_heads, value_heads=value_heads, normed=normed)


def _linear_prefill(name, *, batch, seq, carried, key_heads=16, value_heads=32):
    return _case(name, "linear_prefill", batch=batch, seq=seq, carried=carried, key_heads=key_heads, value_heads=value_heads)


def _projection(name, *, rows, out_features, in_features, packed, dtype="float32"):
    return _case(name, "projection", rows=rows, out_features=out_features, in_features=in_features, packed=packed, dtype=dtype)


# --------------------------------------------------------------------------- inputs


def prepare(case: dict, seed: int):
    return {"case": case, **_INPUTS[case["family"]](case, seed)}


def run(state):
    return _RUN[state["case"]["family"]](state)


def work(case: dict) -> dict:
    return _WORK[case["family"]](case)


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    return _EXACT[case["family"]](state)


def tolerance(case: dict) -> dict:
    # About four times the relative 2-norm error against 64 bits measured on an MI355X: the bf16 results 1.6e-3 to
    # 2.9e-3 (one or two bf16 roundings), an fp32 projection of fewer than 16 rows 2.5e-6 (activations as a bf16
    # pair), of more 2.1e-4 (activations as fp16).
    if case["family"] == "projection" and case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 5e-4} if case["rows"] < 16 else {"rel": 1e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.1}


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=dtype)


def _index_dtype(case):
    return torch.int32 if case["index"] == "int32" else torch.int64


def _lengths(case: dict, what: str, lo: int, hi: int) -> list[int]:
    """Row lengths of a case: part of its shape, so they do not change with the inputs' seed."""
    rng = random.Random(f"{what} {lo} {hi} {case['batch']}")
    return [rng.randint(lo, hi) for _ in range(case["batch"])]


def _paged(case: dict, totals: list[int], gen):
    """Block tables (-1 padded) over a pool with a quarter of its blocks free, blocks in random order."""
    need = [(n + BLOCK - 1) // BLOCK for n in totals]
    blocks = math.ceil(sum(need) * 1.25)
    order = torch.randperm(blocks, generator=gen, device=DEVICE)
    tables = torch.full((len(need), max(need)), -1, dtype=_index_dtype(case), device=DEVICE)
    at = 0
    for row, n in enumerate(need):
        tables[row, :n] = order[at : at + n]
        at += n
    pools = [_randn(gen, blocks, case["kv_heads"], BLOCK, case["dim"]) for _ in range(2)]
    return tables, pools[0], pools[1]


def _decode_inputs(case, seed):
    gen = _generator(seed)
    lens = _lengths(case, "context", case["lo"], case["hi"])
    tables, keys, values = _paged(case, lens, gen)
    query = _randn(gen, case["batch"], case["heads"], 1, case["dim"])
    return {"query": query, "tables": tables, "keys": keys, "values": values, "lens": torch.tensor(lens, dtype=_index_dtype(case), device=DEVICE)}


def _new_tokens(case):
    return _lengths(case, "new", case["new_lo"], case["new_hi"]), _lengths(case, "prefix", case["prefix_lo"], case["prefix_hi"])


def _prefill_inputs(case, seed):
    gen = _generator(seed)
    new, prefix = _new_tokens(case)
    tables, keys, values = _paged(case, [n + p for n, p in zip(new, prefix)], gen)
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    idt = _index_dtype(case)
    heads, dim = case["heads"], case["dim"]
    return {"query": _randn(gen, cu[-1], heads, dim), "gate": _randn(gen, cu[-1], heads * dim), "tables": tables, "keys": keys, "values": values,
            "cu": torch.tensor(cu, dtype=idt, device=DEVICE), "prefix": torch.tensor(prefix, dtype=idt, device=DEVICE), "max_new": max(new)}


def _prologue_inputs(case, seed):
    state = _prefill_inputs(case, seed)
    gen = _generator(seed + 1)
    tokens, heads, kv_heads, dim = state["query"].shape[0], case["heads"], case["kv_heads"], case["dim"]
    state["q_proj"] = _randn(gen, tokens, heads * 2 * dim)
    state["k_proj"] = _randn(gen, tokens, kv_heads * dim)
    state["v_proj"] = _randn(gen, tokens, kv_heads * dim)
    state["q_norm"] = 0.1 * _randn(gen, dim)
    state["k_norm"] = 0.1 * _randn(gen, dim)
    return state


def _linear_weights(case, gen):
    channels = (2 * case["key_heads"] + case["value_heads"]) * 128
    # heads that forget within a token up to heads that remember some hundred tokens
    a_log = torch.linspace(math.log(1 / 64), 0.0, case["value_heads"], device=DEVICE)
    dt_bias = 0.1 * _randn(gen, case["value_heads"], dtype=torch.float32)
    conv_w = 0.5 * _randn(gen, channels, 4, dtype=torch.float32)
    return channels, a_log, dt_bias, conv_w


def _linear_config(case):
    return attention_runtime.parse_attention_config({"text_config": {
        "num_attention_heads": 16, "num_key_value_heads": 2, "head_dim": 256, "attn_output_gate": True, "native_paged_attention": True,
        "linear_num_key_heads": case["key_heads"], "linear_num_value_heads": case["value_heads"], "linear_key_head_dim": 128,
        "linear_value_head_dim": 128, "linear_conv_kernel_dim": 4}})


def _linear_step_inputs(case, seed):
    gen = _generator(seed)
    channels, a_log, dt_bias, conv_w = _linear_weights(case, gen)
    batch, value_heads = case["batch"], case["value_heads"]
    pool = LinearStatePool(batch + 2, value_heads, 128, 128, channels, 4, device=DEVICE)
    pool.state.normal_(0.0, 0.05, generator=gen)
    pool.conv.normal_(0.0, 1.0, generator=gen)
    slots = torch.randperm(batch + 2, generator=gen, device=DEVICE)[:batch].to(torch.int32)
    normed = case["normed"]
    return {"mixed": _randn(gen, batch, channels), "a": _randn(gen, batch, value_heads), "b": _randn(gen, batch, value_heads), "a_log": a_log,
            "dt_bias": dt_bias, "conv_w": conv_w, "pool": pool, "slots": slots, "z": _randn(gen, batch, value_heads * 128) if normed else None,
            "norm_w": (1 + 0.1 * _randn(gen, 128, dtype=torch.float32)).to(torch.bfloat16) if normed else None, "config": _linear_config(case)}


def _linear_prefill_inputs(case, seed):
    gen = _generator(seed)
    channels, a_log, dt_bias, conv_w = _linear_weights(case, gen)
    batch, seq, value_heads = case["batch"], case["seq"], case["value_heads"]
    carried = case["carried"]
    return {"mixed": _randn(gen, batch, seq, channels), "a": _randn(gen, batch, seq, value_heads), "b": _randn(gen, batch, seq, value_heads),
            "a_log": a_log, "dt_bias": dt_bias, "conv_w": conv_w, "z": _randn(gen, batch, seq, value_heads * 128),
            "norm_w": (1 + 0.1 * _randn(gen, 128, dtype=torch.float32)).to(torch.bfloat16), "config": _linear_config(case),
            "conv_state": _randn(gen, batch, channels, 3, dtype=torch.float32) if carried else None,
            "state": 0.05 * _randn(gen, batch, value_heads, 128, 128, dtype=torch.float32) if carried else None}


def _projection_inputs(case, seed):
    gen = _generator(seed)
    rows, n, k = case["rows"], case["out_features"], case["in_features"]
    # a checkpoint's weight: each 128 x 128 block scaled so that its largest element is the largest code
    dense = 0.02 * _randn(gen, n // 128, 128, k // 128, 128, dtype=torch.float32)
    scale = (dense.abs().amax(dim=(1, 3)) / 448.0).to(torch.bfloat16)
    codes = (dense / scale.float()[:, None, :, None]).clamp(-448.0, 448.0).reshape(n, k).to(torch.float8_e4m3fn)
    weight = hip_ops.fp8_pack_weight(codes) if case["packed"] else codes
    return {"x": _randn(gen, rows, k, dtype=getattr(torch, case["dtype"])), "codes": codes, "weight": weight, "scale": scale}


_INPUTS = {"decode": _decode_inputs, "prefill": _prefill_inputs, "prologue": _prologue_inputs, "linear_step": _linear_step_inputs,
           "linear_prefill": _linear_prefill_inputs, "projection": _projection_inputs}


# --------------------------------------------------------------------------- one pass


def _run_decode(s):
    return hip_ops.paged_attention_decode_batched(s["query"], s["tables"], s["keys"], s["values"], s["lens"], BLOCK)


def _run_prefill(s):
    return hip_ops.paged_attention_prefill(s["query"], s["cu"], s["prefix"], s["keys"], s["values"], s["tables"], BLOCK, max_new=s["max_new"],
                                           gate=s["gate"])


def _run_prologue(s):
    query, _gate = hip_ops.qk_norm_rope_kv_append(
        s["q_proj"], s["k_proj"], s["v_proj"], s["q_norm"], s["k_norm"], s["keys"], s["values"], s["tables"], s["cu"], s["prefix"], BLOCK,
        max_new=s["max_new"], eps=EPS, rope_theta=THETA, partial_rotary_factor=ROTARY)
    return query, s["keys"], s["values"]


def _run_linear_step(s):
    out = attention_runtime.linear_attention_decode_batch(s["mixed"], s["a"], s["b"], s["a_log"], s["dt_bias"], s["conv_w"], s["pool"], s["slots"],
                                                          s["config"], z=s["z"], norm_weight=s["norm_w"], eps=EPS)
    return out, s["pool"].state, s["pool"].conv


def _run_linear_prefill(s):
    return attention_runtime.linear_attention_prefill(s["mixed"], s["a"], s["b"], s["a_log"], s["dt_bias"], s["conv_w"], s["config"],
                                                      conv_state=s["conv_state"], initial_state=s["state"], z=s["z"], norm_weight=s["norm_w"], eps=EPS)


def _run_projection(s):
    return hip_ops.fp8_e4m3_bf16_linear(s["x"], s["weight"], s["scale"], out_dtype=s["x"].dtype)


_RUN = {"decode": _run_decode, "prefill": _run_prefill, "prologue": _run_prologue, "linear_step": _run_linear_step,
        "linear_prefill": _run_linear_prefill, "projection": _run_projection}


# --------------------------------------------------------------------------- what a pass cannot do without


def _work_decode(case):
    lens = _lengths(case, "context", case["lo"], case["hi"])
    row = case["heads"] * case["dim"]
    return {"bytes": sum(lens) * case["kv_heads"] * case["dim"] * 4 + 2 * case["batch"] * row * 2, "flops": 4 * row * sum(lens)}


def _work_prefill(case):
    new, prefix = _new_tokens(case)
    row = case["heads"] * case["dim"]
    keys = sum(n + p for n, p in zip(new, prefix))
    return {"bytes": keys * case["kv_heads"] * case["dim"] * 4 + 3 * sum(new) * row * 2,
            "flops": sum(4 * row * (n * p + n * (n + 1) // 2) for n, p in zip(new, prefix))}


def _work_prologue(case):
    tokens = sum(_new_tokens(case)[0])
    return {"bytes": 2 * tokens * case["dim"] * (case["heads"] + 2 * case["kv_heads"]) * 2, "flops": 0}


def _work_linear_step(case):
    heads = case["value_heads"]
    channels = (2 * case["key_heads"] + heads) * 128
    per_row = 2 * heads * 128 * 128 * 4 + 2 * channels * 3 * 4 + channels * 2 + heads * 128 * (4 if case["normed"] else 2)
    return {"bytes": case["batch"] * per_row, "flops": case["batch"] * heads * 128 * 128 * 7}


def _work_linear_prefill(case):
    tokens, heads = case["batch"] * case["seq"], case["value_heads"]
    channels = (2 * case["key_heads"] + heads) * 128
    states = case["batch"] * (heads * 128 * 128 * 4 + channels * 3 * 4) * (2 if case["carried"] else 1)
    # per 64-token chunk and value head: 2 C^2 (3 dk + 2 dv) + 6 C dk dv + C^3 / 3
    per_chunk = 2 * 64 * 64 * (3 * 128 + 2 * 128) + 6 * 64 * 128 * 128 + 64**3 // 3
    return {"bytes": tokens * (channels * 2 + heads * 4 + 2 * heads * 128 * 2) + states, "flops": per_chunk * heads * tokens // 64}


def _work_projection(case):
    rows, n, k = case["rows"], case["out_features"], case["in_features"]
    size = 4 if case["dtype"] == "float32" else 2
    return {"bytes": n * k + n * k // 8192 + rows * (n + k) * size, "flops": 2 * rows * n * k}


_WORK = {"decode": _work_decode, "prefill": _work_prefill, "prologue": _work_prologue, "linear_step": _work_linear_step,
         "linear_prefill": _work_linear_prefill, "projection": _work_projection}


# --------------------------------------------------------------------------- the same in 64 bits


def _row_kv(s, row, length):
    """Keys and values (kv_heads, length, dim) of a row, in 64 bits."""
    need = (length + BLOCK - 1) // BLOCK
    ids = s["tables"][row, :need].long()
    both = []
    for pool in (s["keys"], s["values"]):
        blocks = pool.index_select(0, ids).double()
        both.append(blocks.transpose(0, 1).reshape(pool.shape[1], need * BLOCK, pool.shape[3])[:, :length].contiguous())
    return both


def _exact_decode(s):
    case = s["case"]
    out = torch.zeros(s["query"].shape, dtype=torch.float64, device=DEVICE)
    group = case["heads"] // case["kv_heads"]
    for row, length in enumerate(s["lens"].tolist()):
        keys, values = _row_kv(s, row, length)
        for g in range(case["kv_heads"]):
            q = s["query"][row, g * group : (g + 1) * group, 0].double()
            out[row, g * group : (g + 1) * group, 0] = torch.softmax(q @ keys[g].T / math.sqrt(case["dim"]), dim=-1) @ values[g]
    return out


def _exact_prefill(s):
    case = s["case"]
    heads, dim = case["heads"], case["dim"]
    out = torch.zeros(s["query"].shape, dtype=torch.float64, device=DEVICE)
    cu, prefix = s["cu"].tolist(), s["prefix"].tolist()
    group = heads // case["kv_heads"]
    for row, p in enumerate(prefix):
        lo, hi = cu[row], cu[row + 1]
        keys, values = _row_kv(s, row, p + hi - lo)
        hidden = torch.arange(p + hi - lo, device=DEVICE)[None] > p + torch.arange(hi - lo, device=DEVICE)[:, None]
        for h in range(heads):
            scores = (s["query"][lo:hi, h].double() @ keys[h // group].T / math.sqrt(dim)).masked_fill(hidden, -math.inf)
            out[lo:hi, h] = torch.softmax(scores, dim=-1) @ values[h // group]
    return out * torch.sigmoid(s["gate"].double()).view(out.shape)


def _exact_norm_rope(x, weight, positions):
    """RMSNorm with the (1 + w) weight, then rotation of the first quarter of each head; x (tokens, heads, dim)."""
    y = x.double()
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * (1 + weight.double())
    half = int(x.shape[-1] * ROTARY) // 2
    angle = positions.double()[:, None] * THETA ** (-torch.arange(half, device=DEVICE, dtype=torch.float64) / half)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = y[..., :half].clone(), y[..., half : 2 * half].clone()
    y[..., :half] = a * cos - b * sin
    y[..., half : 2 * half] = b * cos + a * sin
    return y


def _exact_prologue(s):
    case = s["case"]
    tokens, heads, kv_heads, dim = s["query"].shape[0], case["heads"], case["kv_heads"], case["dim"]
    cu, prefix = s["cu"].tolist(), s["prefix"].tolist()
    positions = torch.cat([p + torch.arange(cu[r + 1] - cu[r], device=DEVICE) for r, p in enumerate(prefix)])
    rows = torch.cat([torch.full((cu[r + 1] - cu[r],), r, device=DEVICE) for r in range(len(prefix))])
    query = _exact_norm_rope(s["q_proj"].view(tokens, heads, 2 * dim)[..., :dim], s["q_norm"], positions)
    keys, values = s["keys"].double(), s["values"].double()
    block = s["tables"].long()[rows, positions // BLOCK]
    keys[block, :, positions % BLOCK] = _exact_norm_rope(s["k_proj"].view(tokens, kv_heads, dim), s["k_norm"], positions)
    values[block, :, positions % BLOCK] = s["v_proj"].view(tokens, kv_heads, dim).double()
    return query, keys, values


def _exact_conv(s, mixed, conv_state):
    """Causal conv and SiLU over (batch, seq, channels), and the last three inputs."""
    padded = torch.cat((conv_state.double().transpose(1, 2), mixed.double()), dim=1)
    seq, taps = mixed.shape[1], s["conv_w"].double()
    out = sum(taps[:, i] * padded[:, i : i + seq] for i in range(4))
    return torch.nn.functional.silu(out), padded[:, -3:].transpose(1, 2)


def _exact_heads(s, act):
    """q, k (normalised, one per value head), v as (batch, heads, seq, 128); g, beta as (batch, heads, seq)."""
    case = s["case"]
    key_heads, heads = case["key_heads"], case["value_heads"]
    batch, seq = act.shape[:2]
    q, k, v = torch.split(act, [key_heads * 128, key_heads * 128, heads * 128], dim=-1)
    unit = lambda x: x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k = (unit(x.reshape(batch, seq, key_heads, 128)).repeat_interleave(heads // key_heads, dim=2).transpose(1, 2) for x in (q, k))
    v = v.reshape(batch, seq, heads, 128).transpose(1, 2)
    g = -s["a_log"].double().exp() * torch.nn.functional.softplus(s["a"].double().reshape(batch, seq, heads) + s["dt_bias"].double())
    beta = torch.sigmoid(s["b"].double().reshape(batch, seq, heads))
    return q / math.sqrt(128), k, v, g.transpose(1, 2), beta.transpose(1, 2)


def _exact_gated_norm(s, core, z):
    """core (..., heads, 128)"""
    n = core * torch.rsqrt(core.square().mean(-1, keepdim=True) + EPS) * s["norm_w"].double()
    return n * torch.nn.functional.silu(z.double().view(core.shape))


def _exact_linear_step(s):
    slots = s["slots"].long()
    state, conv = s["pool"].state.double(), s["pool"].conv.double()
    act, tail = _exact_conv(s, s["mixed"][:, None], conv[slots])
    q, k, v, g, beta = (x[:, :, 0] for x in _exact_heads(s, act))
    old = state[slots] * g.exp()[..., None, None]
    delta = (v - (old * k[..., None]).sum(-2)) * beta[..., None]
    new = old + k[..., None] * delta[..., None, :]
    core = (new * q[..., None]).sum(-2)
    state[slots], conv[slots] = new, tail
    return (core if s["z"] is None else _exact_gated_norm(s, core, s["z"])), state, conv


def _exact_linear_prefill(s):
    case = s["case"]
    batch, seq, heads = case["batch"], case["seq"], case["value_heads"]
    channels = s["mixed"].shape[-1]
    conv = s["conv_state"] if case["carried"] else torch.zeros(batch, channels, 3, device=DEVICE)
    act, tail = _exact_conv(s, s["mixed"], conv)
    q, k, v, g, beta = _exact_heads(s, act)
    del act
    state = s["state"].double().clone() if case["carried"] else torch.zeros(batch, heads, 128, 128, dtype=torch.float64, device=DEVICE)
    core = torch.empty(batch, heads, seq, 128, dtype=torch.float64, device=DEVICE)
    for lo in range(0, seq, 64):
        at = slice(lo, min(seq, lo + 64))
        qc, kc, vc, bc, total = q[:, :, at], k[:, :, at], v[:, :, at], beta[:, :, at], g[:, :, at].cumsum(-1)
        n = qc.shape[2]
        decay = (total[..., :, None] - total[..., None, :]).masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEVICE).triu(1), -math.inf).exp()
        kt = kc.transpose(-1, -2).contiguous()
        system = (bc[..., None] * decay * (kc @ kt)).tril(-1) + torch.eye(n, dtype=torch.float64, device=DEVICE)
        rhs = bc[..., None] * (vc - total.exp()[..., None] * (kc @ state))
        delta = torch.linalg.solve_triangular(system, rhs, upper=False, unitriangular=True)
        core[:, :, at] = total.exp()[..., None] * (qc @ state) + (decay * (qc @ kt)) @ delta
        state = total[..., -1].exp()[..., None, None] * state + kt @ ((total[..., -1:] - total).exp()[..., None] * delta)
    return _exact_gated_norm(s, core.transpose(1, 2), s["z"]).reshape(batch, seq, heads * 128), state, tail


def _exact_projection(s):
    n, k = s["codes"].shape
    weight = s["codes"].to(torch.float64).view(n // 128, 128, k // 128, 128) * s["scale"].double()[:, None, :, None]
    return s["x"].double() @ weight.view(n, k).T


_EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "prologue": _exact_prologue, "linear_step": _exact_linear_step,
          "linear_prefill": _exact_linear_prefill, "projection": _exact_projection}
