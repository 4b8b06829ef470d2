"""Gate layouts of paged prefill: 8-byte loads where every head's gate row is aligned, element loads elsewhere.

Both read the same bits, so the outputs are equal bit for bit; the contiguous one is held to the oracle
(bf16 outputs, ``atol = rtol = 2e-2``).
"""

from __future__ import annotations

import pytest
import torch

from oracle import attention as oracle_attn

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("heads, kv_heads, dim", [(16, 2, 256), (8, 2, 128)])
@pytest.mark.parametrize("new", [1, 17, 33])
def test_gate_layouts_agree(heads, kv_heads, dim, new) -> None:
    import hip_ops

    gen = torch.Generator().manual_seed(new + dim)
    prefix, blocks = 21, 8
    randn = lambda *shape: torch.randn(shape, generator=gen).to(torch.bfloat16)  # noqa: E731
    keys, values = randn(blocks, kv_heads, 16, dim), randn(blocks, kv_heads, 16, dim)
    query, gate = randn(new, heads, dim), randn(new, heads * dim)
    order = torch.randperm(blocks, generator=gen)[: (prefix + new + 15) // 16]
    flat = torch.zeros(new * heads * dim + 1, dtype=torch.bfloat16, device=DEV)
    flat[1:] = gate.to(DEV).view(-1)
    half = torch.zeros(new, heads, 2 * dim, dtype=torch.bfloat16, device=DEV)
    half[..., dim:] = gate.to(DEV).view(new, heads, dim)
    odd = torch.zeros(new, heads, dim + 1, dtype=torch.bfloat16, device=DEV)
    odd[..., :dim] = gate.to(DEV).view(new, heads, dim)
    layouts = {"contiguous": gate.to(DEV), "misaligned base": flat[1:].view(new, heads * dim), "half of q_proj": half[..., dim:],
               "odd head stride": odd[..., :dim]}
    out = {}
    for name, g in layouts.items():
        out[name] = hip_ops.paged_attention_prefill(
            query.to(DEV), torch.tensor([0, new], device=DEV, dtype=torch.int32), torch.tensor([prefix], device=DEV, dtype=torch.int32),
            keys.to(DEV), values.to(DEV), order.to(torch.int32)[None].to(DEV), 16, max_new=new, gate=g).cpu()
        assert torch.equal(out[name], out["contiguous"]), name
    want = oracle_attn.paged_prefill(query, keys, values, [order.tolist()], [prefix], [new], block_size=16, gate=gate)
    torch.testing.assert_close(out["contiguous"].float(), torch.cat(want).float(), atol=2e-2, rtol=2e-2)
