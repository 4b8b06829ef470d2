"""Batched decode with tables wider than the contexts against the CPU oracle.

Tolerance for bf16 outputs as in the other decode tests: ``atol = rtol = 2e-2``.
"""

from __future__ import annotations

import pytest
import torch

from oracle import attention as oracle_attn

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _case(lens, heads, kv_heads, dim, width, index, seed):
    gen = torch.Generator().manual_seed(seed)
    need = [(max(n, 0) + 15) // 16 for n in lens]
    blocks = sum(need) + 3
    keys = torch.randn(blocks, kv_heads, 16, dim, generator=gen).to(torch.bfloat16)
    values = torch.randn(blocks, kv_heads, 16, dim, generator=gen).to(torch.bfloat16)
    query = torch.randn(len(lens), heads, 1, dim, generator=gen).to(torch.bfloat16)
    order = torch.randperm(blocks, generator=gen).tolist()
    tables = torch.full((len(lens), max(width, max(need), 1)), -1, dtype=index)
    rows, at = [], 0
    for r, n in enumerate(need):
        rows.append(order[at : at + n])
        tables[r, :n] = torch.tensor(rows[-1], dtype=index)
        at += n
    return query, keys, values, tables, rows


@pytest.mark.parametrize(
    "lens, heads, kv_heads, dim, width, index",
    [
        ([40], 16, 2, 256, 2048, torch.int32),  # table far wider than the context: most launched waves idle
        ([5, 0, 33, 1], 16, 2, 256, 512, torch.int32),  # the same with an empty row, workgroup merge
        ([0, 0], 8, 2, 128, 64, torch.int32),  # nothing to attend to at all
    ],
)
def test_few_rows_match_oracle(lens, heads, kv_heads, dim, width, index) -> None:
    import hip_ops

    query, keys, values, tables, rows = _case(lens, heads, kv_heads, dim, width, index, seed=len(lens) + dim)
    live = [r for r, n in enumerate(lens) if n > 0]
    want = torch.zeros(query.shape)
    if live:
        want[live] = oracle_attn.paged_decode(query[live], [keys] * len(live), [values] * len(live), [rows[r] for r in live],
                                              [lens[r] for r in live], block_size=16, pool_layout="phbd").float()
    args = [t.to(DEV) for t in (query, tables, keys, values, torch.tensor(lens, dtype=index))]
    for _ in range(2):
        # what the workspace held before must not show: freed memory full of NaN is what torch hands out next
        dirty = [torch.full((size,), float("nan"), device=DEV) for size in (1 << 16, 1 << 20, 5 << 20, 20 << 20)]
        del dirty
        out = hip_ops.paged_attention_decode_batched(*args, 16)
        torch.testing.assert_close(out.cpu().float(), want, atol=2e-2, rtol=2e-2)
