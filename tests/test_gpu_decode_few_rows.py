"""Batched decode with few row groups against the CPU oracle: short chains, both merges, tables wider than the contexts.

For up to 64 row groups the launch has a wave for every two tiles of the full tables, up to 1024 waves and at most 512 a
row group (16 where there are more than 16 row groups); for more a wave for every eight.  With fewer tiles than waves
each tile has a wave.  The merge takes a workgroup per head from a mean of 32 launched waves a row group, which shares
the columns of up to 64 partials and the partials themselves above.  Tolerance for bf16 outputs as in the other decode
tests: ``atol = rtol = 2e-2``.
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
        ([1], 16, 2, 256, 1, torch.int32),  # one tile, one wave per row group
        ([17], 16, 1, 128, 2, torch.int64),
        ([40], 16, 2, 256, 2048, torch.int32),  # table far wider than the context: most launched waves idle
        ([5, 0, 33, 1], 16, 2, 256, 512, torch.int32),  # the same with an empty row, workgroup merge
        ([0, 0], 8, 2, 128, 64, torch.int32),  # nothing to attend to at all
        ([512] * 4, 16, 2, 256, 0, torch.int32),  # 16 partials a row group: wave merge
        ([1023], 16, 2, 256, 0, torch.int32),  # 32 partials: workgroup merge
        ([8191], 16, 1, 128, 0, torch.int32),  # 256 partials, one row group
        ([512], 16, 1, 256, 512, torch.int32),  # 32 partials, all in flight at once
        ([528], 16, 2, 256, 512, torch.int32),  # 33
        ([1024], 8, 1, 128, 512, torch.int32),  # 64, the last whose columns are shared
        ([1040], 8, 1, 256, 512, torch.int32),  # 65
        ([4000, 1, 15, 16, 2047], 8, 2, 128, 0, torch.int64),  # skewed rows
        ([300 + 7 * r for r in range(17)], 8, 2, 128, 0, torch.int32),  # 34 row groups
        ([200 + 3 * r for r in range(33)], 4, 2, 128, 0, torch.int32),  # 66 row groups: past the rule
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
