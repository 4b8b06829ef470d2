"""Which form or plan a size takes, read off the workspace it asks for: host code of the library, no GPU."""

from __future__ import annotations

import pytest

import hip_loader


def _library():
    if not hip_loader.LIBRARY_PATH.exists():
        pytest.fail(f"{hip_loader.LIBRARY_PATH} is not built; run __graft_entry__.build()")
    return hip_loader.load_library()


def _chunk_workspace(batch: int, seq: int, key_heads: int, value_heads: int, split: bool) -> int:
    """Bytes of the chunked delta rule: fp16 q and k, then 16 bytes per token and value head or 17 KB per chunk and value head."""
    chunks = (seq + 63) // 64
    return 2 * batch * chunks * 64 * key_heads * 128 * 2 + batch * value_heads * chunks * (17 * 1024 if split else 64 * 16)


# The split form for up to 64 (row, value head) pairs, and of more than eight value heads per key head only where the
# sequence has as many chunks as there are heads above the eighth
@pytest.mark.parametrize("batch,seq,key_heads,value_heads,split", [
    (1, 1, 16, 32, True), (2, 4096, 16, 32, True), (3, 4096, 16, 32, False), (8, 1, 1, 8, True), (1, 64, 1, 9, True), (1, 64, 1, 10, False),
    (1, 65, 1, 10, True), (1, 512, 1, 32, False), (1, 1472, 1, 32, False), (1, 1473, 1, 32, True), (1, 3520, 1, 64, False), (1, 3521, 1, 64, True),
])
def test_chunked_delta_rule_form(batch, seq, key_heads, value_heads, split) -> None:
    size = _library().qa_chunk_gated_delta_workspace(batch, seq, key_heads, value_heads)
    assert size == _chunk_workspace(batch, seq, key_heads, value_heads, split)


@pytest.mark.parametrize("out_features,in_features", [(2048, 2048), (2048, 4096)])
def test_fp8_linear_workspace_of_more_rows_holds_fewer(out_features, in_features) -> None:
    # 512 to 960 rows: without the block kernel all of them split K in two, with it the larger counts do not split
    sizes = [_library().qa_fp8_linear_workspace(rows, out_features, in_features) for rows in range(512, 961, 32)]
    assert sizes == sorted(sizes)
    assert sizes[0] >= 2 * 512 * out_features * 4 + 512 * in_features * 2  # fp32 partials, then x as fp16
