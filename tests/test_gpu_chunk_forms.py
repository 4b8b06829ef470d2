"""Both forms of the chunked delta rule and both widths of the split form's workgroups, at their edges.

The number of (row, value head) pairs picks the form: up to 32 pairs one 16-column slice per
workgroup, up to 64 two, above that ``chunk_kernel``, which also takes short sequences of more than
eight value heads per key head.  Each at sequence lengths around the conv
history (3 tokens) and the 64-token chunk, with odd and even chunk counts, with and without
carried states, and with token rows that are only 4-byte aligned.  Tolerances as in
``test_gpu_chunk_gated_delta``: outputs 2e-2, fp32 state 1e-3 relative, conv state bit-exact.
"""

from __future__ import annotations

import pytest
import torch

from oracle import gated_delta as gd

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _case(batch: int, key_heads: int, value_heads: int, seq: int, carried: bool, aligned: bool, out_dtype: torch.dtype) -> None:
    import hip_ops

    shape = gd.LinearShape(key_heads, value_heads, 128, 128, 4)
    gen = torch.Generator().manual_seed(1000 * batch + 10 * value_heads + seq)
    mixed = torch.randn(batch, seq, shape.qkv_dim, generator=gen).to(torch.bfloat16)
    a = torch.randn(batch, seq, value_heads, generator=gen)
    b = torch.randn(batch, seq, value_heads, generator=gen)
    a_log = torch.randn(value_heads, generator=gen) - 1.0
    dt_bias = 0.1 * torch.randn(value_heads, generator=gen)
    w = torch.randn(shape.qkv_dim, 1, 4, generator=gen) * 0.5
    tail = torch.randn(batch, shape.qkv_dim, 3, generator=gen) if carried else None
    state = 0.05 * torch.randn(batch, value_heads, 128, 128, generator=gen) if carried else None
    ref, ref_state, ref_tail = gd.linear_attention_core(mixed.float(), a, b, a_log, dt_bias, w, shape, conv_tail=tail, initial_state=state)
    x = mixed.to(DEV)
    if not aligned:  # rows start 4 bytes past a 16-byte boundary
        wide = torch.zeros(batch, seq, shape.qkv_dim + 4, dtype=torch.bfloat16, device=DEV)
        wide[..., 2 : 2 + shape.qkv_dim] = x
        x = wide[..., 2 : 2 + shape.qkv_dim]
    out, new_state, new_tail = hip_ops.chunk_gated_delta_rule(
        x, a.to(DEV), b.to(DEV), a_log.to(DEV), dt_bias.to(DEV), w.to(DEV), key_heads=key_heads, value_heads=value_heads,
        conv_state=None if tail is None else tail.to(DEV), initial_state=None if state is None else state.to(DEV), out_dtype=out_dtype)
    torch.testing.assert_close(out.cpu().float(), ref, atol=2e-2, rtol=2e-2)
    err = float((new_state.double().cpu() - ref_state.double()).norm() / ref_state.double().norm())
    assert err < 1e-3, err
    torch.testing.assert_close(new_tail.cpu(), ref_tail, atol=0, rtol=0)


@pytest.mark.parametrize("batch,key_heads,value_heads", [(1, 1, 1), (1, 1, 5), (2, 4, 16), (3, 1, 11), (4, 8, 16), (5, 1, 13)])
@pytest.mark.parametrize("seq", [1, 3, 64, 65, 130])
def test_forms_match_oracle(batch, key_heads, value_heads, seq) -> None:
    _case(batch, key_heads, value_heads, seq, seq % 2 == 1, True, torch.bfloat16)


@pytest.mark.parametrize("batch,key_heads,value_heads", [(1, 2, 4), (3, 4, 12)])
@pytest.mark.parametrize("seq", [2, 63, 192, 259])
def test_split_form_unaligned_rows_and_fp32_output(batch, key_heads, value_heads, seq) -> None:
    _case(batch, key_heads, value_heads, seq, seq != 192, False, torch.float32)


# either side of the line of the split form where a key head has many value heads: chunks = heads per key head - 8
@pytest.mark.parametrize("batch,key_heads,value_heads,seq", [(1, 1, 10, 64), (1, 1, 10, 65), (2, 1, 12, 192), (2, 1, 12, 193)])
def test_many_value_heads_per_key_head_match_oracle(batch, key_heads, value_heads, seq) -> None:
    _case(batch, key_heads, value_heads, seq, True, True, torch.bfloat16)


def _abi(x, a, b, a_log, dt_bias, w, key_heads, conv_in, conv_out, state_in, state_out, workspace) -> torch.Tensor:
    """``qa_chunk_gated_delta_rule`` on the caller's own buffers, ``workspace`` of its own size."""
    import ctypes

    import hip_loader
    import hip_ops

    lib = hip_loader.load_library()
    batch, seq, _ = x.shape
    heads = a.shape[2]
    out = torch.empty(batch, seq, heads, 128, dtype=torch.bfloat16, device=DEV)
    ptr = lambda t: ctypes.c_void_p(0 if t is None else t.data_ptr())  # noqa: E731
    status = lib.qa_chunk_gated_delta_rule(
        ptr(x), hip_loader.QA_BF16, x.stride(0), x.stride(1), ptr(a), ptr(b), hip_loader.QA_F32, a.stride(0), a.stride(1), ptr(a_log), ptr(dt_bias),
        ptr(w), ptr(conv_in), ptr(conv_out), ptr(state_in), ptr(state_out), ptr(out), hip_loader.QA_BF16, out.stride(0), out.stride(1), batch, seq,
        key_heads, heads, 128, 128, 4, ptr(workspace), workspace.numel(), hip_ops._stream(x.device))
    hip_loader.check(lib, status, "chunk_gated_delta_rule")
    return out


def _device_inputs(batch: int, key_heads: int, value_heads: int, seq: int):
    gen = torch.Generator().manual_seed(100 * batch + seq)
    channels = 2 * key_heads * 128 + value_heads * 128
    x = torch.randn(batch, seq, channels, generator=gen).to(torch.bfloat16).to(DEV)
    a, b = (torch.randn(batch, seq, value_heads, generator=gen).to(DEV) for _ in range(2))
    a_log, dt_bias = (torch.randn(value_heads, generator=gen) - 1.0).to(DEV), torch.zeros(value_heads, device=DEV)
    w = (torch.randn(channels, 4, generator=gen) * 0.5).to(DEV)
    tail = torch.randn(batch, channels, 3, generator=gen).to(DEV)
    state = (0.05 * torch.randn(batch, value_heads, 128, 128, generator=gen)).to(DEV)
    return x, a, b, a_log, dt_bias, w, tail, state


def _workspace(batch: int, seq: int, key_heads: int, value_heads: int) -> torch.Tensor:
    import hip_loader

    size = hip_loader.load_library().qa_chunk_gated_delta_workspace(batch, seq, key_heads, value_heads)
    return torch.empty(size, dtype=torch.uint8, device=DEV)


@pytest.mark.parametrize("batch,key_heads,value_heads", [(1, 2, 4), (3, 4, 12), (5, 1, 13)])
@pytest.mark.parametrize("seq", [1, 2, 3, 33])
def test_states_updated_in_place(batch, key_heads, value_heads, seq) -> None:
    x, a, b, a_log, dt_bias, w, tail, state = _device_inputs(batch, key_heads, value_heads, seq)
    ws = _workspace(batch, seq, key_heads, value_heads)
    new_tail, new_state = torch.empty_like(tail), torch.empty_like(state)
    want = _abi(x, a, b, a_log, dt_bias, w, key_heads, tail, new_tail, state, new_state, ws)
    out = _abi(x, a, b, a_log, dt_bias, w, key_heads, tail, tail, state, state, ws)
    assert torch.equal(out, want)
    assert torch.equal(tail, new_tail)
    assert torch.equal(state, new_state)


def test_workspace_sized_for_more_rows_serves_fewer() -> None:
    # 64 (row, value head) pairs ask for more than 68: the larger batch's buffer holds only the unsplit form's layout
    key_heads, value_heads, seq = 2, 4, 65
    own, reused = _workspace(16, seq, key_heads, value_heads), _workspace(17, seq, key_heads, value_heads)
    assert reused.numel() < own.numel()
    x, a, b, a_log, dt_bias, w, tail, state = _device_inputs(16, key_heads, value_heads, seq)
    args = (x, a, b, a_log, dt_bias, w, key_heads, tail)
    results = []
    for ws in (own, reused):
        new_tail, new_state = torch.empty_like(tail), torch.empty_like(state)
        results.append((_abi(*args, new_tail, state, new_state, ws), new_state, new_tail))
    (want, want_state, want_tail), (out, new_state, new_tail) = results
    torch.testing.assert_close(out.float(), want.float(), atol=2e-2, rtol=2e-2)
    assert float((new_state - want_state).double().norm() / want_state.double().norm()) < 1e-3
    assert torch.equal(new_tail, want_tail)
    least = _workspace(17, seq, key_heads, value_heads).numel() * 16 // 17  # 16 rows of the unsplit layout, whole 256 bytes
    with pytest.raises(RuntimeError, match="workspace"):
        _abi(*args, None, state, None, reused[: least - 256])
