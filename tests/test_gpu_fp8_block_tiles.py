"""The fp8 linear layer's block kernel at the edges of its tiles and of its dispatch rule, against the float64 oracle.

Tolerances as in ``test_gpu_fp8_linear.py``: 1e-5 x max|y| and 1e-3 relative for bf16 rows (exact products, fp32 sums),
1e-3 x max|y| for fp32 rows, which are rounded to fp16; two weight layouts and two output types of one call agree.
"""

from __future__ import annotations

import pytest
import torch

from oracle import fp8_linear as oracle

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _inputs(rows: int, n: int, k: int, dtype: torch.dtype):
    gen = torch.Generator().manual_seed(rows + n + k)
    w = (torch.randn((n, k), generator=gen) * 0.5).to(torch.float8_e4m3fn)
    s = (torch.rand((n // 128, k // 128), generator=gen) * 1.9 + 0.1).to(torch.bfloat16)
    return torch.randn((rows, k), generator=gen).to(dtype), w, s


def _fp64(x: torch.Tensor, w: torch.Tensor, s: torch.Tensor) -> torch.Tensor:
    table = torch.from_numpy(oracle.e4m3_table()).double()
    full = table[w.view(torch.uint8).long()] * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    return x.double() @ full.t()


# tiles of 64 x 128, 128 x 128 and 128 x 256, sizes either side of where the rule changes tile among them; counts of
# tiles just past a whole round; out_features that leave half a tile; one K block (two stages, fewer than the ring) and
# an odd number of them
@pytest.mark.parametrize("rows,n,k", [(129, 8192, 128), (192, 8192, 384), (193, 6912, 128), (257, 8192, 256), (300, 4096, 640), (385, 8064, 128),
                                      (641, 8192, 128), (769, 7296, 384), (767, 4096, 128), (4097, 1664, 128), (2560, 512, 256), (300, 12288, 128), (513, 8192, 128),
                                      (1281, 6144, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_tiles_match_fp64(rows, n, k, dtype) -> None:
    import hip_ops as ops

    x, w, s = _inputs(rows, n, k, dtype)
    xd, wd, sd = x.to(DEV), w.to(DEV), s.to(DEV)
    out = ops.fp8_e4m3_bf16_linear(xd, wd, sd)
    ref = _fp64(x, w, s)
    atol = (1e-3 if dtype == torch.float32 else 1e-5) * ref.abs().max().item()
    torch.testing.assert_close(out.cpu().double(), ref, atol=atol, rtol=1e-3)
    packed = ops.fp8_pack_weight(wd)
    assert torch.equal(ops.fp8_e4m3_bf16_linear(xd, packed, sd), out)
    assert torch.equal(ops.fp8_e4m3_bf16_linear(xd, packed, sd, out_dtype=torch.bfloat16), out.to(torch.bfloat16))


def test_nan_code_and_infinite_row_stay_in_their_column_and_row() -> None:
    import hip_ops as ops

    x, w, s = _inputs(300, 8192, 256, torch.bfloat16)
    codes = w.view(torch.uint8).clone()
    codes[8191, 200] = 0x7F
    x[299, 7] = float("inf")
    out = ops.fp8_e4m3_bf16_linear(x.to(DEV), codes.view(torch.float8_e4m3fn).to(DEV), s.to(DEV)).cpu()
    assert torch.isnan(out[:, 8191]).all().item()
    assert not torch.isfinite(out[299]).any().item()
    assert torch.isfinite(out[:299, :8191]).all().item()


# The largest row stride that the block kernel takes and the next one past it, through the C ABI (the Python entry makes
# x contiguous first): past it the x-resident, wide and tiled kernels (in_features 128 and 2176; up to 256 rows and more)
# and a K split (in_features 2176, 5 x 32 tiles).
@pytest.mark.parametrize("rows,n,k", [(129, 8192, 128), (129, 8192, 2176), (257, 4096, 2176), (385, 4096, 128)])
@pytest.mark.parametrize("past", [0, 8])
def test_rows_further_apart_than_the_block_kernel_takes(rows, n, k, past) -> None:
    import ctypes

    import hip_loader
    import hip_ops as ops

    stride = (1 << 23) + past
    x, w, s = _inputs(rows, n, k, torch.bfloat16)
    xd, wd, sd = torch.empty((rows - 1) * stride + k, dtype=torch.bfloat16, device=DEV).as_strided((rows, k), (stride, 1)), w.to(DEV), s.to(DEV)
    xd.copy_(x.to(DEV))
    lib = hip_loader.load_library()
    workspace = torch.empty(lib.qa_fp8_linear_workspace(rows, n, k), dtype=torch.uint8, device=DEV)
    out = torch.empty(rows, n, device=DEV)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    status = lib.qa_fp8_linear(ptr(xd), hip_loader.QA_BF16, stride, rows, ptr(wd), 0, ptr(sd), n, k, ptr(out), hip_loader.QA_F32, n, ptr(workspace),
                               workspace.numel(), ops._stream(out.device))
    hip_loader.check(lib, status, "fp8_linear")
    ref = _fp64(x, w, s)
    torch.testing.assert_close(out.cpu().double(), ref, atol=1e-5 * ref.abs().max().item(), rtol=1e-3)
