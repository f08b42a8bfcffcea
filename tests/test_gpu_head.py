"""The lm_heads past one 16-row block: every row equal bit for bit to the 16-row kernel's."""
from __future__ import annotations

import ctypes

import pytest

from conftest import gpu_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"
P = ctypes.c_void_p


@pytest.fixture(scope="module")
def ops(pkg):
    from importlib import import_module
    return import_module(pkg.__name__ + ".ops")


# K / 128 = 1, 2, 3, 20, 17, 32: split over 1, 2, 1, 4, 1 and 4 waves, with 1 to 17 steps each
@pytest.mark.parametrize("K", [128, 256, 384, 2560, 2176, 4096])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 81])
def test_fp8_head_rows_equal_16_row_launches(ops, M, K):
    for N in (128, 1152):
        gen = torch.Generator(DEV).manual_seed(M * K + N)
        w = torch.randint(0, 256, (N, K), dtype=torch.uint8, generator=gen, device=DEV)
        w = torch.where((w & 0x7f) == 0x7f, w ^ 1, w).view(torch.float8_e4m3fn)
        ws = torch.rand(N // 128, K // 128, generator=gen, device=DEV) * 0.01
        x = torch.randn(M, K, generator=gen, device=DEV).bfloat16()
        x[M // 2] = 0
        qx, xs = ops.fp8_quant_group(x, 128)
        gpu_case(f"fp8 head M={M} N={N} K={K}")
        y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.gemm_fp8_block_q(qx, xs, w, ws, out=y)
        want = ops.gemm_fp8_block_q(qx, xs, w, ws, npw=4)      # launches of 16 rows
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def test_fp8_head_m64_return_codes(pkg):
    f = pkg.lib().rlu_gemm_fp8blk_m64
    z, s = P(0), P(torch.cuda.current_stream().cuda_stream)
    assert f(*([z] * 5), 20, 1536, 2560, s) == -1
    assert f(*([z] * 5), 65, 1536, 2560, s) == -1 and f(*([z] * 5), 0, 1536, 2560, s) == -1
    assert f(*([z] * 5), 20, 1536 + 64, 2560, s) == -2 and f(*([z] * 5), 20, 1536, 2500, s) == -2
    assert f(*([z] * 5), 20, 1536, 25 * 128, s) == -4          # 25 steps of one wave
