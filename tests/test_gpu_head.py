"""The lm_heads past one 16-row block: fp8 rows equal bit for bit to the 16-row kernel's, W4 rows against
float64."""
from __future__ import annotations

import ctypes

import pytest

from conftest import gpu_case
from w4_bound import w4_limits

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


# the 64-row kernel by itself, also where the entry point above takes the 16-row one; K / 128 = 20, 32,
# 23, 46 and 96: 5, 8, 23, 23 and 24 steps a wave (24 the longest) of 4, 4, 1, 2 and 4 waves
@pytest.mark.parametrize("K", [2560, 4096, 2944, 5888, 12288])
@pytest.mark.parametrize("M", [1, 5, 8, 16, 17, 40, 64])
def test_fp8_head_m64_equals_16_row_kernel(pkg, ops, M, K):
    N = 1152
    gen = torch.Generator(DEV).manual_seed(M + K)
    w = torch.randint(0, 256, (N, K), dtype=torch.uint8, generator=gen, device=DEV)
    w = torch.where((w & 0x7f) == 0x7f, w ^ 1, w).view(torch.float8_e4m3fn)
    ws = torch.rand(N // 128, K // 128, generator=gen, device=DEV) * 0.01
    qx, xs = ops.fp8_quant_group(torch.randn(M, K, generator=gen, device=DEV).bfloat16(), 128)
    gpu_case(f"fp8 head, 64-row kernel alone, M={M} N={N} K={K}")
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
    rc = pkg.lib().rlu_gemm_fp8blk_m64(*[P(t.data_ptr()) for t in (qx, xs, w, ws, y)], M, N, K,
                                       P(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    want = ops.gemm_fp8_block_q(qx, xs, w, ws, npw=2 if M <= 8 else 4)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def test_fp8_head_m64_return_codes(pkg):
    f = pkg.lib().rlu_gemm_fp8blk_m64
    z, s = P(0), P(torch.cuda.current_stream().cuda_stream)
    assert f(*([z] * 5), 20, 1536, 2560, s) == -1
    assert f(*([z] * 5), 65, 1536, 2560, s) == -1 and f(*([z] * 5), 0, 1536, 2560, s) == -1
    assert f(*([z] * 5), 20, 1536 + 64, 2560, s) == -2 and f(*([z] * 5), 20, 1536, 2500, s) == -2
    assert f(*([z] * 5), 20, 1536, 25 * 128, s) == -4          # 25 steps of one wave


def w4_random(N, K, gen):
    """Codes, scales and zeros in the kernel's layout, and the weight they stand for in float64."""
    g = K // 128
    q = torch.randint(0, 16, (N // 16, g, 64, 4, 8), generator=gen, device=DEV)
    shift = torch.tensor([16 * (j % 2) + 4 * (j // 2) for j in range(8)], device=DEV)
    word = (q << shift).sum(-1)                      # lane 16 c + r, dword i: k = 32 i + 8 c + j
    wq = torch.where(word >= 2 ** 31, word - 2 ** 32, word).to(torch.int32)
    scale = (torch.rand(N // 16, g, 16, generator=gen, device=DEV) * 0.01 + 1e-3).bfloat16()
    zero = torch.randint(-20, 36, scale.shape, generator=gen, device=DEV)
    sz = (scale.view(torch.int16).to(torch.int64) & 0xffff) | ((zero & 0xffff) << 16)
    sz = torch.where(sz >= 2 ** 31, sz - 2 ** 32, sz).to(torch.int32)
    codes = q.view(N // 16, g, 4, 16, 4, 8).permute(0, 3, 1, 4, 2, 5).reshape(N, g, 128).double()
    per = lambda t: t.permute(0, 2, 1).reshape(N, g, 1).double()
    w = (codes - per(zero)) * per(scale)
    mag = (codes + 256 + per(zero).abs()) * per(scale)      # what the kernel's terms sum, absolute
    return wq.contiguous(), sz.contiguous(), w.view(N, K), mag.view(N, K)


# strips (N / 16) per wave from none to several, and past five per wave (two passes); K / 128 odd, one
# group, and the longest
@pytest.mark.parametrize("N,K", [(32, 128), (1024, 384), (33024, 256), (65568, 128),
                                 (170016, 640), (4096, 2560), (4096, 4096), (98336, 2560)])
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64, 80, 82])
def test_w4_head_rows_vs_float64(pkg, M, N, K):
    from importlib import import_module
    w4 = import_module(pkg.__name__ + ".w4")
    gen = torch.Generator(DEV).manual_seed(M * K + N)
    wq, sz, w, mag = w4_random(N, K, gen)
    x = torch.randn(M, K, generator=gen, device=DEV).bfloat16()
    x[M // 2] = 0
    gpu_case(f"W4 head M={M} N={N} K={K}")
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
    w4._gemm_into(x, wq.view(torch.uint8).view(N // 16, K // 128, 64, 16), sz, K, y, 0)
    torch.cuda.synchronize()
    for n in range(0, N, 32768):
        low, high = w4_limits(x.double(), w[n:n + 32768], mag[n:n + 32768])
        got = y[:, n:n + 32768].double()
        assert bool(((low <= got) & (got <= high)).all())
    if M == 64:                                      # rows past M stay as they were, M as given
        y2 = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
        w4._gemm_into(x[:50], wq.view(torch.uint8).view(N // 16, K // 128, 64, 16), sz, K, y2, 0)
        torch.cuda.synchronize()
        assert torch.equal(y2[:50].view(torch.int16), y[:50].view(torch.int16))
        assert bool((y2[50:] == 7.0).all())


@pytest.mark.parametrize("off", [1, 2, 8])
def test_heads_take_any_element_aligned_input(pkg, ops, off):
    """Contiguous views that start off a 4- or 16-byte boundary."""
    from importlib import import_module
    w4 = import_module(pkg.__name__ + ".w4")
    gen = torch.Generator(DEV).manual_seed(off)
    M, N, K = 40, 1024, 512
    wq, sz, _, _ = w4_random(N, K, gen)
    wq = wq.view(torch.uint8).view(N // 16, K // 128, 64, 16)
    x = torch.randn(M, K, generator=gen, device=DEV).bfloat16()
    w8 = torch.randint(0, 0x7f, (N, K), dtype=torch.uint8, generator=gen,
                       device=DEV).view(torch.float8_e4m3fn)
    ws = torch.rand(N // 128, K // 128, generator=gen, device=DEV)
    qx, xs = ops.fp8_quant_group(x, 128)
    shift = lambda t: torch.cat([t.view(-1)[:off], t.view(-1)])[off:].view(t.shape)
    gpu_case(f"heads, inputs {off} elements off")
    ya, yb = (torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    w4._gemm_into(x, wq, sz, K, ya, 0)
    w4._gemm_into(shift(x), wq, sz, K, yb, 0)
    f = ops.gemm_fp8_block_q(qx, xs, w8, ws)
    g = ops.gemm_fp8_block_q(shift(qx.view(torch.uint8)).view(torch.float8_e4m3fn), xs, w8, ws)
    torch.cuda.synchronize()
    assert torch.equal(ya.view(torch.int16), yb.view(torch.int16))
    assert torch.equal(f.view(torch.int16), g.view(torch.int16))


def test_w4_head_m64_return_codes(pkg):
    f = pkg.lib().rlu_gemm_w4_m64
    z, s = P(0), P(torch.cuda.current_stream().cuda_stream)
    assert f(z, 20, 2560, z, z, z, 1536, s) == -1
    assert f(z, 16, 2560, z, z, z, 1536, s) == -1 and f(z, 65, 2560, z, z, z, 1536, s) == -1
    for N, K in ((1536 + 16, 2560), (1536, 2500), (1536, 4096 + 128), (1536, 21 * 128)):
        assert f(z, 20, K, z, z, z, N, s) == -2
