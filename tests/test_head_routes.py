"""CPU: which kernel the heads' entry points launch, by rows, N and K (no GPU: the library's calls are
recorded, not made)."""
from __future__ import annotations

from importlib import import_module

import pytest

torch = pytest.importorskip("torch")


class Calls:
    """Stands for the library: records (entry point, its rows), answers 0."""

    def __init__(self, rows_at):
        self.made, self.rows_at = [], rows_at

    def __getattr__(self, name):
        def call(*a):
            self.made.append((name.rsplit("_", 1)[1], a[self.rows_at]))
            return 0
        return call


@pytest.fixture
def fp8_route(pkg, monkeypatch):
    ops = import_module(pkg.__name__ + ".ops")

    def route(M, N, K, **kw):
        lib = Calls(5)
        monkeypatch.setattr(ops, "lib", lambda: lib)
        monkeypatch.setattr(ops, "stream_ptr", lambda: 0)
        w = torch.empty(1, dtype=torch.uint8).expand(N, K)
        ops.gemm_fp8_block_q(torch.empty(M, K, dtype=torch.uint8), torch.empty(M, K // 128), w,
                             w, out=torch.empty(M, N, dtype=torch.bfloat16), **kw)
        return lib.made
    return route


# the 16-row kernel where the 64-row one is slower: few workgroups, long K, one row that fills its ring
@pytest.mark.parametrize("M,N,K", [
    (1, 8192, 2560), (8, 8192, 2048), (8, 10240, 2560), (8, 20480, 3840), (8, 32000, 1664),
    (1, 151936, 2560), (4, 151936, 4096), (8, 32000, 5120), (1, 128256, 7168), (8, 151936, 8192)])
def test_fp8_head_16_row_kernel(fp8_route, M, N, K):
    assert fp8_route(M, N, K) == [("m16", M)]


@pytest.mark.parametrize("M,N,K", [
    (2, 151936, 2560), (8, 12288, 2560), (8, 8192, 1536), (8, 8192, 3072), (8, 50304, 1664), (1, 151936, 3584),
    (8, 151936, 6144), (4, 102400, 5632), (9, 8192, 2560), (16, 151936, 4096), (64, 4096, 4096)])
def test_fp8_head_64_row_kernel(fp8_route, M, N, K):
    assert fp8_route(M, N, K) == [("m64", M)]


def test_fp8_head_row_blocks_and_given_launch_shapes(fp8_route):
    assert fp8_route(133, 32000, 4096) == [("m64", 64), ("m64", 64), ("m16", 5)]
    assert fp8_route(20, 32000, 2560, npw=4) == [("m16", 16), ("m16", 4)]
    assert fp8_route(20, 32000, 2560, wv=2) == [("m16", 16), ("m16", 4)]
