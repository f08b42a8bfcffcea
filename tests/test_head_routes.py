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


# the 16-row kernel where the 64-row one is slower: up to 128 workgroups of it (K split over 4, 2 and 1
# waves), long K, few CUs with a second workgroup, a last round under 0.6 full, one row that fills
# its ring
@pytest.mark.parametrize("M,N,K", [
    (1, 8192, 2560), (8, 8192, 2048), (8, 16384, 3840), (8, 32000, 1664), (2, 20480, 2560),
    (8, 102400, 3840), (8, 151936, 2944), (1, 151936, 2560), (4, 151936, 4096), (8, 32000, 5120),
    (1, 128256, 7168), (8, 151936, 8192), (8, 16384, 8192)])
def test_fp8_head_16_row_kernel(fp8_route, M, N, K):
    assert fp8_route(M, N, K) == [("m16", M)]


# (from 129 to 255 workgroups, and where the ring pads too much of the steps or they are under 4)
@pytest.mark.parametrize("M,N,K", [
    (2, 151936, 2560), (8, 8320, 2560), (1, 10240, 2560), (8, 12288, 8192), (8, 16256, 5120),
    (4, 16512, 3840), (8, 50304, 1664), (8, 128256, 2944), (8, 8192, 1536), (8, 8192, 3072),
    (1, 151936, 3584), (8, 151936, 6144), (4, 102400, 5632), (8, 50304, 5888), (9, 8192, 2560), (16, 151936, 4096),
    (64, 4096, 4096)])
def test_fp8_head_64_row_kernel(fp8_route, M, N, K):
    assert fp8_route(M, N, K) == [("m64", M)]


def test_fp8_head_row_blocks_and_given_launch_shapes(fp8_route):
    assert fp8_route(133, 32000, 4096) == [("m64", 64), ("m64", 64), ("m16", 5)]
    assert fp8_route(20, 32000, 2560, npw=4) == [("m16", 16), ("m16", 4)]
    assert fp8_route(20, 32000, 2560, wv=2) == [("m16", 16), ("m16", 4)]


@pytest.fixture
def w4_route(pkg, monkeypatch):
    w4 = import_module(pkg.__name__ + ".w4")

    def route(M, N, K, wv=0):
        lib = Calls(1)
        monkeypatch.setattr(w4, "lib", lambda: lib)
        monkeypatch.setattr(w4, "stream_ptr", lambda: 0)
        wq = torch.empty(1, dtype=torch.uint8).expand(N // 16, K // 128, 64, 16)
        w4._gemm_into(torch.empty(M, K, dtype=torch.bfloat16), wq, torch.empty(1), K,
                      torch.empty(M, N, dtype=torch.bfloat16), wv)
        return lib.made
    return route


# few output rows and a K whose last half ring is padding: 16 rows at a time up to 32 of them
@pytest.mark.parametrize("M,N,K,made", [
    (32, 4096, 2560, [16, 16]), (17, 1024, 3584, [16, 1]), (24, 4096, 1536, [16, 8]),
    (16, 151936, 2560, [16]), (88, 4096, 2560, [64, 16, 8]), (33, 4096, 2560, [33]),
    (32, 4128, 2560, [32]), (32, 4096, 2048, [32]), (32, 1024, 512, [32]),
    (17, 1024, 1792, [17]), (64, 151936, 2560, [64]), (82, 151936, 2560, [64, 18])])
def test_w4_head_routes(w4_route, M, N, K, made):
    assert w4_route(M, N, K) == [("m64" if m > 16 else "m16", m) for m in made]
    assert w4_route(20, 151936, 2560, wv=2) == [("m16", 16), ("m16", 4)]
