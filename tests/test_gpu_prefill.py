"""The streamed prefill GEMMs (the unrolled K = 768 kernel and the rolled one for other K) against the general tiled kernel, which runs the same sequence of operations per
output: equal bit for bit, over row distributions that take each branch of the tiles' schedule.
"""
from __future__ import annotations

import pytest

from conftest import gpu_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops(pkg):
    from importlib import import_module
    return import_module(pkg.__name__ + ".ops")


# rows per expert: tiles of one and of several per expert mixed, at 24 rows per tile or more (the
# workgroups are split between the two kinds) and below (list order); only one kind; fewer items
# than XCDs; no tile at all.
ROWS = {
    "mixed": [300, 5, 40, 17, 128, 129, 1, 0, 16, 700, 96, 250, 33] * 4,
    "mixed_few": [300, 40, 130],
    "alone": [128, 100, 90, 77] * 6,
    "shared": [400] * 5,
    "thin": [9] * 40 + [200],
    "one": [3],
    "none": [],
}
SHAPES = [(768, 512), (1024, 256), (1536, 256), (2048, 768), (2560, 512), (4096, 256)]


def align(rows, order, mtk=None):
    """One align of sum(rows) ids dealt to the experts in the given order, padded with mtk."""
    mtk = sum(rows) if mtk is None else mtk
    sid, eid, pos = [], [], 0
    for e, r in enumerate(rows):
        nb = (r + 15) // 16
        sid += order[pos:pos + r] + [mtk] * (nb * 16 - r)
        eid += [e] * nb
        pos += r
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    n = len(eid)
    return dev(sid or [mtk] * 16), dev(eid or [-1]), dev([16 * n])


def weights(E, N, K, gen):
    """Finite e4m3 bytes (0x7f and 0xff are NaN) and positive block scales."""
    w = torch.randint(0, 256, (E, N, K), dtype=torch.uint8, generator=gen, device=DEV)
    w = torch.where((w & 0x7f) == 0x7f, w ^ 1, w).view(torch.float8_e4m3fn)
    return w, torch.rand(E, N // 128, K // 128, generator=gen, device=DEV) * 0.01


def tile_list(rows):
    """moe_gemm_tiles of that align, where it has more blocks than the builder takes."""
    out, b = [], 0
    for r in rows:
        nb = (r + 15) // 16
        for s in range(0, nb, 8):
            out += [b + s, min(8, nb - s)]
        b += nb
    out = out + [0] * (2 * b - len(out)) + [len(out) // 2]
    return torch.tensor(out, dtype=torch.int32, device=DEV)


def check(ops, name, rows, K, N, routed, E=None):
    gen = torch.Generator(DEV).manual_seed(K + N)
    E = E or max(len(rows), 1)
    mtk = max(sum(rows), 1)
    w, ws = weights(E, N, K, gen)
    order = torch.randperm(mtk, generator=torch.Generator().manual_seed(1)).tolist()
    al = align(rows, order)
    if len(rows) > E:
        al[1].remainder_(E)                          # neighbours stay of different experts
    tiles = tile_list(rows) if len(rows) > E else None
    qx = torch.randint(0, 0x7f, (mtk, K), dtype=torch.uint8, generator=gen, device=DEV)
    qx = (qx ^ 0x80 * (qx & 1)).view(torch.float8_e4m3fn)     # signs by the lowest bit
    xs = torch.rand(mtk, K // 128, generator=gen, device=DEV)
    tw = torch.rand(mtk, generator=gen, device=DEV) if routed else None
    out = []
    for wv in (0, 2):
        y = torch.full((mtk, N), 7.0, dtype=torch.bfloat16, device=DEV)
        gpu_case(f"streamed prefill gemm {name} K={K} N={N} wv={wv}")
        ops.moe_gemm_tiled(y, qx, xs, w, ws, *al, tw, mtk, 1, wv=wv, tiles=tiles,
                           tiles_ready=tiles is not None)
        torch.cuda.synchronize()
        out.append(y.view(torch.int16))
    assert torch.equal(*out)
    assert bool((out[0] != 0x40e0).any()) == bool(rows)      # 7.0 where nothing was written


@pytest.mark.parametrize("K,N", SHAPES)
@pytest.mark.parametrize("name", ROWS)
def test_streamed_equals_general_tiled(ops, name, K, N):
    check(ops, name, ROWS[name], K, N, routed=N % 512 == 0)


# K of one chunk of 4 steps, with 1, 2 and 3 steps in the last one; these take the kernel from two
# items per CU on (the row counts repeated until there are), and the general one below
@pytest.mark.parametrize("K,N", [(512, 1536), (640, 2560), (1408, 2048), (1792, 1792)])
@pytest.mark.parametrize("name", ["mixed", "alone", "shared", "thin", "mixed_few"])
def test_streamed_broken_k_equals_general_tiled(ops, name, K, N):
    rows = ROWS[name]
    if name != "mixed_few":
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        rows = rows * -(-2 * 128 * 256 * cus // (N * sum(rows)))
    check(ops, name, rows, K, N, routed=name != "shared")


@pytest.mark.parametrize("K", [768, 1024])
@pytest.mark.parametrize("n", [16000, 16380, 17000])
def test_streamed_at_the_orders_capacity(ops, n, K):
    """Tiles up to what the XCDs' orders hold (2048 each), and past that and past what the
    scheduler takes (16384)."""
    check(ops, f"{n} tiles", [40] * n + [200], K, 256, routed=True, E=64)


@pytest.mark.parametrize("K", [2560, 2688])
def test_streamed_activations_past_2gb(ops, K):
    """Row offsets past 31 bits take the 64-bit addresses: 2.2 GB of activations, of which the
    align names rows at both ends."""
    tokens, N = 860_000, 256
    gen = torch.Generator(DEV).manual_seed(7)
    w, ws = weights(3, N, K, gen)
    qx = torch.randint(0, 0x7f, (tokens, K), dtype=torch.uint8, generator=gen,
                       device=DEV).view(torch.float8_e4m3fn)
    xs = torch.rand(tokens, K // 128, generator=gen, device=DEV)
    ids = list(range(300)) + list(range(tokens - 212, tokens))
    sid = torch.tensor(ids, dtype=torch.int32, device=DEV)
    eid = torch.tensor([0] * 10 + [1] * 3 + [2] * 19, dtype=torch.int32, device=DEV)
    npad = torch.tensor([512], dtype=torch.int32, device=DEV)
    out = []
    for wv in (0, 2):
        y = torch.zeros(tokens, N, dtype=torch.bfloat16, device=DEV)
        gpu_case(f"streamed prefill gemm, activations past 2 GB, wv={wv}")
        ops.moe_gemm_tiled(y, qx, xs, w, ws, sid, eid, npad, None, tokens, 1, wv=wv)
        torch.cuda.synchronize()
        out.append(y.view(torch.int16))
    assert torch.equal(*out) and bool(out[0][ids].any())


# whole and broken K; few items (the broken K then has no kernel) and two per CU
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("K,I,rep", [(1024, 256, 1), (2048, 384, 1), (640, 640, 4), (1408, 512, 6)])
def test_layer_prefill_gemm_equals_its_parts(ops, K, I, rep, two):
    """moe_gemm_prefill (one or two aligns; plain with routed weights, or with the activation) against
    the general tiled kernel on each align and silu_mul_quant."""
    N, rows = 2 * I, ROWS["mixed"] * rep
    gen = torch.Generator(DEV).manual_seed(K + I)
    rows1 = [r if i % 3 else 0 for i, r in enumerate(rows)] if two else rows
    rows2 = [r - q for r, q in zip(rows, rows1)]
    mtk = sum(rows)
    assert ops.moe_gemm_prefill_takes(mtk, K, N) and ops.moe_gemm_prefill_takes(mtk, K, N, True)
    order = torch.randperm(mtk, generator=torch.Generator().manual_seed(2)).tolist()
    sets = []
    for rs, o in ((rows1, order[:sum(rows1)]), (rows2, order[sum(rows1):]))[:1 + two]:
        sets.append((*weights(len(rows), N, K, gen), align(rs, o, mtk)))
    qx = torch.randint(0, 0x7f, (mtk, K), dtype=torch.uint8, generator=gen, device=DEV)
    qx = (qx ^ 0x80 * (qx & 1)).view(torch.float8_e4m3fn)
    xs = torch.rand(mtk, K // 128, generator=gen, device=DEV)
    tw = torch.rand(mtk, generator=gen, device=DEV)
    (w, s, al), second = sets[0], (sets[1] if two else None)
    tiles = ops.moe_gemm_tiles_split(al[1:], second[2][1:]) if two else ops.moe_gemm_tiles(*al[1:])
    gpu_case(f"layer prefill gemm K={K} N={N} two={two}")
    want, routed = (torch.empty(mtk, N, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    for w_, s_, al_ in sets:
        ops.moe_gemm_tiled(want, qx, xs, w_, s_, *al_, None, mtk, 1, wv=2)
        ops.moe_gemm_tiled(routed, qx, xs, w_, s_, *al_, tw, mtk, 1, wv=2)
    q0, s0 = ops.silu_mul_quant(want, group=128)[1:]
    y = torch.empty_like(want)
    q2, s2 = torch.empty_like(q0), torch.empty_like(s0)
    ops.moe_gemm_prefill(y, qx, xs, w, s, al, second, tw, mtk, 1, tiles)
    ops.moe_gemm_prefill((q2, s2), qx, xs, w, s, al, second, None, mtk, 1, tiles)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), routed.view(torch.int16))
    assert torch.equal(q2.view(torch.uint8), q0.view(torch.uint8)) and torch.equal(s2, s0)


def test_layer_prefill_gemm_shapes_and_return_codes(pkg, ops):
    import ctypes
    P = ctypes.c_void_p
    takes = ops.moe_gemm_prefill_takes
    assert takes(1, 2560, 1536, True) and takes(1, 768, 2560) and not takes(1, 768, 2560, True)
    assert takes(1, 1024, 256) and not takes(1, 1024, 384) and not takes(0, 2560, 1536)
    assert not takes(4096, 640, 256) and not takes(1 << 20, 384, 2048)
    assert not takes(1 << 20, 1000, 2048)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert takes(256 * cus, 640, 256) and not takes(256 * cus - 1, 640, 256)
    f, s = pkg.lib().rlu_moe_gemm_prefill, P(torch.cuda.current_stream().cuda_stream)
    z = P(0)
    call = lambda mtk, K, N, y, q: f(*([z] * 12), 1, z, y, q, z, mtk, 1, K, N, s)
    assert call(20, 2560, 1536, z, z) == -1 and call(20, 384, 1536, z, z) == -6
    assert call(20, 768, 2560, z, P(1)) == -6 and call(20, 2560, 1500, z, z) == -2
    assert call(0, 2560, 1536, z, z) == 0


@pytest.mark.parametrize("K,N", [(768, 512), (1024, 512), (2560, 256)])
def test_second_set_in_host_memory(ops, K, N):
    """The second align's weights in pinned host memory (unshared tiles are then walked from the
    end): the bits of the same call over device copies, eager and in a replayed graph."""
    gen = torch.Generator(DEV).manual_seed(K + N)
    # unshared tiles of both sets, 0 to 4 of them per XCD, beside shared ones
    rows = [300, 40, 17, 128, 1, 0, 700, 96, 33] * 4 + [50] * 3
    rows1 = [r if i % 2 else 0 for i, r in enumerate(rows)]
    rows2 = [r - q for r, q in zip(rows, rows1)]
    mtk = sum(rows)
    order = torch.randperm(mtk, generator=torch.Generator().manual_seed(3)).tolist()
    w0, s0 = weights(len(rows), N, K, gen)
    w1, s1 = weights(len(rows), N, K, gen)
    al0 = align(rows1, order[:sum(rows1)], mtk)
    al1 = align(rows2, order[sum(rows1):], mtk)
    host = [torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t) for t in (w1, s1)]
    qx = torch.randint(0, 0x7f, (mtk, K), dtype=torch.uint8, generator=gen,
                       device=DEV).view(torch.float8_e4m3fn)
    xs = torch.rand(mtk, K // 128, generator=gen, device=DEV)
    tw = torch.rand(mtk, generator=gen, device=DEV)
    tiles = ops.moe_gemm_tiles_split(al0[1:], al1[1:])
    want, y = (torch.full((mtk, N), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    gpu_case(f"prefill gemm, second set in host memory, K={K} N={N}")
    ops.moe_gemm_prefill(want, qx, xs, w0, s0, al0, (w1, s1, al1), tw, mtk, 1, tiles)
    call = lambda: ops.moe_gemm_prefill(y, qx, xs, w0, s0, al0, (*host, al1), tw, mtk, 1, tiles)
    call()
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        y.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
