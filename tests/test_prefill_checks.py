"""CPU: ops.moe_gemm_prefill refuses operands that the kernel would read at other places than they lie (no
GPU: the library's call is recorded, not made)."""
from __future__ import annotations

from importlib import import_module
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")
K, N, MTK, TOP_K, BLOCKS = 512, 256, 30, 3, 4


@pytest.fixture
def call(pkg, monkeypatch):
    ops = import_module(pkg.__name__ + ".ops")
    made = []
    lib = SimpleNamespace(rlu_moe_gemm_prefill=lambda *a: made.append(a) or 0)
    for name, stub in (("lib", lambda: lib), ("stream_ptr", lambda: 0),
                       ("device_ptr", lambda t: t.data_ptr())):
        monkeypatch.setattr(ops, name, stub)
    e = lambda *s, dtype=torch.float32: torch.empty(*s, dtype=dtype)
    args = dict(out=e(MTK, N, dtype=torch.bfloat16), qx=e(MTK // TOP_K, K, dtype=ops.FP8),
                x_scale=e(MTK // TOP_K, K // 128), w0=e(2, N, K, dtype=ops.FP8),
                s0=e(2, N // 128, K // 128), second=None, topk_weights=e(MTK), mtk=MTK,
                top_k=TOP_K, tiles=e(2 * BLOCKS + 1, dtype=torch.int32),
                al0=(e(16 * BLOCKS, dtype=torch.int32), e(BLOCKS, dtype=torch.int32),
                     e(1, dtype=torch.int32)))

    def run(**kw):
        ops.moe_gemm_prefill(**{**args, **kw})
        return len(made)
    run.fp8 = ops.FP8
    return run


def test_operands_that_fit_are_taken(call):
    assert call() == 1
    assert call(topk_weights=None, x_scale=torch.empty(MTK // TOP_K * (K // 128))) == 2
    assert call(qx=torch.empty(MTK // TOP_K + 2, K, dtype=call.fp8),
                x_scale=torch.empty(MTK // TOP_K + 2, K // 128),
                topk_weights=torch.empty(MTK // TOP_K, TOP_K)) == 3


@pytest.mark.parametrize("bad", [
    dict(qx=lambda f: torch.empty(MTK // TOP_K, 2 * K, dtype=f)[:, :K]),         # strided rows
    dict(qx=lambda f: torch.empty(MTK // TOP_K - 1, K, dtype=f)),                # a row too few
    dict(x_scale=lambda f: torch.empty(MTK // TOP_K, K // 128 - 1)),             # a step too few
    dict(x_scale=lambda f: torch.empty(K // 128, MTK // TOP_K).T),               # transposed
    dict(x_scale=lambda f: torch.empty(MTK // TOP_K, K // 128, dtype=torch.bfloat16)),
    dict(topk_weights=lambda f: torch.empty(MTK, dtype=torch.bfloat16)),
    dict(topk_weights=lambda f: torch.empty(MTK - 1)),
    dict(topk_weights=lambda f: torch.empty(2 * MTK)[::2])])
def test_operands_that_do_not_fit_are_refused(call, bad):
    with pytest.raises(AssertionError):
        call(**{k: v(call.fp8) for k, v in bad.items()})
