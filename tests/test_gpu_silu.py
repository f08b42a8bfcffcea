"""The quantizing kernels' SiLU over its whole input space."""
from __future__ import annotations

import ctypes

import pytest

from conftest import gpu_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
P = ctypes.c_void_p


def test_silu_equals_the_float32_restatement_on_every_bf16(pkg):
    """SiLU is taken of bf16 values: with the chip's exponential and reciprocal it rounds to the bits of
    the exp_f32 / IEEE division form (the oracle's) on all 2^16 of them."""
    bad = torch.zeros(1, dtype=torch.int64, device="cuda")
    gpu_case("silu self-test over 2^16 inputs")
    assert pkg.lib().rlu_selftest_silu(P(bad.data_ptr()),
                                       P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert int(bad.item()) == 0
    assert pkg.lib().rlu_selftest_silu(None, None) == -1
