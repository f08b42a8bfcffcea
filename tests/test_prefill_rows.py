"""CPU: the rolled prefill kernel's activation loads stay inside their own row, with nothing but the
vector offset in a buffer's range check, and it loads each weight step once (the kernel's own load
rules, run on the host)."""
from __future__ import annotations

import ctypes

import pytest


def outside(pkg, rows, K):
    if not pkg.LIB_PATH.exists():
        pytest.skip("librlu.so not built")
    bad = ctypes.c_ulonglong(999)
    rc = pkg.lib().rlu_selftest_prefill_rows(rows, K, ctypes.byref(bad))
    return rc, bad.value


# whole chunks of 4 steps; 1, 2 and 3 steps in the last one; a single chunk; the longest row
@pytest.mark.parametrize("K", [1024, 2048, 2560, 640, 896, 1408, 1664, 1792, 2688, 512, 1 << 20])
@pytest.mark.parametrize("rows", [1, 2, 2047])
def test_row_loads_stay_inside_their_row(pkg, rows, K):
    assert outside(pkg, rows, K) == (0, 0)


def test_row_load_check_refuses_bad_sizes(pkg):
    assert outside(pkg, 0, 1024)[0] == -1 and outside(pkg, 1, 0)[0] == -1
    assert outside(pkg, 1, 1000)[0] == -2 and outside(pkg, 1, 384)[0] == -2
    assert outside(pkg, 4096, 1 << 20)[0] == -2
    assert pkg.lib().rlu_selftest_prefill_rows(1, 1024, None) == -1


@pytest.mark.parametrize("K", [512, 640, 896, 1024, 1152, 1408, 1536, 1664, 2048, 2560])
@pytest.mark.parametrize("items", [1, 2, 3, 17])
def test_each_weight_step_is_loaded_once(pkg, items, K):
    """None twice, and none after the last item (over 256 workgroups 33 MB, 0.55 ms of the host link)."""
    steps = ctypes.c_ulonglong(999)
    assert pkg.lib().rlu_selftest_prefill_steps(items, K, ctypes.byref(steps)) == 0
    assert steps.value == items * K // 128


def test_weight_step_count_refuses_bad_sizes(pkg):
    n = ctypes.c_ulonglong(0)
    f = pkg.lib().rlu_selftest_prefill_steps
    assert f(0, 1024, ctypes.byref(n)) == -1 and f(1, 0, ctypes.byref(n)) == -1
    assert f(1, 1000, ctypes.byref(n)) == -2 and f(1, 384, ctypes.byref(n)) == -2
    assert f(1, 1024, None) == -1
