"""CPU: the rolled prefill kernel's activation loads stay inside their own row, with nothing but the
vector offset in a buffer's range check (the kernel's own load rule, run on the host)."""
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
