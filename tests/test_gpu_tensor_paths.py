"""The tensor build's paths that small bases do not reach or that pinned tuning
hides, against the oracle: rows so long that each XCD takes a slice of their
chunks, of odd length and of even length off the 128-byte lines, by every shape
that takes them; diagonal cells whose workgroups take several groups of
multipoles, by the rule of an untuned build and with chunks that leave an odd
remainder.

Tolerance: 1e-12 relative per element, the bar of the other tensor tests.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import bs2e  # noqa: E402
from bs2e import capi  # noqa: E402


def _even_grid(k, n_b):
    n_iv = n_b + 3 - k
    return np.concatenate([np.zeros(k), np.arange(1, n_iv) * 0.4, np.full(k, n_iv * 0.4)])


def _fill_nan(rk):
    capi.lib()
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMemset.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
    ptr, n = rk.device_ptr()
    assert hip.hipMemset(ptr, 0xFF, 8 * n) == 0 and hip.hipDeviceSynchronize() == 0


def _rows_ref(oracle, k, t, k_GL, max_k, rows):
    n_b = len(t) - k - 2
    return oracle.rk_rows(k, n_b, max_k, oracle.slater_off_diag(k, t, k_GL, max_k),
                          oracle.slater_diag(k, t, k_GL, max_k), rows)


@pytest.mark.parametrize("n_b", [299, 300])     # 2081 pairs (rows of odd length) and 2088 (even, off the lines)
def test_sliced_rows(n_b, oracle):
    k, k_GL, max_k = 4, 6, 62
    t = _even_grid(k, n_b)
    ctx = bs2e.Context(0)
    rk = bs2e.RkTensor.build(k, t, k_GL, max_k, ctx=ctx, compute=False)
    n, rowlen = rk.n_pairs, rk.n_pairs * rk.K
    assert 2 * 8 * rowlen > 2 << 20 and rowlen % 16 != 0
    rows = np.array([0, 1, 7, n // 2, n // 2 + 1, n - 2, n - 1])
    ref = _rows_ref(oracle, k, t, k_GL, max_k, rows)
    shapes = [None, *range(7)] if rowlen % 2 == 0 else [None, 5, 6]
    for shape in shapes:
        if shape is not None:
            rk.set_tuning(shape, rk.tuning()[1])
        _fill_nan(rk)
        rk.compute()
        got = rk.rows(rows)
        assert np.all(np.abs(got - ref) <= 1e-12 * np.abs(ref)), shape
    rk.release()
    ctx.close()


@pytest.mark.parametrize("k,n_b,k_GL,max_k", [(4, 33, 7, 18), (9, 39, 11, 16), (8, 150, 9, 12), (12, 40, 14, 6)])
def test_cells_in_groups_of_multipoles(k, n_b, k_GL, max_k, oracle):
    t = _even_grid(k, n_b)
    ctx = bs2e.Context(0)
    rk = bs2e.RkTensor.build(k, t, k_GL, max_k, ctx=ctx, compute=False)
    n = rk.n_pairs
    rows = np.array([0, n // 3, n // 2, n - 1])
    ref = _rows_ref(oracle, k, t, k_GL, max_k, rows)
    taken = []
    for kc in (None, 3, 5, 6, 7, 13):
        if kc is not None:
            try:
                rk.set_tuning(rk.tuning()[0], kc)
            except bs2e.Bs2eError:
                continue
        _fill_nan(rk)
        rk.compute()
        assert np.all(np.abs(rk.rows(rows) - ref) <= 1e-12 * np.abs(ref)), kc
        taken.append(kc)
    assert 3 in taken and (k > 9 or 7 in taken)
    rk.release()
    ctx.close()
