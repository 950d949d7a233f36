"""One-electron matrices at the sizes where the band assembly can go wrong:
fewer splines than the order (every element in the band), one past a whole
number of 256-row strips, one l, a whole group of l and one more, GL orders
whose potentials leave a workgroup fewer l.

Bar: every element within 1e-12 of the matrix's largest element, as the other
one-electron tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import bs2e  # noqa: E402


def _even_grid(k, n_b):
    n_iv = n_b + 3 - k
    return np.concatenate([np.zeros(k), np.arange(1, n_iv) * 0.4, np.full(k, n_iv * 0.4)])


@pytest.mark.parametrize("k,n_b,k_GL,ls", [(2, 2, 3, range(1)), (6, 5, 8, range(9)), (8, 8, 14, range(3, 4)),
                                           (4, 257, 7, range(8)), (9, 40, 64, range(6)), (16, 20, 40, range(17))])
def test_one_electron_band_at_edges(k, n_b, k_GL, ls, oracle):
    t = _even_grid(k, n_b)
    assert len(t) - k - 2 == n_b
    spl = bs2e.b_spline(k, t)
    cap = (3, 0.6 * t[-1], 0.02 + 0.005j)
    S = bs2e.setup_S(spl, k_GL)
    ref = oracle.setup_S(k, t, k_GL)
    assert np.abs(S - ref).max() <= 1e-12 * np.abs(ref).max()
    H = bs2e.setup_H_one_particle(2, cap, ls, spl, k_GL)
    for i, l in enumerate(ls):
        ref = oracle.setup_H1p(k, t, k_GL, 2, l, cap_order=cap[0], cap_r0=cap[1], cap_eta=cap[2])
        assert np.abs(H[i] - ref).max() <= 1e-12 * np.abs(ref).max(), l
