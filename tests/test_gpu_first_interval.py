"""The off-diagonal moments of the interval next to r = 0, element by element
against their definition in extended precision.

There the outer point r = h x + c is a small difference of h and c, and the
moments take its powers up to 1 / r^(k+1), so a point rounded once more than
needed shows in them many times over.

Bar, in units of 2^-53 and from the operations alone (every term is positive):
the point rounded once, k + 1 of it in a power to k + 1 and k more from the
multiplications; two splines, each from k_s - 1 steps of five roundings and
k_s - 1 powers of the point at most; the sum over k_GL points; six more for the
weights, the reciprocal and the interval's width.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import bs2e  # noqa: E402


def _splines(t, k, r):
    """The k splines non-zero on the first interval at r (Cox-de Boor), in extended precision."""
    t = t.astype(np.longdouble)
    i = k - 1
    b = [np.longdouble(1)]
    for j in range(1, k):
        saved, nxt = np.longdouble(0), []
        for m in range(j):
            right, left = t[i + 1 + m] - r, r - t[i + 1 - j + m]
            term = b[m] / (right + left)
            nxt.append(saved + right * term)
            saved = left * term
        b = nxt + [saved]
    return b


def _moments(t, k, k_GL, max_k, oracle):
    """P, Q [a][c][k] of the first interval for its local splines."""
    x, w = (v.astype(np.longdouble) for v in oracle.gauss_legendre(k_GL))
    lim1, lim2 = np.longdouble(t[k - 1]), np.longdouble(t[k])
    h, c = (lim2 - lim1) / 2, (lim2 + lim1) / 2
    P, Q = (np.zeros((k, k, max_k + 1), np.longdouble) for _ in range(2))
    for q in range(k_GL):
        r = h * x[q] + c
        B = np.array(_splines(t, k, r))
        BB = h * w[q] * B[:, None] * B[None, :]
        for m in range(max_k + 1):
            P[:, :, m] += BB * r ** m
            Q[:, :, m] += BB / r ** (m + 1)
    return P, Q


# Widths of the first interval that are no power of two, where h x would be exact.
@pytest.mark.parametrize("width", [0.05, 0.07, 0.13])
@pytest.mark.parametrize("k,k_GL,max_k", [(4, 6, 2), (4, 16, 30), (8, 12, 15), (9, 14, 24), (12, 20, 8), (16, 26, 12)])
def test_moments_next_to_the_origin(k, k_GL, max_k, width, oracle):
    t = bs2e.generate_grid(k, 3, 2, 1.0, 10.0)
    t = t * (width / t[k])
    spl = bs2e.b_spline(k, t)
    r_k, r_m_k, r_d_k = (x().init(max_k, spl) for x in (bs2e.sparse_4d, bs2e.sparse_4d, bs2e.sparse_6d))
    bs2e.setup_Slater_integrals(spl, max_k, k_GL, r_k, r_m_k, r_d_k)
    bar = (2 * np.arange(max_k + 1) + 1 + 12 * (k - 1) + k_GL + 6) * 2.0 ** -53
    for got, ref, name in zip((r_k, r_m_k), _moments(t, k, k_GL, max_k, oracle), ("P", "Q")):
        n = got.iv == 1
        assert n.sum() == (k - 1) ** 2
        # basis function b is spline b + 1, the local spline b of the first interval
        want = ref[got.i[n], got.j[n]]
        err = np.abs((got.data[n] - want) / want).max(axis=0).astype(float)
        print(f"{name}: worst error over bar {float((err / bar).max()):.3f}", flush=True)
        assert np.all(err <= bar), (name, err, bar)
