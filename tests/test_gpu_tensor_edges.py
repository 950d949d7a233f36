"""The tensor kernels at the sizes where they can go wrong, against the oracle:
one multipole and few (element indices by reciprocals of K), rows whose length
is odd, even and a whole number of 128-byte lines, bases with barely more
splines than the order (no column lies apart from a row's window) and rows just
past a whole number of 512-element chunks; each rank-one fill shape that the
basis takes, into a tensor filled with NaN before.  The diagonal cells at orders
above 9, GL orders above 16 and off multiples of four, and tables that fit LDS
for one multipole only (order 14 with 29 points, order 16 with 26).

Tolerance: 1e-12 relative per element, the bar of the other tensor tests (every
value is a sum of at most about 16^2 positive terms, each rounded a few times).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import bs2e  # noqa: E402
from bs2e import capi  # noqa: E402
from bs2e.workloads import solve_h_max  # noqa: E402

# (order, B-splines, k_GL, max_k): n_pairs = n_b (2k - 1) - k (k - 1)
CASES = [(6, 5, 8, 3), (8, 8, 10, 2), (2, 9, 4, 0), (2, 40, 4, 1), (3, 30, 5, 0), (4, 21, 6, 2), (4, 64, 6, 0), (5, 33, 7, 6), (7, 35, 9, 8),
         (8, 40, 10, 4), (9, 39, 11, 16), (10, 41, 12, 2), (12, 40, 14, 1),
         (11, 25, 17, 9), (13, 17, 19, 5), (14, 16, 29, 4), (16, 17, 26, 2), (3, 12, 33, 12)]


def _fill_nan(rk):
    """Every byte of the tensor 0xff (a NaN), through the HIP runtime that the library runs on."""
    capi.lib()
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMemset.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
    ptr, n = rk.device_ptr()
    assert hip.hipMemset(ptr, 0xFF, 8 * n) == 0 and hip.hipDeviceSynchronize() == 0


def _knots(k, n_b):
    for r in (12.0, 20.0, 35.0, 6.0, 60.0):
        h = solve_h_max(k, 3, 2, r, n_b)
        if h is not None:
            return bs2e.generate_grid(k, 3, 2, h, r)
    # fewer splines than the geometric ramp takes: an even grid
    return np.concatenate([np.zeros(k), np.arange(1, n_b + 3 - k) * 0.4, np.full(k, (n_b + 3 - k) * 0.4)])


@pytest.mark.parametrize("k,n_b,k_GL,max_k", [(4, 21, 6, 2), (10, 21, 17, 5), (12, 16, 14, 3), (14, 16, 29, 1)])
def test_diagonal_containers_at_edges(k, n_b, k_GL, max_k, oracle):
    t = _knots(k, n_b)
    spl = bs2e.b_spline(k, t)
    r_k, r_m_k, r_d_k = (x().init(max_k, spl) for x in (bs2e.sparse_4d, bs2e.sparse_4d, bs2e.sparse_6d))
    bs2e.setup_Slater_integrals(spl, max_k, k_GL, r_k, r_m_k, r_d_k)
    ref = oracle.slater_diag(k, t, k_GL, max_k)["rdk"]
    assert np.all(np.abs(r_d_k.data - ref) <= 1e-12 * np.abs(ref))


@pytest.mark.parametrize("k,n_b,k_GL,max_k", [(2, 2, 4, 0), (2, 9, 4, 4), (5, 4, 7, 3), (8, 8, 10, 8), (9, 12, 14, 5),
                                              (11, 23, 17, 16), (14, 16, 29, 4), (16, 17, 26, 2)])
def test_window_moments_at_edges(k, n_b, k_GL, max_k, oracle):
    """One column and odd counts of columns, fewer splines than the order, multipoles in one and several chunks."""
    t = _knots(k, n_b)
    spl = bs2e.b_spline(k, t)
    r_k, r_m_k, r_d_k = (x().init(max_k, spl) for x in (bs2e.sparse_4d, bs2e.sparse_4d, bs2e.sparse_6d))
    bs2e.setup_Slater_integrals(spl, max_k, k_GL, r_k, r_m_k, r_d_k)
    ref = oracle.slater_off_diag(k, t, k_GL, max_k)
    for got, name in ((r_k, "rk"), (r_m_k, "rmk")):
        assert np.all(np.abs(got.data - ref[name]) <= 1e-12 * np.abs(ref[name])), name


@pytest.mark.parametrize("k,n_b,k_GL,max_k", CASES)
def test_fill_shapes_at_edges(k, n_b, k_GL, max_k, oracle):
    t = _knots(k, n_b)
    assert len(t) - k - 2 == n_b
    ref = oracle.rk_dense(k, n_b, max_k, oracle.slater_off_diag(k, t, k_GL, max_k),
                          oracle.slater_diag(k, t, k_GL, max_k))
    ctx = bs2e.Context(0)
    rk = bs2e.RkTensor.build(k, t, k_GL, max_k, ctx=ctx, compute=False)
    shapes = []
    for shape in range(16):
        try:
            rk.set_tuning(shape, 1)
        except bs2e.Bs2eError:
            continue
        _fill_nan(rk)
        rk.compute()
        R = rk.to_host()
        assert np.all(np.abs(R - ref) <= 1e-12 * np.abs(ref)), (shape, float(np.nanmax(np.abs(R - ref) / np.abs(ref))))
        shapes.append(shape)
    assert (len(shapes) == 7) == (rk.n_pairs * rk.K % 2 == 0) and shapes
    rk.release()
    ctx.close()


@pytest.mark.parametrize("max_k", [0, 1, 2])
@pytest.mark.parametrize("k", [2, 3])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_one_basis_function(k, max_k, precision, oracle):
    """Rows of one, two and three elements, none of them rank-one, by every shape that takes them and the default."""
    t = _knots(k, 1)
    assert len(t) - k - 2 == 1
    ref = oracle.rk_dense(k, 1, max_k, oracle.slater_off_diag(k, t, 6, max_k), oracle.slater_diag(k, t, 6, max_k))
    tol = 1e-12 if precision == "fp64" else 1e-10
    ctx = bs2e.Context(0)
    for shape in (None, *range(7)):
        rk = bs2e.RkTensor.build(k, t, 6, max_k, ctx=ctx, compute=False, precision=precision)
        try:
            if shape is not None:
                rk.set_tuning(shape, 1)
        except bs2e.Bs2eError:
            assert shape < 5 and rk.K % 2 == 1
            continue
        _fill_nan(rk)
        rk.compute()
        assert np.all(np.abs(rk.to_host() - ref) <= tol * np.abs(ref)), shape
        rk.release()
    ctx.close()
