"""The device blocks that a context keeps and its copies to the host: a tensor
built in a released (and poisoned) block holds the values of one built in fresh
memory, also when several threads build and release on contexts of their own; copies from
a few bytes to several pinned buffers arrive whole.  Bit for bit (the same
kernels on the same inputs)."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import bs2e  # noqa: E402
from bs2e import capi  # noqa: E402
from bs2e.workloads import perturb_breakpoints  # noqa: E402


def _poison(rk):
    capi.lib()
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMemset.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
    ptr, n = rk.device_ptr()
    assert hip.hipMemset(ptr, 0xFF, 8 * n) == 0 and hip.hipDeviceSynchronize() == 0


# tensors of 80 KB, 1.4 MB, 17 MB (ring of small buffers) and 112 MB (ring filled more than once)
SIZES = [(2, 6.0, 4, 0), (4, 8.0, 6, 2), (8, 15.0, 14, 4), (8, 60.0, 12, 7)]


@pytest.mark.parametrize("k,r_max,k_GL,max_k", SIZES)
def test_kept_blocks_and_copies(k, r_max, k_GL, max_k):
    grid = bs2e.generate_grid(k, 3, 2, 1.0, r_max)
    bases = [perturb_breakpoints(grid, k, seed) for seed in (1, 2, 3)]
    ref = []
    for t in bases:
        fresh = bs2e.Context(0)
        rk = bs2e.RkTensor.build(k, t, k_GL, max_k, ctx=fresh)
        ref.append(rk.to_host())
        rows = rk.rows([0, rk.n_pairs - 1])
        assert np.array_equal(rows, ref[-1][[0, -1]])
        rk.release()
        fresh.close()
    ctx = bs2e.Context(0)
    for i in (0, 1, 2, 0):
        rk = bs2e.RkTensor.build(k, bases[i], k_GL, max_k, ctx=ctx)
        assert np.array_equal(rk.to_host(), ref[i])
        _poison(rk)
        rk.release()
    bad = []

    def work(i):
        mine = bs2e.Context(0)
        for _ in range(3):
            rk = bs2e.RkTensor.build(k, bases[i], k_GL, max_k, ctx=mine)
            if not np.array_equal(rk.to_host(), ref[i]):
                bad.append(i)
            rk.release()
        mine.close()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad
    ctx.close()
