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


def test_blocks_between_streams():
    """A block released while its builds still run on one of the caller's streams is the next
    tensor's on another: neither holds the other's values."""
    capi.lib()
    hip = C.CDLL("libamdhip64.so.7")
    streams = [C.c_void_p() for _ in range(2)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    k, k_GL, max_k = 8, 12, 7
    grid = bs2e.generate_grid(k, 3, 2, 1.0, 60.0)
    bases = [perturb_breakpoints(grid, k, seed) for seed in (4, 5)]
    ref = []
    for t in bases:
        fresh = bs2e.Context(0)
        ref.append(bs2e.RkTensor.build(k, t, k_GL, max_k, ctx=fresh).to_host())
    ctx = bs2e.Context(0)
    last = None
    for i in range(6):
        ctx.set_stream(streams[i % 2].value)
        rk = bs2e.RkTensor.build(k, bases[i % 2], k_GL, max_k, ctx=ctx)
        ptr = rk.device_ptr()[0]
        assert last in (None, ptr)     # the block was kept and taken again
        last = ptr
        if i >= 3:
            assert np.array_equal(rk.to_host(), ref[i % 2])
        for _ in range(20):
            rk.compute()
        rk.release()                   # (twenty builds are still enqueued)
    ctx.set_stream(None)
    ctx.close()
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0


@pytest.mark.parametrize("mode,thread", [(1, True), (2, False), (2, True)])
def test_releases_spare_captures(mode, thread):
    """A stream capture (1: of its thread, 2: relaxed) is not ended by handles that are made and
    released meanwhile, where the mode lets them be."""
    capi.lib()
    hip = C.CDLL("libamdhip64.so.7")
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    ctx = bs2e.Context(0)
    t = bs2e.generate_grid(4, 3, 2, 1.0, 20.0)

    def calls():
        for _ in range(3):
            rk = bs2e.RkTensor.build(4, t, 6, 2, ctx=ctx)
            rk.release()
        bs2e.setup_S(bs2e.b_spline(4, t), 6, ctx=ctx)

    calls()
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    if thread:
        th = threading.Thread(target=calls)
        th.start()
        th.join()
    else:
        calls()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipStreamDestroy(stream) == 0
    ctx.close()
