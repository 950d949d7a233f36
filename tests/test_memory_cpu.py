"""The library's device blocks, host copies and tuning without a device, over a stand-in
for the HIP runtime (fake_hip.cpp): each scenario in a process of its own, as the
stand-in has to be loaded before the library.
"""
import ctypes as C
import os
import subprocess
import sys
import threading
import time

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
K, K_GL, MAX_K = 4, 6, 2


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.cpp"), "-o", so,
                    "-lpthread"], check=True)
    return so


# ------------------------------------------------------------- in the process
def _load(so):
    sys.path.insert(0, os.path.join(ROOT, "b-spline-two-e_amd"))
    f = C.CDLL(so, mode=C.RTLD_GLOBAL)
    for name, res, args in (("fake_capacity", None, [C.c_size_t]), ("fake_used", C.c_size_t, []),
                            ("fake_mallocs", C.c_int64, []), ("fake_memcpys", C.c_int64, []),
                            ("fake_fail_new", None, [C.c_int]), ("fake_stream", C.c_void_p, [C.c_int]),
                            ("fake_block", None, [C.c_void_p, C.c_int]), ("fake_pinned", C.c_void_p, [C.c_size_t]),
                            ("fake_capture", None, [C.c_int]), ("fake_captures_ended", C.c_int, []),
                            ("fake_holds", C.c_int, [C.c_void_p, C.c_size_t])):
        getattr(f, name).restype = res
        getattr(f, name).argtypes = args
    import bs2e
    bs2e.capi.lib()
    return f, bs2e


def _knots(bs2e, r_max):
    return bs2e.generate_grid(K, 3, 2, 1.0, r_max)


def scenario_other_contexts_give_back(f, bs2e):
    """An allocation that fails takes what other contexts of the device keep."""
    a, b = bs2e.Context(0), bs2e.Context(0)
    t = _knots(bs2e, 40.0)
    rk = bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=a, compute=False)
    need = f.fake_used()
    rk.release()
    assert f.fake_used() == need          # kept
    f.fake_capacity(need + need // 2)
    bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=b, compute=False).release()
    s = bs2e.Server(need + need // 4, 1)      # a service's arena is one allocation
    s.close()


def scenario_other_devices_keep(f, bs2e):
    """Blocks kept on another device are left alone."""
    a, b = bs2e.Context(0), bs2e.Context(1)
    t = _knots(bs2e, 40.0)
    bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=a, compute=False).release()
    kept = f.fake_used()
    f.fake_capacity(kept + kept // 2)
    with pytest.raises(bs2e.Bs2eError):
        bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=b, compute=False)
    b.close()
    assert f.fake_used() == kept


def scenario_trim_gives_back(f, bs2e):
    """Context.trim returns what no handle holds, and nothing else."""
    ctx = bs2e.Context(0)
    t = _knots(bs2e, 40.0)
    held = bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=ctx, compute=False)
    used = f.fake_used()
    bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=ctx, compute=False).release()
    assert f.fake_used() > used
    ctx.trim()
    assert f.fake_used() == used
    held.release()
    ctx.close()
    assert f.fake_used() == 0


def scenario_host_memory_runs_out(f, bs2e):
    """Host allocations that fail in the middle of a call that only moves device
    blocks end in an error code or in a block given back, never in an exception."""
    ctx = bs2e.Context(0)
    t = _knots(bs2e, 20.0)
    rk = bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=ctx)
    n_b = len(t) - K - 2
    cfg = bs2e.count_configs(bs2e.sym(0), 1, n_b, K, n_b, n_b, 1)
    L, n = (C.c_int64 * 1)(0), (C.c_int64 * 1)(len(cfg))
    cfg = np.ascontiguousarray(cfg, np.int64)
    lib, codes = bs2e.capi.lib(), set()
    for fail_at in range(12):
        h = C.c_void_p()
        bs2e.capi.check(lib.bs2e_blockset_create(rk.handle, 1, L, n, cfg.ctypes.data_as(C.POINTER(C.c_int64)), 1,
                                                 C.byref(h)), ctx.handle)
        for size in (1000, 5000, 1000):     # (later rounds take kept blocks)
            f.fake_fail_new(fail_at)
            codes.add(lib.bs2e_blockset_reserve(h, size * (fail_at + 1), size * (fail_at + 1)))
            f.fake_fail_new(-1)
        f.fake_fail_new(fail_at)
        codes.add(lib.bs2e_blockset_release(h))
        f.fake_fail_new(-1)
    assert codes == {0, bs2e.capi.BS2E_ENOMEM}, codes
    rk.release()
    ctx.close()
    assert f.fake_used() == 0


def _write(rk, values):
    p, n = rk.device_ptr()
    assert n == values.size
    C.memmove(p, values.ctypes.data, values.nbytes)


def scenario_service_reads_overlap(f, bs2e):
    """A job's results are read while another slot's stream is busy, and while a
    thread waits for that slot's: long reads, middle ones and the copy out of the mirror."""
    s = bs2e.Server(1 << 30, 2)
    slot0 = f.fake_stream(2)              # streams: two of the service's own context, two of each slot
    t = _knots(bs2e, 80.0)
    f.fake_block(slot0, 1)
    a = s.submit(K, t, K_GL, MAX_K)
    b = s.submit(K, t, K_GL, MAX_K)
    s.wait(b)
    f.fake_block(slot0, 0)
    s.wait(a)
    ra, rb = s.tensor(a), s.tensor(b)
    va, vb = (np.random.default_rng(i).random(ra.device_ptr()[1]) for i in (0, 1))
    assert va.nbytes > 4 << 20
    _write(ra, va)
    _write(rb, vb)
    f.fake_block(slot0, 1)
    got = {}

    def read(name, rk):
        got[name] = rk.to_host().ravel()

    def middle(name, rk):
        out = np.empty((20, rk.n_pairs, rk.K))
        assert 16 << 10 < out.nbytes < 2 << 20
        bs2e.capi.check(bs2e.capi.lib().bs2e_rk_copy_rows(rk.handle, 0, 20, out.ctypes.data_as(C.POINTER(C.c_double))))
        got[name] = out.ravel()

    first = threading.Thread(target=read, args=("a", ra), daemon=True)
    first.start()
    time.sleep(0.3)                       # (it waits for its slot's stream)
    others = [threading.Thread(target=w, args=(n, rb), daemon=True) for w, n in ((middle, "m"), (read, "b"))]
    for th in others:
        th.start()
        th.join(20)
        assert not th.is_alive()
    assert first.is_alive()
    assert np.array_equal(got["b"], vb) and np.array_equal(got["m"], vb[:got["m"].size])
    f.fake_block(slot0, 0)
    first.join(20)
    assert np.array_equal(got["a"], va)
    s.close()


def scenario_many_threads_read_one_context(f, bs2e):
    """Reads of several tensors of one context from a thread each arrive whole."""
    ctx = bs2e.Context(0)
    rks = [bs2e.RkTensor.build(K, _knots(bs2e, r), K_GL, MAX_K, ctx=ctx) for r in (80.0, 90.0, 60.0, 30.0)]
    vals = [np.random.default_rng(i).random(rk.device_ptr()[1]) for i, rk in enumerate(rks)]
    for rk, v in zip(rks, vals):
        _write(rk, v)
    bad = []

    def read(rk, v):
        for _ in range(5):
            rk.compute()                  # (drops the mirror)
            if not np.array_equal(rk.to_host().ravel(), v):
                bad.append(v.size)

    threads = [threading.Thread(target=read, args=p) for p in zip(rks, vals)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad
    for rk in rks:
        rk.release()
    ctx.close()


def scenario_uploads_longer_than_the_ring(f, bs2e):
    """Containers of more than eight buffers of 8 MiB reach the device byte for byte."""
    ctx = bs2e.Context(0)
    k, max_k = 8, 9
    t = bs2e.generate_grid(k, 3, 2, 0.5, 60.0)
    spl = bs2e.b_spline(k, t)
    r_k, r_m_k, r_d_k = (x().init(max_k, spl) for x in (bs2e.sparse_4d, bs2e.sparse_4d, bs2e.sparse_6d))
    rng = np.random.default_rng(5)
    for x in (r_k, r_m_k, r_d_k):
        x.data = np.asfortranarray(rng.random(x.data.shape))
    r_d_k.i_p = rng.integers(0, 1 << 40, r_d_k.nnz)
    assert r_d_k.data.nbytes + 40 * r_d_k.nnz > 64 << 20
    R = bs2e.Nd_DOK()
    bs2e.compute_R_K_map(r_d_k, r_k, r_m_k, spl, max_k, R, ctx=ctx)
    for x in (r_k, r_m_k, r_d_k):         # (the blocks are kept, with what was uploaded)
        flat = x.data.ravel(order="F")
        assert f.fake_holds(flat.ctypes.data, flat.nbytes)
    cols = np.concatenate([r_d_k.iv, r_d_k.i, r_d_k.i_p, r_d_k.j, r_d_k.j_p])
    assert f.fake_holds(cols.ctypes.data, cols.nbytes)


def scenario_pinned_arrays_are_copied_straight(f, bs2e):
    """A long result for a pinned array is one copy into it; a pageable one takes the ring and arrives whole."""
    ctx = bs2e.Context(0)
    rk = bs2e.RkTensor.build(K, _knots(bs2e, 80.0), K_GL, MAX_K, ctx=ctx)
    v = np.random.default_rng(3).random(rk.device_ptr()[1])
    assert v.nbytes > 4 << 20
    _write(rk, v)
    P = C.POINTER(C.c_double)

    def copies(address):
        n = f.fake_memcpys()
        bs2e.capi.check(bs2e.capi.lib().bs2e_rk_copy_rows(rk.handle, 0, rk.n_pairs, C.cast(address, P)))
        return f.fake_memcpys() - n

    pinned, page = f.fake_pinned(v.nbytes), np.zeros(v.size)
    assert copies(pinned) == 1
    assert copies(page.ctypes.data) > 1
    got = np.ctypeslib.as_array(C.cast(pinned, P), (v.size,))
    assert np.array_equal(got, v) and np.array_equal(page, v)


def scenario_tuning_keeps_the_default(f, bs2e):
    """Where every candidate takes the same time (as all do here), the autotuner leaves the
    multipole chunk of an untuned build, also one that is no power of two and not the largest."""
    ctx = bs2e.Context(0)
    t = bs2e.generate_grid(6, 3, 2, 1.0, 280.0)
    rk = bs2e.RkTensor.build(6, t, 8, 16, ctx=ctx, compute=False)
    untuned = rk.tuning()[1]
    assert untuned == 12
    rk.autotune(force=True)
    assert rk.tuning()[1] == untuned
    other = bs2e.RkTensor.build(6, t, 8, 16, ctx=ctx, compute=False)
    other.autotune()                      # (taken from what the process has timed)
    assert other.tuning()[1] == untuned


def scenario_releases_spare_captures(f, bs2e):
    """Handles made and released, and the calls that do so inside, leave stream captures of the
    process alone; the device is waited for all the same before a block is taken again."""
    ctx = bs2e.Context(0)
    t = _knots(bs2e, 40.0)
    spl = bs2e.b_spline(K, t)
    f.fake_capture(1)
    rk = bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=ctx)
    rk.to_host()
    rk.release()
    kept = f.fake_mallocs()
    bs2e.setup_S(spl, K_GL, ctx=ctx)
    bs2e.setup_H_one_particle(2, (2, 10.0, 0.0), range(3), spl, K_GL, ctx=ctx)
    rk = bs2e.RkTensor.build(K, t, K_GL, MAX_K, ctx=ctx)
    assert not f.fake_captures_ended()
    f.fake_capture(0)
    other = f.fake_stream(1)                     # (not the stream that the context builds on)
    f.fake_block(other, 1)
    th = threading.Thread(target=rk.release, daemon=True)
    th.start()
    th.join(0.5)
    assert th.is_alive()
    f.fake_block(other, 0)
    th.join(20)
    assert not th.is_alive() and f.fake_mallocs() < kept + 20
    ctx.close()
    assert f.fake_used() == 0


def scenario_threads_share_a_context(f, bs2e):
    """Handles made and released by several threads on one context leave nothing behind."""
    ctx = bs2e.Context(0)

    def work(i):
        for j in range(60):
            rk = bs2e.RkTensor.build(K, _knots(bs2e, 8.0 + i + j % 7), K_GL, MAX_K, ctx=ctx, compute=False)
            rk.release()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    ctx.close()
    assert f.fake_used() == 0


SCENARIOS = [n[len("scenario_"):] for n in list(globals()) if n.startswith("scenario_")]


@pytest.mark.parametrize("name", SCENARIOS)
def test_scenario(name, fake):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake, name], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:]


if __name__ == "__main__":
    globals()["scenario_" + sys.argv[2]](*_load(sys.argv[1]))
