"""The blocks the library keeps for streams: whose they are and how much they
hold, read from the device's free memory."""
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import d3s
    import hiprt
    d3s.lib()
    if hiprt.device_count() < 1:
        pytest.skip("no GPU")
    return d3s


class PerThread:
    ptr = 2  # hipStreamPerThread


def in_thread(fn):
    out = []

    def body():
        try:
            out.append(fn())
        except BaseException as e:  # raised again below
            out.append(e)
    t = threading.Thread(target=body)
    t.start()
    t.join()
    if isinstance(out[0], BaseException):
        raise out[0]
    return out[0]


def test_per_thread_stream_has_a_block_per_thread(gpu, oracle):
    """hipStreamPerThread is one handle for a stream of each thread's own, whose
    calls may overlap: a second thread's first call takes a block of its own,
    and a thread's release leaves the other's"""
    import hiprt
    N, V = 64, 40009
    rng = np.random.default_rng(1)
    x = (rng.standard_normal((N, V)) * 3).astype(np.float32)
    u = oracle.uniform(2, 1, N, V)
    exp = oracle.sample(x, u, 1.0, 0.9, n_threads=8, detail=False)["ids"]
    need = gpu.workspace_bytes(gpu.DTYPE_F32, N, V, V)
    assert need > 32 << 20  # far above what else the process allocates meanwhile
    go = [threading.Event() for _ in range(2)]
    held = []

    def call():
        free = hiprt.free_memory()
        got = gpu.sample(x, u, 1.0, 0.9, want_probs=False, stream=PerThread)
        assert got["rc"] == 0 and np.array_equal(got["ids"], exp)
        return free - hiprt.free_memory()

    def first():
        held.append(call())
        go[0].set()
        go[1].wait(60)
        held.append(call())  # its block is still there
        assert gpu.lib().d3s_stream_workspace_release(PerThread.ptr) == 0

    def second():
        took = call()
        assert gpu.lib().d3s_stream_workspace_release(PerThread.ptr) == 0
        return took

    t = threading.Thread(target=first)
    t.start()
    assert go[0].wait(60)
    try:
        took = in_thread(second)
    finally:
        go[1].set()
        t.join()
    assert len(held) == 2
    assert held[0] > 0.9 * need and abs(held[1]) < 0.5 * need
    assert took > 0.9 * need


def test_per_thread_stream_calls_beside_each_other(gpu, oracle):
    """two threads' calls on hipStreamPerThread at once: every call's ids are
    the oracle's"""
    import hiprt
    rng = np.random.default_rng(3)
    cases = []
    for V, k in ((151936, 30), (20001, 300), (20001, 20001)):
        x = (rng.standard_normal((6, V)) * 3).astype(np.float32)
        u = oracle.uniform(4, V + k, 6, k)
        cases.append((x, u, oracle.sample(x, u, 0.8, 0.9, n_threads=4, detail=False)["ids"]))
    errors = []

    def worker(order):
        try:
            bufs = [(hiprt.to_device(x), hiprt.to_device(u), hiprt.DeviceBuffer(4 * len(x))) for x, u, _ in cases]
            for rep in range(8):
                for i in order:
                    x, u, exp = cases[i]
                    bx, bu, ids = bufs[i]
                    N, V = x.shape
                    rc = gpu.sample_raw(bx.ptr, gpu.DTYPE_F32, N, V, V, bu.ptr, u.shape[1], 0.8, 0.9, None, ids.ptr,
                                        stream=PerThread.ptr)
                    hiprt.check(hiprt.hip().hipStreamSynchronize(PerThread.ptr), "synchronize")
                    if rc or not np.array_equal(ids.download((N,), np.int32), exp):
                        errors.append((rep, i, rc))
            gpu.lib().d3s_stream_workspace_release(PerThread.ptr)
        except Exception as e:  # reported below
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=(o,)) for o in ((0, 1, 2), (2, 1, 0))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("V,k,want_probs", [(32768, 100, False), (20011, 20011, False), (20011, 6000, True)])
def test_growing_calls_keep_little(gpu, V, k, want_probs):
    """a batch that grows a row at a time: the stream's block and the blocks it
    has outgrown, which stay until its release, hold a few times the last call's
    need (the sum of every call's need is over thirty times that)"""
    import hiprt
    N = 64
    need = gpu.workspace_bytes(gpu.DTYPE_F32, N, V, k)
    bx = hiprt.to_device(np.random.default_rng(5).standard_normal((N, V)).astype(np.float32))
    bu, ids = hiprt.to_device(np.random.default_rng(6).random((N, k), np.float32)), hiprt.DeviceBuffer(4 * N)
    probs, cand = hiprt.DeviceBuffer(4 * N * k), hiprt.DeviceBuffer(4 * N * k)
    s = hiprt.Stream()

    def call(n):
        assert gpu.sample_raw(bx.ptr, gpu.DTYPE_F32, n, V, V, bu.ptr, k, 1.0, 0.9, None, ids.ptr,
                              probs.ptr if want_probs else None, cand.ptr if want_probs else None, stream=s.ptr) == 0

    call(N)  # what the runtime itself takes with a stream's first launches
    assert gpu.lib().d3s_stream_workspace_release(s.ptr) == 0
    hiprt.synchronize()
    time.sleep(0.5)  # (freed memory shows in the count a little later)
    free = hiprt.free_memory()
    for n in range(1, N + 1):
        call(n)
    s.synchronize()
    held = free - hiprt.free_memory()
    assert gpu.lib().d3s_stream_workspace_release(s.ptr) == 0
    for _ in range(50):
        back = free - hiprt.free_memory()
        if back < 0.5 * need:
            break
        time.sleep(0.1)
    s.destroy()
    assert 0.5 * need < held < 4.5 * need + (8 << 20), (held, need)
    assert back < 0.5 * need + (4 << 20), (back, need)
