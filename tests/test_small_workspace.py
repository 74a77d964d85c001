"""A workspace that holds few of a call's rows: the call takes it when the rows'
rounds of launches are worth it, and else runs as it does without one.  The
launches are read from a captured graph; every form gives the oracle's bits."""
import ctypes

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


# rows, V, k, probabilities, workspace (None: d3s_sample_noalloc), kernel nodes at most
CASES = [
    (300, 20001, 100, False, None, 1), (300, 20001, 100, False, 520 << 10, 1), (300, 8193, 65, True, 2 << 20, 1),
    (40, 40001, 6000, False, None, 1), (40, 40001, 6000, True, 4 << 20, 1),
    # few rounds, still worth it
    (3, 60001, 100, False, None, 12), (2, 151936, 8000, False, 4 << 20, 12), (2, 151936, 8000, True, 4 << 20, 22),
    # beyond the streaming kernel's k: the sort, or the wide nucleus kernels where they take no more time
    (6, 40001, 40001, False, 4_708_352, 9), (6, 40001, 40001, False, None, 12)]


@pytest.mark.parametrize("N,V,k,want_probs,ws_bytes,nodes", CASES)
def test_launches(gpu, oracle, N, V, k, want_probs, ws_bytes, nodes):
    import hiprt
    H = hiprt.hip()
    x = (np.random.default_rng(V + k).standard_normal((N, V)) * 3).astype(np.float32)
    u = oracle.uniform(7, 1, N, k)
    bx, bu, ids = hiprt.to_device(x), hiprt.to_device(u), hiprt.DeviceBuffer(4 * N)
    probs, cand = hiprt.DeviceBuffer(4 * N * k), hiprt.DeviceBuffer(4 * N * k)
    ws = gpu.Workspace(ws_bytes) if ws_bytes else None
    s = hiprt.Stream()
    hiprt.synchronize()
    graph = ctypes.c_void_p()
    hiprt.check(H.hipStreamBeginCapture(s.ptr, 0), "begin capture")
    args = (bx.ptr, gpu.DTYPE_F32, N, V, V, bu.ptr, k, 0.9, 0.9, None, ids.ptr) + (
        (probs.ptr, cand.ptr) if want_probs else (None, None))
    how = dict(workspace=ws.arg()) if ws else dict(noalloc=True)
    rc = gpu.sample_raw(*args, stream=s.ptr, **how)
    hiprt.check(H.hipStreamEndCapture(s.ptr, ctypes.byref(graph)), "end capture")
    got = len(hiprt.graph_node_types(graph))
    H.hipGraphDestroy(graph)
    assert rc == 0 and got <= nodes, got
    assert gpu.sample_raw(*args, stream=s.ptr, **how) == 0
    s.synchronize()
    exp = oracle.sample(x, u, 0.9, 0.9, n_threads=8)
    assert np.array_equal(ids.download((N,), np.int32), exp["ids"])
    if want_probs:
        assert np.array_equal(probs.download((N, k), np.float32), exp["probs"])
        assert np.array_equal(cand.download((N, k), np.int32), exp["cand"])
    s.destroy()
