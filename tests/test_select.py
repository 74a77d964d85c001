"""The selecting kernels (64 < k <= 4096 on rows longer than 8192, and small k
on rows wider than the segmented kernel's) and the wide nucleus kernels (k >
4096, ids only) against the oracle, bit for bit:
row lengths at segment and chunk edges, row starts off 16 bytes, k at its
limits, ties across the k-th place, rows the kernels leave to the generic
procedure, and every workspace mode."""
import numpy as np
import pytest

import d3s_workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import d3s
    import hiprt
    d3s.lib()
    if hiprt.device_count() < 1:
        pytest.skip("no GPU")
    return d3s


def rows(rng, N, stride, dtype, sigma=3.0):
    x = (rng.standard_normal((N, stride)) * sigma).astype(np.float32)
    return x if dtype == "f32" else W.f32_to_bf16_bits(x)


def check(gpu, oracle, x, u, T, P, **kw):
    okw = {a: b for a, b in kw.items() if a in ("banned", "vocab")}
    exp = oracle.sample(x, u, T, P, **okw)
    got = gpu.sample(x, u, T, P, **kw)
    assert got["rc"] == 0
    assert np.array_equal(got["ids"], exp["ids"])
    if kw.get("want_probs", True):
        assert np.array_equal(got["cand"], exp["cand"])
        assert np.array_equal(got["probs"], exp["probs"], equal_nan=True)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N,V,k,T,P", [
    (1, 8193, 65, 1.0, 0.95), (3, 8197, 1000, 0.7, 0.9), (2, 16384, 4096, 1.0, 1.0), (5, 20001, 129, 0.6, 0.5),
    (1, 151936, 4095, 1.0, 0.95), (33, 32771, 200, 1.3, 0.99), (2, 270001, 64, 1.0, 0.9), (1, 700001, 1, 1.0, 0.9)])
def test_shapes(gpu, oracle, dtype, N, V, k, T, P):
    rng = np.random.default_rng([N, V, k])
    check(gpu, oracle, rows(rng, N, V, dtype), oracle.uniform(3, 1, N, k), T, P)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_strided_banned_per_row(gpu, oracle, dtype):
    rng = np.random.default_rng(5)
    N, V, k = 9, 12345, 300
    x = rows(rng, N, V + 7, dtype)
    T = np.array([0.7, 1.0, 0.0, 1e-4, 2.0 ** -21, 2.0 ** 22, 50.0, 1.0, 0.9], np.float32)
    P = np.array([0.9, 0.0, 0.5, 1.0, 1.5, 0.95, 0.3, 0.999, 0.7], np.float32)
    ban = np.array([0, -1, V - 1, V, 17, 5, -1, 12000, 1], np.int32)
    check(gpu, oracle, x, oracle.uniform(4, 1, N, k), T, P, banned=ban, vocab=V)


def test_ties_and_special_rows(gpu, oracle):
    rng = np.random.default_rng(6)
    V, k = 30011, 500
    x = rng.standard_normal((14, V)).astype(np.float32) * 2
    x[0] = 1.5                                   # all equal: more keys than LDS holds
    x[1] = np.round(x[1])                        # ties by the thousand
    x[2] = np.round(x[2] * 8) / 8                # ties across the k-th place
    x[3, 100:] = -np.inf                         # fewer finite values than k
    x[4] = -np.inf
    x[5, 777] = np.nan
    x[6, 29000] = np.inf
    x[7] *= 1e30                                 # nearly all elements far below the max
    x[8] *= 1e-30
    x[9] = 0.0
    x[9, ::2] = -0.0
    x[10] = x[10] * 0.01 + 1e6                   # a large offset: x - m in few steps
    x[11] = -np.abs(x[11]) - 1e4
    x[12] = np.sort(x[12])[::-1]                 # the top k in one segment
    x[13] = 3e38 * np.sign(x[13])
    check(gpu, oracle, x, oracle.uniform(8, 1, 14, k), 1.0, 0.9)
    check(gpu, oracle, x, oracle.uniform(8, 2, 14, k), 0.7, 0.5)
    T = np.full(14, np.inf, np.float32)
    T[7:] = np.nan
    check(gpu, oracle, x[:3], oracle.uniform(8, 3, 3, k), T[:3], 0.9)
    check(gpu, oracle, x[7:9], oracle.uniform(8, 3, 2, k), T[7:9], 0.9)


def test_zero_and_one_uniforms(gpu, oracle):
    rng = np.random.default_rng(7)
    x = rows(rng, 3, 9000, "f32")
    u = np.zeros((3, 100), np.float32)
    u[1] = np.float32(1) - np.float32(2.0 ** -24)
    u[2, 50:] = 0.25
    check(gpu, oracle, x, u, 1.0, 0.8)


def test_workspace_modes_agree(gpu, oracle):
    """the query's workspace, one that holds a row at a time, none (the streaming
    kernel), and the allocation-free entry point: the same bits"""
    rng = np.random.default_rng(8)
    N, V, k = 5, 60001, 700
    x, u = rows(rng, N, V, "bf16"), oracle.uniform(9, 1, N, k)
    need = gpu.workspace_bytes(gpu.DTYPE_BF16, N, V, k)
    one = gpu.workspace_bytes(gpu.DTYPE_BF16, 1, V, k)
    assert 0 < one < need
    for nbytes in (need, one, 300 << 10):
        ws = gpu.Workspace(nbytes)
        check(gpu, oracle, x, u, 0.8, 0.95, workspace=ws)
        check(gpu, oracle, x, u, 0.8, 0.95, workspace=ws, want_probs=False)
        ws.free()
    check(gpu, oracle, x, u, 0.8, 0.95, workspace=(None, 0))
    check(gpu, oracle, x, u, 0.8, 0.95, noalloc=True)
    check(gpu, oracle, x, u, 0.8, 0.95, flags=gpu.FLAG_GENERIC)


@pytest.mark.parametrize("own_workspace", [True, False, None])
def test_captured_and_replayed(gpu, oracle, own_workspace):
    """d3s_sample_ws (the selecting kernels) and d3s_sample on a stream that has
    no block yet (nothing is allocated under capture: the streaming kernel),
    captured and replayed with new inputs between the replays; None: a stream
    whose block is large enough, released before the replays (a graph does not
    hold it)"""
    import ctypes
    import hiprt
    H = hiprt.hip()
    N, V, k = 3, 20011, 150
    bx, bu, bids = hiprt.DeviceBuffer(4 * N * V), hiprt.DeviceBuffer(4 * N * k), hiprt.DeviceBuffer(4 * N)
    s = hiprt.Stream()
    ws = gpu.Workspace(gpu.workspace_bytes(gpu.DTYPE_F32, N, V, k)) if own_workspace else None
    if own_workspace is None:
        bx.upload(rows(np.random.default_rng(9), N, V, "f32"))
        bu.upload(oracle.uniform(1, 9, N, k))
        assert gpu.sample_raw(bx.ptr, gpu.DTYPE_F32, N, V, V, bu.ptr, k, 0.8, 0.9, None, bids.ptr, stream=s.ptr) == 0
    hiprt.synchronize()
    graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
    hiprt.check(H.hipStreamBeginCapture(s.ptr, 0), "begin capture")
    rc = gpu.sample_raw(bx.ptr, gpu.DTYPE_F32, N, V, V, bu.ptr, k, 0.8, 0.9, None, bids.ptr, stream=s.ptr,
                        workspace=ws.arg() if ws else None)
    hiprt.check(H.hipStreamEndCapture(s.ptr, ctypes.byref(graph)), "end capture")
    assert rc == 0
    assert set(hiprt.graph_node_types(graph)) == {"kernel"}
    if own_workspace is None:  # the streaming kernel alone
        assert len(hiprt.graph_node_types(graph)) == 1
        assert gpu.lib().d3s_stream_workspace_release(s.ptr) == 0
    hiprt.check(H.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0), "instantiate")
    try:
        for rep in range(4):
            x, u = rows(np.random.default_rng(rep), N, V, "f32"), oracle.uniform(1, rep, N, k)
            bx.upload(x)
            bu.upload(u)
            hiprt.synchronize()
            hiprt.check(H.hipGraphLaunch(exe, s.ptr), "graph launch")
            s.synchronize()
            assert np.array_equal(bids.download((N,), np.int32), oracle.sample(x, u, 0.8, 0.9)["ids"]), rep
            # an eager call between the replays
            check(gpu, oracle, x, u, 0.8, 0.9, want_probs=False)
    finally:
        H.hipGraphExecDestroy(exe)
        H.hipGraphDestroy(graph)
        gpu.lib().d3s_stream_workspace_release(s.ptr)
        s.destroy()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("sigma", [0.1, 1.0, 3.0, 8.0])
def test_ids_only_large_k_gathers_the_kept_ranks(gpu, oracle, dtype, sigma):
    """k > 4096, ids only (the wide nucleus kernels):
    every top_p from 0 to beyond 1, temperatures, banned indices, strides"""
    rng = np.random.default_rng([int(sigma * 10), dtype == "f32"])
    V = 24007
    P = np.array([0.0, 0.1, 0.5, 0.9, 0.95, 0.99, 0.9999, 1.0, 1.5, -1.0, np.nan], np.float32)
    N = len(P)
    x = rows(rng, N, V + 3, dtype, sigma)
    ban = np.where(rng.random(N) < 0.5, rng.integers(0, V, N), -1).astype(np.int32)
    for T, k in ((1.0, V), (0.7, 17000), (np.linspace(0.3, 2.0, N).astype(np.float32), V), (1.3, 5000)):
        check(gpu, oracle, x, oracle.uniform(11, 1, N, k), T, P, banned=ban, vocab=V, want_probs=False)


def test_ids_only_large_k_special_rows(gpu, oracle):
    rng = np.random.default_rng(12)
    V = 20480
    x = (rng.standard_normal((12, V)) * 3).astype(np.float32)
    x[0] = 2.0
    x[1] = np.round(x[1])
    x[2, 10:] = -np.inf
    x[3] = -np.inf
    x[4, 5] = np.nan
    x[5, V - 1] = np.inf
    x[6] = x[6] * 0.01 + 1e7      # lse rounds in whole units: no bound on the cut
    x[7] *= 1e30
    x[8, 7] = 60.0                # one element holds all the mass
    x[9] = np.sort(x[9])
    x[10, ::2] = -0.0
    x[10, 1::2] = 0.0
    x[11, 1000:] = -1e30
    u = oracle.uniform(13, 1, 12, V)
    for T in (1.0, 0.7, np.inf):
        check(gpu, oracle, x, u, T, 0.9, want_probs=False)
    check(gpu, oracle, x, u[:, :6000], 0.9, 0.95, want_probs=False)
    check(gpu, oracle, x, u[:, :6000], 0.9, 0.95)
    # kept ranks that cannot win: a dropped rank far past them does
    u = u.copy()
    u[:, :15000] = 0.0
    check(gpu, oracle, x, u, 1.0, 0.9, want_probs=False)
    u[:, :] = 0.0
    check(gpu, oracle, x, u, 1.0, 0.9, want_probs=False)
    u[:, 3:] = 1.0
    check(gpu, oracle, x, u, 1.0, 0.2, want_probs=False)
    u[:] = 2.0
    u[:, 20000] = 0.5
    check(gpu, oracle, x, u, 1.0, 0.2, want_probs=False)


def test_sorting_workspace_modes_agree(gpu, oracle):
    """the query's workspace, one that holds only the sort's keys (what the call
    requires), and the allocation-free entry point"""
    rng = np.random.default_rng(14)
    N, V = 3, 40009
    x, u = rows(rng, N, V, "bf16"), oracle.uniform(9, 1, N, V)
    need = gpu.workspace_bytes(gpu.DTYPE_BF16, N, V, V)
    plain = (256 << 10) + N * (2 * ((V + 63) & ~63) * 8 + 6 * 16 * 256 * 4 + 16 * 64 + 2 * 40 * 8)
    assert plain < need
    for nbytes in (need, plain):
        ws = gpu.Workspace((nbytes + 255) & ~255)
        check(gpu, oracle, x, u, 0.8, 0.95, workspace=ws, want_probs=False)
        check(gpu, oracle, x, u, 0.8, 0.95, workspace=ws)
        ws.free()
    check(gpu, oracle, x, u, 0.8, 0.95, noalloc=True, want_probs=False)
    u = u[:, :9000]
    check(gpu, oracle, x, u, 0.8, 0.95, noalloc=True, want_probs=False)
    check(gpu, oracle, x, u, 0.8, 0.95, workspace=(None, 0), want_probs=False)


@pytest.mark.parametrize("k", [100, 6000, 20001])
def test_head_with_its_logits_in_the_workspace(gpu, k):
    """the heads' logits lie in the workspace behind the sample's part when the
    caller keeps none: the routes that use a workspace when they have one must
    not take that part for theirs"""
    rng = np.random.default_rng(k)
    N, K, V = 8, 128, 20001
    x = W.f32_to_bf16_bits(rng.standard_normal((N, K)).astype(np.float32))
    w = W.f32_to_bf16_bits((rng.standard_normal((V, K)) * 0.2).astype(np.float32))
    u = rng.random((N, k)).astype(np.float32)
    for want_probs in (True, False):
        kept = gpu.linear_sample_bf16(x, w, u, 1.0, 0.9, want_probs=want_probs)
        got = gpu.linear_sample_bf16(x, w, u, 1.0, 0.9, want_probs=want_probs, keep_logits=False)
        assert kept["rc"] == 0 and got["rc"] == 0
        for name in ("ids", "cand", "probs") if want_probs else ("ids",):
            assert np.array_equal(kept[name], got[name]), name


def test_small_k_leaves_the_workspace(gpu, oracle):
    """k up to 64: the size query says 0, and a workspace given all the same is
    not written"""
    import hiprt
    N, V, k = 2, 700001, 20
    x, u = rows(np.random.default_rng(15), N, V, "f32"), oracle.uniform(5, 1, N, k)
    assert gpu.workspace_bytes(gpu.DTYPE_F32, N, V, k) == 0
    fill = np.full(16 << 18, 0x5a5a5a5a, np.uint32)
    ws, bx, bu, bids = hiprt.to_device(fill), hiprt.to_device(x), hiprt.to_device(u), hiprt.DeviceBuffer(4 * N)
    assert gpu.sample_raw(bx.ptr, gpu.DTYPE_F32, N, V, V, bu.ptr, k, 0.8, 0.9, None, bids.ptr,
                          workspace=(ws.ptr, fill.nbytes)) == 0
    hiprt.synchronize()
    assert np.array_equal(bids.download((N,), np.int32), oracle.sample(x, u, 0.8, 0.9)["ids"])
    assert np.array_equal(ws.download(fill.shape, np.uint32), fill)


def crowded_rows(rng, V, dtype):
    """rows whose k-th element is one of thousands in one place, or far below
    the first"""
    x = rows(rng, 12, V, "f32")
    fmin = np.float32(-3.3e38)
    few = rng.random((12, V)) < 40.0 / V
    x[0] = np.where(few[0], x[0], -np.inf)       # masked: nearly every rank is -inf
    x[1] = np.where(few[1], x[1], fmin)          # by the type's lowest values (-inf after / 0.7)
    x[2] = np.where(few[2], x[2], -1e4)
    x[3] = np.where(rng.random(V) < 0.5, np.where(few[3], x[3], fmin), -np.inf)  # two kinds of mask
    x[4] = np.round(x[4])
    x[5] = np.round(x[5] / 4) * 4
    x[6] = 1.5
    x[6, V // 2] = 1.5 + 2.0 ** -7
    x[7] = x[7] * 100                            # a wide scale
    x[8] = x[8] * 1e-3 + 1000                    # the last places of a large offset
    x[9] = np.where(few[9], 30.0, -x[9] ** 2 * 1e5)  # the rest 0 to some millions down
    x[10] = np.where(few[10], x[10], -(np.arange(V) // 900) - 50.0)  # ties in runs, the last ones first
    x[11] = np.round(x[11] * 2) / 2
    x[11, ::3] = -np.inf
    return x if dtype == "f32" else W.f32_to_bf16_bits(x)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V,k", [(8193, 65), (8193, 4096), (30011, 1000), (61003, 4096), (151936, 1025)])
def test_crowded_and_far(gpu, oracle, dtype, V, k):
    """the k-th element's bucket of more elements than LDS holds, or tens to
    millions of units below the first, at temperatures from the smallest on"""
    rng = np.random.default_rng([V, k])
    x = crowded_rows(rng, V, dtype)
    u = oracle.uniform(21, V, len(x), k)
    for T in (1.0, 0.7, 0.1, 0.0, 40.0):
        check(gpu, oracle, x, u, T, 0.9)
    ban = np.where(np.arange(12) % 2, 0, V - 1).astype(np.int32)
    check(gpu, oracle, x, u, 0.3, 1.0, banned=ban)


@pytest.mark.parametrize("T", [1e-5, 0.05, 0.3])
def test_small_temperatures(gpu, oracle, T):
    rng = np.random.default_rng(22)
    for V, k, dtype in ((8193, 300, "f32"), (50021, 4096, "bf16"), (700001, 64, "bf16")):
        check(gpu, oracle, rows(rng, 3, V, dtype), oracle.uniform(23, V, 3, k), T, 0.95)
    # the sorting path's front
    for k in (5000, 24000):
        check(gpu, oracle, rows(rng, 3, 50021, "f32"), oracle.uniform(24, k, 3, k), T, 0.95)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N,V,k,step", [(3, 8193, 500, 1.0), (2, 20011, 4096, 1.0), (2, 40003, 4000, 0.25), (3, 9001, 1024, 4.0),
                                        (2, 30001, 2500, 2.0 ** -7)])
def test_quantised_logits(gpu, oracle, dtype, N, V, k, step):
    """logits of few different values: the gathered keys crowd in k_sel_sort's
    buckets and go through its radix sort, 1 to 4 passes of it"""
    rng = np.random.default_rng([V, k])
    x = (np.round(rng.standard_normal((N, V)) * 3 / step) * step).astype(np.float32)
    x[0, :40] += 9.5
    x[-1] -= 100.25  # below zero, the last places in use at T = 0.7
    x = x if dtype == "f32" else W.f32_to_bf16_bits(x)
    u = oracle.uniform(25, V, N, k)
    for T in (1.0, 0.7):
        check(gpu, oracle, x, u, T, 0.97)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V,k", [(8200, 8200), (24007, 24007), (24007, 5000), (100003, 100003)])
def test_ids_only_small_temperatures_and_whole_rows(gpu, oracle, dtype, V, k):
    """the wide nucleus kernels where the cut's bounds are hard to come by: T
    from the smallest on (lse of some millions), top_p at and about 1 (cuts in the
    last elements of any mass, or none), crowded and masked rows"""
    rng = np.random.default_rng([V, k])
    x = crowded_rows(rng, V, dtype)
    u = oracle.uniform(31, k, len(x), k)
    eps = np.float32(2.0 ** -24)
    P = np.array([0.9, 1.0, 1 - eps, 1 + 2 * eps, 0.99999, 0.0, 0.5, 1.0, 1.0, 1.0, 1.0, 0.999], np.float32)
    for T in (0.0, 0.1, 0.4, 1.0, 30.0):
        check(gpu, oracle, x, u, T, P, want_probs=False)
    ban = np.where(np.arange(12) % 2, 5, V - 1).astype(np.int32)
    check(gpu, oracle, x, u, 0.0, 1.0, banned=ban, want_probs=False)
    check(gpu, oracle, x[:5], u[:5], 1.0, 1.0, want_probs=False)  # (short bf16 rows: sorted)
    check(gpu, oracle, x[5:], u[5:], 1.0, 1.5, want_probs=False)
    x = rows(rng, 24, V, dtype)  # (rounding decides whether the prefix passes 1)
    check(gpu, oracle, x, oracle.uniform(32, k, 24, k), np.linspace(0.2, 2.0, 24).astype(np.float32), 1.0,
          want_probs=False)


def test_ids_only_many_rows(gpu, oracle):
    """more rows than CUs (k_nuc_final's other form)"""
    rng = np.random.default_rng(35)
    N, V = 300, 8200
    x = rows(rng, N, V, "bf16", 1.0)
    x[::3] = W.f32_to_bf16_bits(np.round(rng.standard_normal((100, V)) * 2).astype(np.float32))
    u = oracle.uniform(36, 1, N, V)
    P = np.where(np.arange(N) % 2, 1.0, 0.9).astype(np.float32)
    check(gpu, oracle, x, u, 0.7, P, want_probs=False)


def test_ids_only_winners_in_large_sets(gpu, oracle):
    """the race won in a set of thousands of equal or nearly equal elements, by
    rank: uniforms so small that those ranks win over all others"""
    V = 40009
    rng = np.random.default_rng(33)
    x = np.stack([np.full(V, 2.0), np.round(rng.standard_normal(V) * 2), 1 + rng.random(V) * 1e-3,
                  rng.standard_normal(V) * 1e-2]).astype(np.float32)
    for at in (0, 1, 777, 20000, 39000):
        u = oracle.uniform(34, at, 4, V)
        u[:, at] = np.float32(2.0 ** -24)
        u[:, at + 5] = np.float32(2.0 ** -23)
        for T, P in ((1.0, 1.0), (0.5, 0.98), (1.0, 0.5)):
            check(gpu, oracle, x, u, T, P, want_probs=False)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_ids_only_where_no_rank_scores(gpu, oracle, dtype):
    """uniforms for which every score counts as -1: the first rank; and one rank
    that does score, kept or dropped"""
    rng = np.random.default_rng(37)
    x = crowded_rows(rng, 20011, dtype)
    u = np.zeros((12, 20011), np.float32)
    u[1] = 1.5
    u[2] = 2.0 ** -26
    u[3, ::2] = np.nan
    u[7, 19999] = 0.25
    u[8, 3] = 1.0
    u[9, 0] = 0.5
    for T, P in ((1.0, 0.9), (0.0, 1.0), (0.7, 0.3)):
        check(gpu, oracle, x, u, T, P, want_probs=False)
