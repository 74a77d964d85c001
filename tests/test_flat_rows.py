"""Near-flat rows of more elements than one wave's 32-bit partial sums hold (a
lane's share of the exact sum past 2^50): the rows' sums on every route that
streams them by one workgroup, against the oracle, bit for bit."""
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


def check(gpu, oracle, x, u, top_p, **kw):
    exp = oracle.sample(x, u, 1.0, top_p, n_threads=8)
    got = gpu.sample(x, u, 1.0, top_p, **kw)
    assert got["rc"] == 0 and np.array_equal(got["ids"], exp["ids"])
    if kw.get("want_probs", True):
        assert np.array_equal(got["cand"], exp["cand"]) and np.array_equal(got["probs"], exp["probs"])
        # the sum decides the cut: neither all ranks nor the first alone
        assert 1 < (exp["probs"] > 0).sum() < u.shape[1]


def test_streamed_row(gpu, oracle):
    """1024 threads a row, more than 1024 elements of weight 1 each"""
    V = 1_200_000
    x = (np.arange(V, dtype=np.float32) * np.float32(-2.0 ** -26))[None]
    check(gpu, oracle, x, oracle.uniform(1, 1, 1, 30), 12.5 / V, flags=gpu.FLAG_GENERIC)
    check(gpu, oracle, x, oracle.uniform(1, 1, 1, 30), 12.5 / V)
    check(gpu, oracle, np.full_like(x, 2.5), oracle.uniform(1, 2, 1, 200), 150.5 / V)


def test_segmented_exact_sum(gpu, oracle):
    """the segmented kernel's exact sum: 512 threads a row"""
    V = 620_000
    x = (np.arange(V, dtype=np.float32) * np.float32(-2.0 ** -26))[None]
    x = np.ascontiguousarray(x.reshape(1, -1, 1000).transpose(0, 2, 1).reshape(1, V))  # over every segment
    check(gpu, oracle, x, oracle.uniform(1, 1, 1, 30), 12.5 / V, flags=gpu.FLAG_EXACT_LSE)


def test_sorted_row(gpu, oracle):
    """the wide nucleus path's sort of a row none of whose kept ranks has a
    positive score: 2^20 equal ranks, whose sum once wrapped to 0; only rank 1
    scores 0 (its noise is infinite), the others lose to it"""
    V = 1 << 20
    u = np.zeros((1, V), np.float32)
    u[0, 1] = 1.0
    check(gpu, oracle, np.full((1, V), 0.5, np.float32), u, 1.5, want_probs=False)
