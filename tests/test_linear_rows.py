"""The heads' gemv of several rows (the matrix-core kernel) against the oracle's
single-row order, bit for bit: tile edges and remainders of the hidden rows,
the weight rows and the 128-element blocks, both tile shapes, weights and rows
8 bytes off 16, and sums that are subnormal, overflow or are not finite.  Up to
10 240 logits, and three rows on weights that fit the L2s, go to the one-row
kernel: both sides of those lines."""
import numpy as np
import pytest

import d3s_workloads as W

pytestmark = pytest.mark.gpu


def bf16(a):
    return W.f32_to_bf16_bits(np.asarray(a, np.float32))


@pytest.fixture(scope="module")
def gpu():
    import d3s
    import hiprt
    d3s.lib()
    if hiprt.device_count() < 1:
        pytest.skip("no GPU")
    return d3s


@pytest.mark.parametrize("N,K,V", [
    (3, 128, 1), (3, 256, 4), (16, 384, 5), (17, 128, 15), (4, 640, 16), (31, 512, 17), (16, 1920, 20),
    (33, 256, 21), (5, 2048, 4097), (64, 2048, 1000), (100, 384, 36), (3, 896, 127),
    # the matrix-core kernel's 16 x 16 tiles: few weight rows, many hidden rows
    (10241, 128, 1), (2561, 256, 4), (2053, 384, 5), (700, 128, 15), (641, 640, 16), (605, 512, 17), (513, 1920, 20),
    (489, 256, 21), (289, 384, 36), (81, 896, 127),
    # the dispatch's lines: 10 240 logits and one row of them more; three rows
    (10, 256, 1024), (11, 256, 1024), (10240, 128, 1), (3, 384, 4097), (3, 512, 4100), (3, 512, 4101), (4, 512, 4101),
    (3, 384, 8192), (3, 2560, 7813),
    # 32 x 32 tiles (at least 256 of them): remainders 0, 1, 4, 5 and 31 of V, partly filled row tiles
    (33, 128, 4096), (64, 256, 4097), (65, 384, 4100), (40, 640, 4101), (97, 128, 8223)])
def test_rows_equal_the_oracle(gpu, oracle, N, K, V):
    rng = np.random.default_rng([N, K, V])
    x = bf16(rng.standard_normal((N, K)))
    w = bf16(rng.standard_normal((V, K)) * 0.05)
    rc, y = gpu.linear_bf16(x, w)
    assert rc == 0
    assert np.array_equal(y, oracle.linear_bf16(x, w))


@pytest.mark.parametrize("N,V", [(5, 40), (300, 40), (36, 4097)])
@pytest.mark.parametrize("scale", [2.0 ** -68, 2.0 ** 62, None])
def test_rows_equal_one_row_calls_on_extreme_values(gpu, N, V, scale):
    """subnormal sums, overflowing sums, and arbitrary bit patterns (infinities
    and NaN among them): the bits of the one-row kernel, a NaN for a NaN"""
    rng = np.random.default_rng(7)
    K = 384
    if scale is None:
        x, w = (rng.integers(0, 1 << 16, s).astype(np.uint16) for s in ((N, K), (V, K)))
        w[rng.random((V, K)) < 0.97] = 0  # few enough that finite sums remain
        x[(x & 0x7f80) == 0x7f80] &= 0x3fff  # 0 * infinity would make every sum NaN
    else:
        x, w = (bf16(rng.standard_normal(s) * scale) for s in ((N, K), (V, K)))
    rc, y = gpu.linear_bf16(x, w)
    assert rc == 0
    for n in range(0, N, 7):
        one = gpu.linear_bf16(x[n:n + 1], w)[1][0]
        nan = (one & 0x7fff) > 0x7f80
        assert np.array_equal(nan, (y[n] & 0x7fff) > 0x7f80)
        assert np.array_equal(y[n][~nan], one[~nan]) and (~nan).any()


@pytest.mark.parametrize("N", [20, 220])
def test_rows_at_8_byte_boundaries(gpu, oracle, N):
    import hiprt
    K, V = 256, 50
    rng = np.random.default_rng(3)
    x, w = bf16(rng.standard_normal((N, K))), bf16(rng.standard_normal((V, K)))
    bx, bw = hiprt.DeviceBuffer(x.nbytes + 8), hiprt.DeviceBuffer(w.nbytes + 8)
    bx.upload(x, 8)
    bw.upload(w, 8)
    by = hiprt.to_device(np.full(N * V + 8, 0x1234, np.uint16))
    assert gpu.lib().d3s_linear_bf16(bx.ptr + 8, bw.ptr + 8, N, K, V, by.ptr + 2, None) == 0
    hiprt.synchronize()
    y = by.download((N * V + 8,), np.uint16)
    assert np.array_equal(y[1:1 + N * V].reshape(N, V), oracle.linear_bf16(x, w))
    assert y[0] == 0x1234 and (y[1 + N * V:] == 0x1234).all()
