"""d3s_uniform_fill's four-at-a-time kernel against the oracle's uniforms: every
remainder of the count, starts off 16 bytes (scalar stores), and nothing
written past the end."""
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


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 1023, 1024, 1025, 262_147])
@pytest.mark.parametrize("off", [0, 1, 2, 3])
def test_fill_remainders_and_alignment(gpu, oracle, n, off):
    import hiprt
    seed, draw = 0x123456789ABCDEF, (1 << 40) + 5
    buf = hiprt.to_device(np.full(n + off + 8, -1.0, np.float32))
    assert gpu.lib().d3s_uniform_fill(buf.ptr + 4 * off, n, seed, draw, None) == 0
    hiprt.synchronize()
    got = buf.download((n + off + 8,), np.float32)
    assert np.array_equal(got[off:off + n], oracle.uniform(seed, draw, 1, n)[0])
    assert (got[:off] == -1.0).all() and (got[off + n:] == -1.0).all()
