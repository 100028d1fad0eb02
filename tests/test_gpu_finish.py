"""Short series take one launch for prefix sums, denominators and g2 (N <= 4096), longer
ones the chain of kernels: both sides of the line, series around the 256-lag blocks and
the 4-frame steps, every count type (uint16 with and without wide pixels), sums small
enough for FP64 products and sums that need 128 bits.  Numerators, sums and denominators
equal the oracle's exact integers; g2 is one rounding away.  Marked gpu."""
import sys

import numpy as np
import pytest

from oracle import g2 as og

pytestmark = pytest.mark.gpu


def _check(f, q):
    from dynamix_amd.correlator.dense import MatMulCorrelator
    n = f.shape[0]
    c = MatMulCorrelator(q.shape, n, q)
    g2 = c.correlate(f)
    ref = og.dense_g2(f, q)
    np.testing.assert_array_equal(c.last_numerators.cpu().numpy(), ref["num"])
    np.testing.assert_array_equal(c.last_sums.cpu().numpy(), ref["sums"])
    den = og.denominators(ref["sums"]).astype(np.float64)
    np.testing.assert_array_equal(c.last_denominators.cpu().numpy(), den)
    assert np.array_equal(np.isnan(g2), np.isnan(ref["g2"]))
    fin = np.isfinite(ref["g2"])
    # float32 rounding of the FP64 quotient
    np.testing.assert_allclose(g2[fin], ref["g2"][fin], rtol=1.2e-7)


def _stack(n, dtype, seed):
    rng = np.random.default_rng(seed)
    f = rng.poisson(0.4, size=(n, 6, 8)).astype(np.int64)
    if dtype == np.int8:
        f -= rng.integers(0, 2, size=f.shape)
    if dtype == np.uint16:
        f[:, 1, 2] += rng.integers(0, 3000, size=n)   # one wide pixel in bin 1
    f[n // 2] = 0                                     # an empty frame
    q = np.zeros((6, 8), np.int32)
    q[:2] = 1
    q[2:5] = 2
    q[5, :4] = 4                                      # bin 3 has no pixel
    return f.astype(dtype), q


@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.uint16])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 256, 257, 300, 1023, 4095, 4096, 4097])
def test_finish_line(dtype, n):
    print("[case] finish dtype=%s n=%d" % (np.dtype(dtype).name, n), flush=True)
    sys.stdout.flush()
    _check(*_stack(n, dtype, n))


@pytest.mark.parametrize("n", [17, 700])
def test_finish_128_bit_sums(n):
    """40,000 full-range uint16 pixels: N max|S|^2 > 2^52, so products go to 128 bits
    (S = 2.6e9; Den < 2^73, rounded once to FP64)."""
    print("[case] finish 128-bit n=%d" % n, flush=True)
    from dynamix_amd.correlator.dense import MatMulCorrelator
    f = np.full((n, 200, 200), 65535, np.uint16)
    f[::3] -= 1
    c = MatMulCorrelator((200, 200), n)
    g2 = c.correlate(f)
    s = [int(x) for x in f.reshape(n, -1).sum(axis=1, dtype=np.uint64)]
    np.testing.assert_array_equal(c.last_sums.cpu().numpy()[0], np.array(s, np.int64))
    den = c.last_denominators.cpu().numpy()[0]
    for tau in (0, 1, n // 2, n - 1):
        exact = sum(a * b for a, b in zip(s[:n - tau], s[tau:]))
        # hi * 2^64 + lo, each rounded once: 2 ulp
        assert abs(den[tau] - float(exact)) <= 2 * np.spacing(float(exact)), tau
    v = f[:, 0, 0].astype(object)
    for tau in (0, 1, n - 1):
        exact = 40000.0 ** 2 * float(sum(a * b for a, b in zip(v[:n - tau], v[tau:]))) / float(
            sum(a * b for a, b in zip(s[:n - tau], s[tau:])))
        assert abs(g2[0, tau] - exact) <= 2.4e-7 * exact, tau
