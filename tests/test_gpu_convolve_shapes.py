"""ear_convolve at the edges of its transforms' shapes: the smallest length,
both sides of powers of two (odd and even logs: square and oblong splits), the
longest sequence of the binary64 kernels and the first one past it."""
import numpy as np
import pytest

from ear_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fade", [False, True])
@pytest.mark.parametrize("n_out", [2, 3, 4095, 4096, 4097, 8192, 8193, 16385, 100_003, 1 << 19, (1 << 19) + 1,
                                   (1 << 22) - 1, 1 << 22, (1 << 22) + 1])
def test_lengths_around_powers_of_two(gpu_ctx, n_out, fade):
    """Against a binary64 transform: the kernels' result is the convolution
    rounded to binary32 (half an ulp of the largest sample, 2^-24, plus
    binary64 noise); past 2^22 samples the binary32 library transforms keep
    their 2e-6 per stage."""
    rng = np.random.default_rng(n_out)
    m = max(1, n_out // 5)
    n = n_out - 1 - m
    ir, ir2 = (rng.normal(size=k).astype(np.float32) for k in (m, max(1, m // 2)))
    sig = rng.uniform(-1, 1, n).astype(np.float32)
    out = api.convolve(gpu_ctx, ir, sig, ir2 if fade else None)
    assert len(out) == n_out
    L = 1 << n_out.bit_length()

    def conv(a, b):
        return np.fft.irfft(np.fft.rfft(a.astype(np.float64), L) * np.fft.rfft(b.astype(np.float64), L), L)[:n_out]

    if fade:
        df = np.float32(1.0) / np.float32(max(1, n))
        down, up = np.full(n, -df, np.float32), np.full(n, df, np.float32)
        down[:1], up[:1] = 1.0, 0.0
        ref = conv(ir, sig * np.cumsum(down, dtype=np.float32)) + conv(ir2, sig * np.cumsum(up, dtype=np.float32))
    else:
        ref = conv(ir, sig)
    top = np.abs(ref).max() if n else 0.0
    tol = (2.0 ** -24 + 1e-13) * top if n_out <= 1 << 22 else 2e-6 * top * np.log2(n_out)
    assert np.max(np.abs(out - ref)) <= tol
