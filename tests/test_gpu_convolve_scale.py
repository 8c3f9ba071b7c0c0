"""ear_convolve with operands of very different size: the error is relative to
the result, whatever the sizes of the response and the sound, and silence in
is silence out."""
import numpy as np
import pytest

from ear_amd import api

pytestmark = pytest.mark.gpu

M, N = 300, 900
N_OUT = M + N + 1


def _conv(a, b, L=4096):
    return np.fft.irfft(np.fft.rfft(a.astype(np.float64), L) * np.fft.rfft(b.astype(np.float64), L), L)[:N_OUT]


def _fades(sig):
    n = len(sig)
    df = np.float32(1.0) / np.float32(n)
    down, up = np.full(n, -df, np.float32), np.full(n, df, np.float32)
    down[0], up[0] = 1.0, 0.0
    return sig * np.cumsum(down, dtype=np.float32), sig * np.cumsum(up, dtype=np.float32)


def _draw():
    rng = np.random.default_rng(7)
    return (rng.normal(size=M).astype(np.float32), rng.normal(size=M).astype(np.float32),
            np.clip(0.2 * rng.normal(size=N), -1, 1).astype(np.float32))


def _close(out, ref):
    """Rounded once to binary32: half an ulp of the largest sample (2^-24 of
    it) plus binary64 noise, or half the smallest subnormal."""
    assert np.max(np.abs(out - ref)) <= max((2.0 ** -24 + 1e-13) * np.abs(ref).max(), 2.0 ** -150)


@pytest.mark.parametrize("scale", [1e-6, 1e-9, 1e-12, 1e-20, 1e-30, 1e-37, 1e-42, 1e12, 1e30])
@pytest.mark.parametrize("which", ["track", "signal"])
def test_error_does_not_depend_on_the_operands_sizes(gpu_ctx, which, scale):
    ir, _, sig = _draw()
    ir, sig = ((ir * np.float64(scale)).astype(np.float32), sig) if which == "track" else \
        (ir, (sig * np.float64(scale)).astype(np.float32))
    _close(api.convolve(gpu_ctx, ir, sig), _conv(ir, sig))


@pytest.mark.parametrize("s1,s2,ss", [(1.0, 1e-9, 1.0), (1e-12, 1.0, 1.0), (1e-12, 1e-12, 1.0), (1e-20, 1e-17, 1.0),
                                      (1.0, 1e-20, 1e-12), (1e-25, 1e10, 1e8)])
def test_fade_between_tracks_of_different_level(gpu_ctx, s1, s2, ss):
    ir, ir2, sig = _draw()
    ir, ir2, sig = (ir * np.float64(s1)).astype(np.float32), (ir2 * np.float64(s2)).astype(np.float32), \
        (sig * np.float64(ss)).astype(np.float32)
    down, up = _fades(sig)
    _close(api.convolve(gpu_ctx, ir, sig, ir2), _conv(ir, down) + _conv(ir2, up))


def test_silence_stays_silence(gpu_ctx):
    ir, ir2, sig = _draw()
    zt, zs = np.zeros(M, np.float32), np.zeros(N, np.float32)
    for args in [(zt, sig), (ir, zs), (zt, zs), (zt, sig, zt), (ir, zs, ir2)]:
        out = api.convolve(gpu_ctx, *args)
        assert len(out) == N_OUT and not out.any()
    down, up = _fades(sig)
    _close(api.convolve(gpu_ctx, zt, sig, ir2), _conv(ir2, up))
    _close(api.convolve(gpu_ctx, ir, sig, zt), _conv(ir, down))


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_sample_that_is_no_number_reaches_every_output(gpu_ctx, bad):
    """As transforms of the whole sequence carry it, also beside a silent track."""
    ir, _, sig = _draw()
    ir_bad, sig_bad = ir.copy(), sig.copy()
    ir_bad[5] = sig_bad[7] = bad
    for args in [(ir_bad, sig), (ir, sig_bad), (np.zeros(M, np.float32), sig_bad)]:
        assert not np.isfinite(api.convolve(gpu_ctx, *args)).any()
