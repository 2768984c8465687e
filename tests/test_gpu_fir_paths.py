"""FirFilter's kernels at the sizes where they change over or run out: chunk
lengths around a tile (256 and 1024 outputs) and the split form's limit, tap
counts around the matrix form's K rounds and the LDS limits, real and complex
taps, histories longer than a chunk, non-finite samples."""
import numpy as np
import pytest

import libfalcon_dsp_amd as fd
from libfalcon_dsp_amd.signals import cwgn
from oracle import oracle as O

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _taps(m, real, seed=0):
    rng = np.random.default_rng(1000 * m + seed)
    h = rng.standard_normal(m) + (0 if real else 1j * rng.standard_normal(m))
    return (h / np.sqrt(m)).astype(np.complex64)


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("m,lens", [(1, [1, 255, 256, 257]), (2, [1023, 1, 1024, 1025]), (17, [16, 15, 4096, 3]),
                                    (33, [5, 2000, 131_072, 131_073]), (129, [100, 28, 140_001]),
                                    (1840, [700, 131_075]), (1850, [131_075, 1000]), (3800, [600, 4000]),
                                    (3900, [5000, 1]), (6145, [3000, 2500])])
def test_float_chunks(m, lens, real):
    h = _taps(m, real)
    x = cwgn(70 + m, sum(lens))
    x64, h64 = x.astype(np.complex128), h.astype(np.complex128)
    size = 1 << int(x.size + m).bit_length()
    want = np.fft.ifft(np.fft.fft(x64, size) * np.fft.fft(h64, size))[: x.size]
    f, at = fd.FirFilter(h), 0
    # m rounded products and sums of random sign: about sqrt(m) u of the
    # output's scale, the largest of 10^5 outputs about five times that
    tol = 10 * np.sqrt(m + 4) * U * np.sqrt(np.mean(np.abs(x64) ** 2) * np.sum(np.abs(h64) ** 2))
    for n in lens:
        got = f.apply(x[at:at + n])
        assert np.max(np.abs(got - want[at:at + n])) <= tol, (m, real, at, n)
        at += n


@pytest.mark.parametrize("n_chan,m,n", [(3, 1, 1), (5, 4, 1023), (3, 17, 1025), (300, 33, 4097), (600, 64, 2049),
                                        (1400, 20, 9001), (4, 4300, 5000), (4, 5100, 4000)])
def test_bank_groups_a_wave(n_chan, m, n):
    # one, two and three column groups a wave (blocks of 1024, 2048 and 3072
    # outputs), ragged last blocks, the longest windows of the matrix form and
    # the VALU form beyond them, the history carried into a second chunk
    rng = np.random.default_rng(m)
    taps = (rng.standard_normal((n_chan, m)) / np.sqrt(m)).astype(np.float32)
    x = cwgn(11 + m, n_chan * 2 * n).reshape(n_chan, 2 * n)
    bank = fd.FirBank(taps)
    got = np.concatenate([bank.apply(x[:, :n]), bank.apply(x[:, n:])], axis=1)
    tol = 10 * np.sqrt(m + 4) * U
    for c in {0, 1, n_chan // 2, n_chan - 1}:
        size = 1 << int(2 * n + m).bit_length()
        want = np.fft.ifft(np.fft.fft(x[c].astype(np.complex128), size) * np.fft.fft(taps[c].astype(float), size))
        scale = np.sqrt(np.mean(np.abs(x[c]) ** 2) * np.sum(taps[c].astype(float) ** 2))
        assert np.max(np.abs(got[c] - want[:2 * n])) <= tol * scale, (n_chan, m, n, c)


@pytest.mark.parametrize("n", [3000, 140_000])
@pytest.mark.parametrize("real", [False, True])
def test_non_finite_samples_reach_their_windows_only(n, real):
    m = 40
    h = _taps(m, real)
    x = cwgn(5, n)
    want = fd.FirFilter(h).apply(x)
    bad = x.copy()
    bad[[7, 1500, n - 3]] = [np.inf, np.nan, complex(0, -np.inf)]
    f = fd.FirFilter(h)
    got = f.apply(bad)
    hit = np.zeros(n, bool)
    for p in (7, 1500, n - 3):
        hit[p:p + m] = True
    assert not np.isfinite(got[hit]).any()
    assert np.max(np.abs(got[~hit] - want[~hit])) <= 20 * np.sqrt(m) * U * np.sqrt(np.mean(np.abs(x) ** 2))
    # carried into the next chunk, and out of it
    nxt = f.apply(x[:200])
    assert not np.isfinite(nxt[: m - 3]).any() and np.isfinite(nxt[m - 3:]).all()


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("m", [1, 7, 8, 9, 64, 300, 6145])
def test_int16_chunks_are_the_sequential_sums(m, real):
    h = _taps(m, real, seed=1)
    x = (np.random.default_rng(m).standard_normal((9000, 2)) * 6000).round().astype(np.int16)
    f, o, at = fd.FirFilter(h), O.Fir(h), 0
    for n in (1, 255, 256, 257, 3, 513, 7000):
        np.testing.assert_array_equal(f.apply_ci16(x[at:at + n]), o.apply_ci16(x[at:at + n]), err_msg=f"{m} {at} {n}")
        at += n
