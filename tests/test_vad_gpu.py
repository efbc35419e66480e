"""Voice activity: the probabilities of any number of windows, through one slot of pinned memory and through two in turn, at every window length, against the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 33, 128, 129, 400, 511, 512, 513, 1024, 1025, 1700])
def test_numbers_of_windows(gpu, n):
    vad = gpu.Vad()
    x = np.random.default_rng(n).normal(0, 0.3, (n, 480)).astype(np.float32)
    want = O.vad_probabilities(7, x)
    assert np.array_equal(vad.probabilities(x).view(np.uint32), want.view(np.uint32))
    assert np.array_equal(vad.probabilities(x[::-1]).view(np.uint32), want[::-1].view(np.uint32))  # the same buffers again


@pytest.mark.gpu
@pytest.mark.parametrize("rate", [8000, 16000, 48000])
def test_window_lengths_and_not_finite_sound(gpu, rate):
    vad = gpu.Vad(sample_rate=rate)
    w = int(rate * 30 / 1000)
    x = np.random.default_rng(rate).normal(0, 0.3, (3, w)).astype(np.float32)
    one = [vad.probabilities(x[i:i + 1])[0] for i in range(3)]
    assert np.array_equal(vad.probabilities(x), np.array(one, np.float32)) and len(set(one)) == 3
    x[1, w // 2] = np.nan
    got = vad.probabilities(x)
    assert got[0] == one[0] and got[2] == one[2]


# half of what four waves hold, all of it, and the windows that one wave walks; rows with a sample of each special value
@pytest.mark.gpu
@pytest.mark.parametrize("rate", [8000, 16000, 48000])
def test_shares_of_a_window(gpu, rate):
    vad, w = gpu.Vad(sample_rate=rate), rate * 30 // 1000
    x = np.random.default_rng(rate).normal(0, 0.3, (7, w)).astype(np.float32)
    x[3], x[4, ::2], x[5, w - 1], x[6, 0] = 0.0, -0.0, np.inf, -np.inf
    got, want = vad.probabilities(x), O.vad_probabilities(7, x)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~np.isnan(got)].view(np.uint32), want[~np.isnan(want)].view(np.uint32))
