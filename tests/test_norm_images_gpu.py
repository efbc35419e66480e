"""Norms and convolution columns that are written as operand images: encoder and decoder of widths in every form, rows that fill no tile."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


# two and four times 256 columns a row, the widest of a tile in LDS, rows by themselves in registers, longer ones; 23 and 32 positions, one clip and three
@pytest.mark.parametrize("state,positions,clips", [(128, 23, 1), (512, 32, 3), (640, 23, 3), (896, 16, 1), (1024, 23, 1), (1280, 17, 3), (1408, 23, 1)])
def test_states_and_logits_match_the_oracle(gpu, state, positions, clips):
    geometry = (80, positions, state, state // 64, 1, 8, state, state // 64, 1, 512)
    asr = gpu.Asr(hp=gpu.WhisperHP(*geometry), seed=2, max_batch=clips)
    pcm = np.random.default_rng(state).integers(-6000, 6000, (clips, 4000)).astype(np.int16)
    ids, _, enc, logits = asr.transcribe_tokens(pcm, 2)
    want, _, we, wl = O.OracleWhisper(O.WhisperHP(*geometry), seed=2).transcribe(pcm, 2)
    for got, exact in ((enc, we), (logits, wl)):
        assert np.array_equal(got.view(np.uint32), exact.view(np.uint32))
    assert np.array_equal(ids, want)
    asr.close()
