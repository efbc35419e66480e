"""A prompt's positions go through the decoder several at a time; ids, logits and log-probabilities stay those of one position after the other."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


# a prompt of four (the vocabulary makes it one): whole in one pass with the norms made by the products and without, in two with a remainder of one and of two, position by position
@pytest.mark.parametrize("clips,state,heads,layers", [(1, 384, 6, 2), (2, 128, 2, 1), (7, 128, 1, 2), (40, 128, 8, 1), (64, 128, 2, 2), (130, 128, 2, 2)])
def test_prompts_in_spans_match_the_oracle(gpu, clips, state, heads, layers):
    geometry = (80, 30, state, heads, 1, 40, state, heads, layers, 51865)
    asr = gpu.Asr(hp=gpu.WhisperHP(*geometry), seed=8, max_batch=clips)
    assert len(asr.prompt_tokens()) == 4
    orc = O.OracleWhisper(O.WhisperHP(*geometry), seed=8)
    pcm = np.random.default_rng(clips).integers(-6000, 6000, (clips, 4000)).astype(np.int16)
    ids, _, _, logits = asr.transcribe_tokens(pcm, 2)
    want, _, _, wl = orc.transcribe(pcm, 2, prompt=asr.prompt_tokens())
    assert np.array_equal(ids, want) and np.array_equal(logits.view(np.uint32), wl.view(np.uint32))
    ids, lp = asr.transcribe_policy(pcm[:7], 3, temperature=0.7, seed=5)   # a draw's counter is its position
    want, wlp = orc.transcribe_policy(pcm[:7], 3, 0.7, 5, prompt=asr.prompt_tokens())
    assert np.array_equal(ids, want) and np.array_equal(lp.view(np.uint32), wlp.view(np.uint32))
    asr.close()
