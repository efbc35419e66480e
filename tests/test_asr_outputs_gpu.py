"""Mel, encoder states and logits on their way to the caller: whatever their size they pass through a bounded piece of pinned memory that the context keeps."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CAP = 64 << 20


def staging(gpu, asr):
    f = gpu.lib().tk_mi355x_asr_staging_bytes
    f.restype = C.c_uint64
    return f(asr.h)


# floats that a clip's outputs take: whole in the pinned memory, in pieces (two of them filled in turn, the last one short), logits larger than half of it
@pytest.mark.parametrize("ctx,state,vocab,clips", [(40, 128, 515, 3), (1500, 128, 512, 41), (700, 256, 51864, 60), (30, 128, 140000, 64)])
def test_outputs_of_many_clips_are_those_of_one(gpu, ctx, state, vocab, clips):
    hp = gpu.WhisperHP(80, ctx, state, state // 64, 1, 8, state, state // 64, 1, vocab)
    asr, one = gpu.Asr(hp=hp, seed=4, max_batch=clips), gpu.Asr(hp=hp, seed=4, max_batch=1)
    pcm = np.random.default_rng(ctx).integers(-6000, 6000, (clips, 160 * ctx)).astype(np.int16)
    held = []
    for n in (clips, 1, clips):  # wide and narrow calls in turn
        ids, mel, enc, logits = asr.transcribe_tokens(pcm[:n], 2)
        held.append(staging(gpu, asr))
        for b in {0, n // 2, n - 1}:
            i1, m1, e1, l1 = one.transcribe_tokens(pcm[b:b + 1], 2)
            for got, want in ((ids, i1), (mel, m1), (enc, e1), (logits, l1)):
                assert np.array_equal(got[b:b + 1].view(np.uint32), want.view(np.uint32))
    total = 4 * (mel.size + enc.size + logits.size)
    assert held[0] == held[1] == held[2] <= CAP and (held[0] >= total or held[0] == CAP)
    assert staging(gpu, one) <= CAP


def test_calls_for_tokens_alone_pin_nothing(gpu):
    asr = gpu.Asr(hp=gpu.WhisperHP(80, 40, 128, 2, 1, 8, 128, 2, 1, 512), seed=4, max_batch=2)
    asr.transcribe_tokens(np.zeros((2, 3000), np.int16), 2, want_aux=False)
    assert staging(gpu, asr) == 0
