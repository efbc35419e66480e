"""An encoder layer's attention in one kernel (heads of 64, up to 1536 positions) against the oracle, bit for bit: tiles of 16 rows and keys, quarters and rounds of 256 keys,
clips whose rows start inside a tile, and scores so far apart that quotients leave the normal range."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def geometry(ctx, state, heads):
    hp = O.whisper_tiny_test()
    hp.n_audio_ctx, hp.n_audio_state, hp.n_audio_head, hp.n_audio_layer = ctx, state, heads, 1
    hp.n_text_ctx, hp.n_text_state, hp.n_text_head, hp.n_text_layer = 8, state, heads, 1
    return hp


@pytest.mark.parametrize("ctx,state,heads,clips", [
    (1, 128, 2, 2), (2, 128, 2, 3), (15, 128, 2, 3), (16, 384, 6, 2), (17, 128, 2, 3), (63, 128, 2, 2), (65, 256, 4, 3), (250, 128, 2, 3), (256, 128, 2, 1), (257, 128, 2, 2),
    (512, 128, 2, 1), (527, 128, 2, 2), (770, 128, 2, 1), (1027, 128, 2, 2), (1281, 128, 2, 1), (1499, 128, 2, 2), (1535, 128, 2, 1), (1536, 128, 2, 2),
    (1537, 128, 2, 1),       # the three launches
    (40, 128, 4, 2), (40, 192, 3, 2),   # heads of 32; a width without tiled weights
])
def test_encoder_attention_over_contexts(gpu, ctx, state, heads, clips):
    hp = geometry(ctx, state, heads)
    pcm = np.clip(np.random.default_rng(ctx).normal(0, 3000, (clips, min(9000, 320 * ctx))), -32768, 32767).astype(np.int16)
    asr = gpu.Asr(hp=gpu.WhisperHP(*[getattr(hp, n) for n, _ in hp._fields_]), seed=3, max_batch=clips)
    _, _, enc, _ = asr.transcribe_tokens(pcm, 1)
    _, _, want, _ = O.OracleWhisper(hp, seed=3).transcribe(pcm, 1)
    assert np.array_equal(enc, want), np.abs(enc - want).max()


@pytest.mark.parametrize("ctx,spread", [(40, 30.0), (300, 300.0), (600, 3000.0)])
def test_encoder_attention_over_spreads_of_scores(gpu, tmp_path, ctx, spread):
    """query weights times `spread`: rows whose smallest exponentials are 2^-100 and less, subnormal quotients among them, and zero"""
    import ggml_whisper_util as G
    hp = geometry(ctx, 128, 2)
    orc = O.OracleWhisper(hp, seed=5)
    T = orc.tensors()
    T["encoder.blocks.0.attn.query.weight"] = T["encoder.blocks.0.attn.query.weight"] * np.float32(spread)
    rounded, file_t = G.checkpoint_tensors(T, hp)
    orc.set_tensors(rounded)
    path = tmp_path / "ggml.bin"
    G.write_ggml(path, hp, T["frontend.mel_filters"], [(" w%d" % i).encode() for i in range(hp.n_vocab - 7)], file_t)
    asr = gpu.Asr(model=str(path))
    pcm = np.clip(np.random.default_rng(ctx).normal(0, 3000, (1, 9000)), -32768, 32767).astype(np.int16)
    _, _, enc, _ = asr.transcribe_tokens(pcm, 1)
    _, _, want, _ = orc.transcribe(pcm, 1)
    assert np.array_equal(enc, want), np.abs(enc - want).max()
