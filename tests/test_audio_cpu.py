"""What the host decides for the audio streams before anything is launched."""
import ctypes as C

import pytest

import trackiellm_amd as tk


def up(n, m=64):
    return (n + m - 1) // m * m


def image(rows, k):
    """floats of a matrix as the tiled product's operand: whole blocks of 16, 32, 64, 128 or 256 rows"""
    block = next((b for b in (16, 32, 64, 128) if rows <= b), 256)
    return up(up(rows, block) * k)


@pytest.mark.parametrize("ctx,text_ctx,state,heads,layers,vocab", [
    (1500, 448, 384, 6, 4, 51864), (200, 448, 1344, 21, 1, 512), (40, 144, 1280, 80, 1, 512), (300, 448, 512, 2, 2, 512), (600, 448, 288, 2, 2, 512), (8, 448, 128, 2, 6, 64),
])
@pytest.mark.parametrize("clips", [1, 5, 32, 256])
def test_scratch_of_a_transcription_holds_its_decoder_steps(ctx, text_ctx, state, heads, layers, vocab, clips):
    """everything that stays for the whole call, the decode loop's tables, and the largest pair of operand images of a step (fc1 with fc2) on top"""
    B, R, T, d = clips, clips * ctx, 2 * ctx, state
    pitch = lambda n: up(n, 32)
    stays = [B * T * 400, B * T * 402, B * T * 201, B * T * 80, B * 64, B * T * 240, B * T * d, R * 3 * d] + 6 * [R * d] + [4 * R * d, B * heads * ctx * pitch(ctx), R * d]
    stays += layers * [R * d, R * d, B * text_ctx * d, B * text_ctx * d] + 6 * [B * d] + [4 * B * d, B * heads * pitch(max(ctx, text_ctx)), B * vocab, B, B, B]
    tables = (text_ctx + 2 * (text_ctx - 1)) * B
    images = (image(B, d) if d % 128 == 0 else 0) + (image(B, 4 * d) if 4 * d % 128 == 0 else 0)
    hp, size = tk.WhisperHP(80, ctx, state, heads, 1, text_ctx, state, heads, layers, vocab), C.c_uint64()
    assert tk.lib().tk_mi355x_asr_arena_bytes(C.byref(hp), clips, C.byref(size)) == 0
    assert size.value >= 4 * (sum(map(up, stays)) + up(tables) + images)


def test_scratch_size_refuses_bad_geometries():
    size = C.c_uint64()
    hp = lambda **kw: tk.WhisperHP(**{**dict(n_mels=80, n_audio_ctx=50, n_audio_state=64, n_audio_head=2, n_audio_layer=2, n_text_ctx=32, n_text_state=64, n_text_head=2, n_text_layer=2, n_vocab=512), **kw})
    f = tk.lib().tk_mi355x_asr_arena_bytes
    assert f(C.byref(hp()), 1, C.byref(size)) == 0
    assert f(None, 1, C.byref(size)) != 0 and f(C.byref(hp()), 1, None) != 0 and f(C.byref(hp()), 0, C.byref(size)) != 0 and f(C.byref(hp()), 257, C.byref(size)) != 0
    for n in ("n_mels", "n_audio_ctx", "n_audio_state", "n_audio_head", "n_text_ctx", "n_text_state", "n_text_head", "n_vocab"):
        assert f(C.byref(hp(**{n: 0})), 1, C.byref(size)) != 0
