"""The tiled exact product in the cuts that its cost rule takes for small matrices (1, 2, 4, 6 and 8 M-tiles a workgroup over many blocks of rows): bit for bit the
LDS-staged kernel, at row counts around the blocks' edges, with padded last tiles and columns, bias, activation and residual."""
import ctypes as C

import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 15, 17, 33, 47, 65, 95, 97, 129, 200, 255, 257, 1500, 3001])
@pytest.mark.parametrize("N,K,act,res", [(384, 384, 0, True), (1152, 384, 0, False), (1531, 384, 2, False), (384, 1536, 0, True), (50, 1152, 2, True), (768, 128, 0, False)])
def test_cut_of_few_tiles_equals_staged(gpu, M, N, K, act, res):
    rng = np.random.default_rng(M + N + K)
    f = lambda *s: rng.normal(0, 1, s).astype(np.float32)
    a, w, b, r = f(M, K), f(N, K) * np.float32(K ** -0.5), f(N), f(M, N) if res else None
    cs, ct = np.empty((M, N), np.float32), np.empty((M, N), np.float32)
    p = lambda x: x.ctypes.data_as(C.c_void_p) if x is not None else None
    gpu.check(gpu.lib().tk_mi355x_gemm_pair(0, M, N, K, p(a), p(w), p(b), p(r), act, 0, p(cs), p(ct)))
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,act,res", [
    (257, 2048, 128, 2, False), (544, 1024, 128, 0, True), (543, 1024, 128, 3, True), (577, 992, 256, 1, True), (1441, 384, 384, 2, True), (2047, 288, 128, 0, False),   # tiles of 32 x 32
    (1825, 2176, 512, 0, True), (1857, 2176, 512, 2, False), (3841, 1088, 1024, 1, True), (3872, 1056, 1024, 0, True),                            # of 64 x 32
])
def test_wide_tiles_equal_staged(gpu, M, N, K, act, res):
    test_cut_of_few_tiles_equals_staged(gpu, M, N, K, act, res)


@pytest.mark.gpu
@pytest.mark.parametrize("ctx,width", [(100, 1024), (33, 1280), (97, 384)])
def test_wide_tiles_and_images_in_an_encoder(gpu, ctx, width):
    """a clip's encoder states do not depend on how many clips run with it: from 20 on its layers, and the images between them, are made in wide tiles"""
    hp = gpu.WhisperHP(80, ctx, width, width // 64, 1, 8, width, width // 64, 1, 512)
    asr = gpu.Asr(hp=hp, seed=4, max_batch=59)
    pcm = np.random.default_rng(ctx).integers(-6000, 6000, (59, 320 * ctx)).astype(np.int16)
    _, _, enc, logits = asr.transcribe_tokens(pcm, 1)
    for b in (0, 7, 58):
        _, _, one, lg = asr.transcribe_tokens(pcm[b:b + 1], 1)
        assert np.array_equal(one[0].view(np.uint32), enc[b].view(np.uint32)) and np.array_equal(lg[0].view(np.uint32), logits[b].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("width", [64, 128, 384, 768, 1024, 1152])
def test_norms_inside_products_of_a_few_rows(gpu, width):
    """a decoder's norms are made by the products behind them for up to four sequences and widths of 128 .. 1024 in steps of 128, as launches else: tokens and logits of
    a clip are the same bits whatever number of clips runs with it"""
    hp = gpu.WhisperHP(80, 40, 128, 2, 1, 24, width, width // 64, 2, 515)
    asr = gpu.Asr(hp=hp, seed=9, max_batch=6)
    pcm = np.random.default_rng(width).integers(-6000, 6000, (6, 5000)).astype(np.int16)
    ids, mel, enc, logits = asr.transcribe_tokens(pcm, 5)
    for n in (1, 2, 3, 4, 5):
        i2, m2, e2, l2 = asr.transcribe_tokens(pcm[:n], 5)
        assert np.array_equal(i2, ids[:n]) and np.array_equal(l2.view(np.uint32), logits[:n].view(np.uint32))
        assert np.array_equal(m2.view(np.uint32), mel[:n].view(np.uint32)) and np.array_equal(e2.view(np.uint32), enc[:n].view(np.uint32))
