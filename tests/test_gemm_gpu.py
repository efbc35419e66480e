"""The two exact fp32 GEMMs against each other and against a float32 fma chain: the LDS-staged kernel (k_gemm_f32 / k_gemm_f32_big) and the
tiled kernel (csrc/nn/tk_gemm_tiled.hip) must agree bit for bit on every shape class the Whisper and fp16-LLM paths send them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(gpu, M, N, K, act=0, f16=0, bias=True, residual=False, seed=0):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((M, K)).astype(np.float32)
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32) if bias else None
    r = rng.standard_normal((M, N)).astype(np.float32) if residual else None
    cs, ct = np.empty((M, N), np.float32), np.empty((M, N), np.float32)
    p = lambda x: x.ctypes.data_as(C.c_void_p) if x is not None else None
    gpu.check(gpu.lib().tk_mi355x_gemm_pair(0, M, N, K, p(a), p(w), p(b), p(r), act, f16, p(cs), p(ct)))
    return a, w, b, r, cs, ct


@pytest.mark.parametrize("M,N,K,act,bias,res", [
    (1, 16, 128, 0, False, False),        # one live row, one tile
    (32, 384, 384, 0, True, False),       # Whisper decoder linear, 32 utterances (2 M-tiles)
    (64, 1536, 384, 2, True, False),      # fc1 + GELU, 4 M-tiles
    (33, 51864 // 8, 384, 0, False, False),  # N not a multiple of 16 (6483): padded last tile
    (300, 384, 1536, 0, True, True),      # more than one 256-row block, residual epilogue
    (1500, 384, 1152, 2, True, False),    # conv2 as a GEMM, six row blocks, K = 9 * 128
    (257, 48, 128, 3, True, True),        # tails everywhere
])
def test_tiled_equals_staged_bitwise(gpu, M, N, K, act, bias, res):
    a, w, b, r, cs, ct = _pair(gpu, M, N, K, act, 0, bias, res, seed=M + N)
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))
    # a few outputs against the definition: one fma chain over k ascending from zero (float32 fma emulated in float64: exact for one step)
    rng = np.random.default_rng(1)
    for _ in range(8):
        i, j = int(rng.integers(M)), int(rng.integers(N))
        acc = np.float32(0)
        for k in range(K):
            acc = np.float32(np.float64(a[i, k]) * np.float64(w[j, k]) + np.float64(acc))
        if act == 0 and not res:
            want = np.float32(acc + (b[j] if bias else np.float32(0)))
            assert ct[i, j] == want


@pytest.mark.parametrize("M,N,K", [
    (1, 1, 128), (31, 17, 128), (401, 255, 1152), (33, 65, 2304),      # one element, tails on both sides, a long chain
    (6400, 80, 768), (6401, 16, 640), (12800, 64, 1152), (3201, 257, 1152), (12801, 128, 640), (12800, 130, 1152),
    (12795, 80, 2304), (51201, 79, 1152), (25600, 32, 128), (51200, 33, 128), (9000, 384, 128),
])
def test_block_forms_equal_the_chain(gpu, M, N, K):
    """sizes that fill no block, in whatever blocks the staged kernels cut them into (each form by number: below): the tiled kernel's bits, and the definition
    at the corners"""
    a, w, b, r, cs, ct = _pair(gpu, M, N, K, seed=M + N)
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))
    for i, j in ((0, 0), (M - 1, N - 1), (0, N - 1), (M // 2, N // 2)):
        acc = np.float32(0)
        for k in range(K):
            acc = np.float32(np.float64(a[i, k]) * np.float64(w[j, k]) + np.float64(acc))
        assert cs[i, j] == np.float32(acc + b[j])


FORMS = [(32, 32), (64, 16), (64, 32), (64, 64), (64, 80), (128, 80), (128, 32), (128, 64), (128, 96), (128, 128), (64, 64)]


def _form(gpu, form, a, w, K, b, r, act=0, conv=None, M=None):
    N, c = w.shape[0], np.empty((M or a.shape[0], w.shape[0]), np.float32)
    p = lambda x: x.ctypes.data_as(C.c_void_p) if x is not None else None
    gpu.check(gpu.lib().tk_mi355x_gemm_f32(0, form, c.shape[0], N, K, 0 if conv else a.shape[1], w.shape[1], p(a), p(w), p(b), p(r), act, conv and (C.c_int * 9)(*conv), p(c)))
    return c


@pytest.mark.parametrize("form", range(11))
def test_each_form_equals_the_chain(gpu, form):
    """every exact kernel by number, at sizes that fill no block of it: one element, a slab of k and its neighbours, a row and a column less and more than a
    block; aligned operands and (pitch K + 3, K odd) unaligned ones.  Reference: the 64 x 64 kernel, which is held to the definition at the corners"""
    rows, cols = FORMS[form]
    tall = 6 <= form < 9
    rng = np.random.default_rng(form)
    for M, N, K, pad in ((1, 1, 1, 0), (1, 1, 4, 0), (rows - 1, cols, 33, 3), (rows + 1, cols if tall else cols + 1, 31, 0), (2 * rows + 3, cols - 1, 64, 0), (rows, cols, 68, 4),
                         (rows + 17, cols - 5 if tall else 2 * cols + 5, 129, 3), (3 * rows, cols if tall else 3 * cols, 260, 0)):
        a = rng.standard_normal((M, K + pad)).astype(np.float32)
        w = rng.standard_normal((N, K + pad)).astype(np.float32)
        b, r = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
        got, want = _form(gpu, form, a, w, K, b, r), _form(gpu, 10, a, w, K, b, r)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (M, N, K, pad)
        for i, j in ((0, 0), (M - 1, N - 1), (0, N - 1)):
            acc = np.float32(0)
            for k in range(K):
                acc = np.float32(np.float64(a[i, k]) * np.float64(w[j, k]) + np.float64(acc))
            assert want[i, j] == np.float32(np.float32(acc + b[j]) + r[i, j])


@pytest.mark.parametrize("form", range(11))
def test_each_form_convolves(gpu, form):
    """the same kernels on a convolution's input against the column matrix: images of odd sides, strides, pitches wider than the channels, a 1 x 1 image"""
    rows, cols = FORMS[form]
    rng = np.random.default_rng(form)
    for images, H, W, ch, ld, kw, stride, pad in ((2, 9, 13, 8, 12, 3, 1, 1), (1, 1, 1, 4, 4, 3, 1, 1), (3, 17, 11, 4, 4, 5, 2, 2), (1, 12, 10, 20, 20, 3, 2, 1), (2, 7, 7, 16, 16, 1, 1, 0)):
        N, Ho, Wo = cols - 3, (H + 2 * pad - kw) // stride + 1, (W + 2 * pad - kw) // stride + 1
        x = rng.standard_normal((images, H, W, ld)).astype(np.float32)
        w = rng.standard_normal((N, kw * kw * ch)).astype(np.float32)
        b = rng.standard_normal(N).astype(np.float32)
        full = np.zeros((images, H + 2 * pad, W + 2 * pad, ch), np.float32)
        full[:, pad:pad + H, pad:pad + W] = x[..., :ch]
        cols_of = [full[:, ky:ky + stride * Ho:stride, kx:kx + stride * Wo:stride][:, :Ho, :Wo] for ky in range(kw) for kx in range(kw)]
        a = np.ascontiguousarray(np.stack(cols_of, 3).reshape(images * Ho * Wo, -1))
        got = _form(gpu, form, x, w, w.shape[1], b, None, 1, (ch, H, W, ld, kw, stride, pad, Ho, Wo), a.shape[0])
        want = _form(gpu, 10, a, w, w.shape[1], b, None, 1)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (images, H, W, ch)


@pytest.mark.parametrize("M,N,K,f16", [
    (1, 48, 384, 0), (16, 80, 2048, 0), (7, 64, 1536, 1),               # 16 rows: the whole range in the LDS, waves without a tile, the longest range
    (16, 80, 2176, 0), (3, 48, 4096, 1),                                # in a ring
    (17, 48, 1024, 0), (32, 80, 896, 1), (31, 96, 1152, 0),             # 32 rows: the longest whole range, one of 128s, a ring
    (32, 4112, 256, 0), (1, 8208, 256, 1),                              # more than one tile per wave's workgroup
])
def test_few_rows_with_the_whole_range_or_a_ring(gpu, M, N, K, f16):
    _, _, _, _, cs, ct = _pair(gpu, M, N, K, 0, f16, not f16, False, seed=K + M)
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))


@pytest.mark.parametrize("M,N,K", [(16, 256, 1024), (48, 4096, 512), (256, 64, 256)])
def test_f16_weight_tiles_equal_the_staged_f16_path(gpu, M, N, K):
    """fp16-checkpoint semantics: f16 weights, activations rounded through f16, fp32 chain"""
    a, w, b, r, cs, ct = _pair(gpu, M, N, K, 0, 1, False, False, seed=7)
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))
    i, j = M - 1, N - 1
    acc = np.float32(0)
    for k in range(K):
        acc = np.float32(np.float64(np.float32(np.float16(a[i, k]))) * np.float64(np.float32(np.float16(w[j, k]))) + np.float64(acc))
    assert ct[i, j] == np.float32(acc + np.float32(0))


def test_gemm_pair_rejects_bad_shapes(gpu):
    z = np.zeros(4, np.float32).ctypes.data_as(C.c_void_p)
    assert gpu.lib().tk_mi355x_gemm_pair(0, 4, 4, 100, z, z, None, None, 0, 0, z, z) != 0   # K not a multiple of 128
    assert gpu.lib().tk_mi355x_gemm_pair(0, 0, 4, 128, z, z, None, None, 0, 0, z, z) != 0
    assert gpu.lib().tk_mi355x_gemm_pair(99, 4, 4, 128, z, z, None, None, 0, 0, z, z) != 0
    for form, n, lda in ((-1, 4, 8), (11, 4, 8), (6, 33, 8), (7, 65, 8), (8, 97, 8), (0, 4, 7)):   # no such form, more columns than the tall ones have, a pitch below K
        assert gpu.lib().tk_mi355x_gemm_f32(0, form, 4, n, 8, lda, 8, z, z, None, None, 0, None, z) != 0
