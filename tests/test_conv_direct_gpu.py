"""The direct convolution against the exact GEMM over the same column order (64 x 64 kernel, held to the definition elsewhere): the same bits, at sizes that fill no
tile, for every form of cut, one and two sources, upsampled ones, pitches wider than the channels, with and without bias, residual and activation."""
import ctypes as C

import numpy as np
import pytest

p = lambda x: x.ctypes.data_as(C.c_void_p) if x is not None else None


def gemm(gpu, x, w, b, r, k, stride, act):
    B, H, W, ch = x.shape
    ho, wo = (H + 2 * (k // 2) - k) // stride + 1, (W + 2 * (k // 2) - k) // stride + 1
    c = np.empty((B * ho * wo, w.shape[0]), np.float32)
    conv = (C.c_int * 9)(ch, H, W, ch, k, stride, k // 2, ho, wo)
    gpu.check(gpu.lib().tk_mi355x_gemm_f32(0, 10, len(c), w.shape[0], w.shape[1], 0, w.shape[1], p(x), p(w), p(b), p(r), act, conv, p(c)))
    return c.reshape(B, ho, wo, -1)


def wide(rng, a, extra):
    """the same channels in pixels of a wider pitch"""
    out = rng.normal(0, 1, a.shape[:-1] + (a.shape[-1] + extra,)).astype(np.float32)
    out[..., :a.shape[-1]] = a
    return np.ascontiguousarray(out)


def check(gpu, seed, B, H, W, ch, N, k, stride, cut=None, split=0, up=(0, 0), pad=(0, 0, 0, 0), bias=True, res=False, act=1):
    rng = np.random.default_rng(seed)
    f = lambda *s: rng.normal(0, 1, s).astype(np.float32)
    c0 = split or ch
    x0 = f(B, H >> up[0], W >> up[0], c0)
    x1 = f(B, H >> up[1], W >> up[1], ch - c0) if split else None
    grow = lambda a, u: a.repeat(2, 1).repeat(2, 2) if u else a
    x = np.ascontiguousarray(np.concatenate([grow(x0, up[0]), grow(x1, up[1])], 3)) if split else grow(x0, up[0])
    w, b = f(N, k * k * ch) * np.float32((k * k * ch) ** -0.5), f(N) if bias else None
    ho, wo = (H + 2 * (k // 2) - k) // stride + 1, (W + 2 * (k // 2) - k) // stride + 1
    r = f(B, ho, wo, N) if res else None
    want = gemm(gpu, np.ascontiguousarray(x), w, b, r, k, stride, act)
    y = np.full((B, ho, wo, N + pad[2]), 7.0, np.float32)
    xs0, xs1, rs = wide(rng, x0, pad[0]), wide(rng, x1, pad[1]) if split else None, wide(rng, r, pad[3]) if res else None
    shape = (C.c_int * 15)(B, H, W, ch, c0, c0 + pad[0], up[0], ch - c0 + pad[1] if split else 0, up[1], k, stride, N, N + pad[2], N + pad[3] if res else 0, act)
    gpu.check(gpu.lib().tk_mi355x_conv_direct(0, shape, cut and (C.c_int * 5)(*cut), p(xs0), p(xs1), p(w), p(b), p(rs), p(y), None))
    assert np.array_equal(y[..., :N].view(np.uint32), want.view(np.uint32))
    assert (y[..., N:] == 7.0).all()


CUTS = [(1, 1, 1, 4, 4), (1, 1, 2, 3, 5), (1, 2, 2, 4, 8), (2, 1, 4, 6, 5), (2, 2, 3, 1, 13), (4, 1, 2, 8, 8), (4, 4, 1, 7, 10), (2, 8, 1, 3, 24), (1, 1, 8, 2, 8)]


@pytest.mark.gpu
@pytest.mark.parametrize("cut", CUTS)
@pytest.mark.parametrize("k,stride", [(3, 1), (3, 2), (1, 1)])
def test_every_cut_gives_the_gemms_bits(gpu, cut, k, stride):
    check(gpu, 1, 2, 19, 23, 16, 37, k, stride, cut, pad=(4, 0, 3, 1), res=True)
    check(gpu, 2, 1, 8, 8, 48, 16, k, stride, cut, act=0, bias=False)
    check(gpu, 3, 3, 5, 7, 80, 80, k, stride, cut, split=64, pad=(0, 8, 0, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("size", [(1, 1, 1, 16, 1), (1, 40, 40, 64, 64), (1, 20, 20, 256, 80), (5, 13, 31, 32, 33), (2, 3, 160, 16, 16), (33, 6, 5, 128, 144)])
@pytest.mark.parametrize("k,stride", [(3, 1), (3, 2), (1, 1), (1, 2)])
def test_its_own_cut(gpu, size, k, stride):
    check(gpu, 4, *size, k, stride, res=True)


@pytest.mark.gpu
@pytest.mark.parametrize("N,out,res", [(16, 0, 0), (80, 4, 8), (80, 2, 0), (80, 0, 3), (79, 1, 1), (78, 0, 2), (20, 12, 4)])
def test_four_channels_of_a_pixel_at_once_and_one_by_one(gpu, N, out, res):
    """outputs and residuals whose pixels are whole aligned fours of channels, and such that are not"""
    check(gpu, 7, 2, 9, 11, 32, N, 3, 1, pad=(0, 0, out, res), res=True)
    check(gpu, 8, 2, 9, 11, 32, N, 3, 2, (2, 1, 2, 2, 7), pad=(0, 0, out, 0), bias=False, act=0)


@pytest.mark.gpu
@pytest.mark.parametrize("up", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_two_sources(gpu, up):
    check(gpu, 5, 2, 12, 18, 96, 40, 1, 1, split=32, up=up, pad=(4, 12, 0, 0))
    check(gpu, 6, 1, 6, 4, 64, 16, 3, 1, split=48, up=up)


@pytest.mark.gpu
def test_what_it_does_not_take(gpu):
    z = np.zeros(1 << 16, np.float32)
    bad = [(1, 4, 4, 24, 24, 24, 0, 0, 0, 3, 1, 16, 16, 0, 1), (1, 4, 4, 16, 16, 18, 0, 0, 0, 3, 1, 16, 16, 0, 1), (1, 4, 4, 16, 16, 16, 0, 0, 0, 5, 1, 16, 16, 0, 1),
           (1, 4, 4, 16, 16, 16, 0, 0, 0, 3, 3, 16, 16, 0, 1), (1, 5, 4, 16, 16, 16, 1, 0, 0, 3, 1, 16, 16, 0, 1), (1, 4, 4, 16, 16, 16, 0, 0, 0, 3, 1, 16, 16, 0, 2)]
    for s in bad:
        assert gpu.lib().tk_mi355x_conv_direct(0, (C.c_int * 15)(*s), None, p(z), None, p(z), None, None, p(z), None) != 0
    ok = (C.c_int * 15)(1, 64, 64, 16, 16, 16, 0, 0, 0, 3, 1, 16, 16, 0, 1)
    for cut in [(8, 1, 1, 4, 4), (1, 1, 1, 5, 5), (1, 3, 3, 4, 4), (1, 1, 0, 4, 4)]:
        assert gpu.lib().tk_mi355x_conv_direct(0, ok, (C.c_int * 5)(*cut), p(z), None, p(z), None, None, p(z), None) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,batch", [(32, 32, 1), (96, 64, 3), (1344, 32, 1), (32, 1056, 2), (1568, 1344, 1)])
def test_stem_pools_and_heads_at_odd_maps(gpu, w, h, batch):
    """whole network at maps that fill no tile of the stem (32 x 8 outputs), with a pooled map of one pixel to one that no longer fits the LDS: frames (the stem pre-processes)
    against the pre-processed tensor, and a frame alone against the same frame in a batch"""
    det = gpu.ObjectDetector(model="synthetic://yolov8n?seed=5&cls_bias=-0.5", width=w, height=h, max_batch=batch, conf=0.3)
    rng = np.random.default_rng(w)
    frames = [rng.integers(0, 256, (37, 53, 3), np.uint8) for _ in range(batch)]
    got = det.detect_batch(frames) if batch > 1 else [det.detect(frames[0])]
    planar = np.stack([gpu.preprocess(f, w, h) for f in frames])
    raw = det.forward_raw(np.ascontiguousarray(planar.transpose(0, 2, 3, 1)))
    for b, f in enumerate(frames):
        one = gpu.ObjectDetector(model="synthetic://yolov8n?seed=5&cls_bias=-0.5", width=w, height=h, max_batch=1, conf=0.3)
        assert one.detect(f) == got[b] and len(got[b]) > 0
        boxes, cls, anchors = one.last_boxes()
        det.detect_batch(frames) if batch > 1 else det.detect(f)
        assert np.array_equal(one.forward_raw(np.ascontiguousarray(planar[b:b + 1].transpose(0, 2, 3, 1))).view(np.uint32), raw[b:b + 1].view(np.uint32))
        again, cls2, anchors2 = one.last_boxes()
        assert np.array_equal(boxes.view(np.uint32), again.view(np.uint32)) and np.array_equal(cls, cls2) and np.array_equal(anchors, anchors2)
