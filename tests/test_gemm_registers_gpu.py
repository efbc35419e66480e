"""The tiled exact product with operands in registers (f32 weights, up to five 16 x 16 tiles for eight SIMDs): bit for bit the LDS-staged kernel, and so at the first sizes beyond."""
import ctypes as C

import numpy as np
import pytest


# one piece of weights in flight more than there are, four and eight of them; longer than the LDS forms take; last tiles of 1 .. 16 rows and columns; 640 tiles and 656
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,act,res", [
    (1, 16, 128, 0, False), (1, 1, 256, 2, True), (15, 50, 512, 1, True), (16, 384, 384, 0, True), (17, 1531, 384, 2, False), (31, 512, 640, 3, True), (32, 5120, 1280, 0, False),
    (33, 384, 1536, 0, True), (5, 1280, 2176, 2, True), (3, 700, 5120, 0, True), (160, 1024, 128, 2, True), (161, 1024, 128, 0, False), (1, 10240, 256, 0, True), (1, 10256, 256, 0, True),
    (640, 16, 512, 1, False), (10225, 16, 128, 0, True)])
def test_registers_equal_staged(gpu, M, N, K, act, res):
    rng = np.random.default_rng(M + N + K)
    f = lambda *s: rng.normal(0, 1, s).astype(np.float32)
    a, w, b, r = f(M, K), f(N, K) * np.float32(K ** -0.5), f(N), f(M, N) if res else None
    cs, ct = np.empty((M, N), np.float32), np.empty((M, N), np.float32)
    p = lambda x: x.ctypes.data_as(C.c_void_p) if x is not None else None
    gpu.check(gpu.lib().tk_mi355x_gemm_pair(0, M, N, K, p(a), p(w), p(b), p(r), act, 0, p(cs), p(ct)))
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))
