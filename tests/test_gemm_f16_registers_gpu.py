"""The tiled exact product of f16 weights with operands in registers (up to 128 rows; one to four M-tiles a wave): bit for bit the LDS-staged kernel on the same f16-rounded operands."""
import ctypes as C

import numpy as np
import pytest


# rows at the edges of 1 .. 8 M-tiles; fewer tile columns than SIMDs, as many, more (whole workgroups of waves); the first k of four and of eight pieces; first sizes beyond the rule
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,act,res", [
    (1, 16, 128, 0, False), (1, 1, 256, 2, True), (8, 16400, 128, 0, True), (16, 50, 384, 3, True), (16, 16384, 256, 0, False), (17, 384, 384, 0, True), (17, 16400, 128, 2, True),
    (24, 8200, 128, 0, False), (32, 1531, 640, 1, True), (33, 16400, 128, 0, True), (40, 8192, 256, 0, False), (48, 5632, 128, 2, False), (49, 700, 256, 0, True), (64, 16400, 128, 0, True),
    (64, 1024, 2176, 0, False), (65, 3000, 384, 0, True), (96, 16384, 128, 0, False), (113, 5632, 128, 1, True), (128, 9000, 128, 0, True), (128, 24600, 128, 0, False), (129, 512, 256, 0, True)])
def test_f16_registers_equal_staged(gpu, M, N, K, act, res):
    rng = np.random.default_rng(M + N + K)
    f = lambda *s: rng.normal(0, 1, s).astype(np.float32)
    a, w, b, r = f(M, K), f(N, K) * np.float32(K ** -0.5), f(N), f(M, N) if res else None
    cs, ct = np.empty((M, N), np.float32), np.empty((M, N), np.float32)
    p = lambda x: x.ctypes.data_as(C.c_void_p) if x is not None else None
    gpu.check(gpu.lib().tk_mi355x_gemm_pair(0, M, N, K, p(a), p(w), p(b), p(r), act, 1, p(cs), p(ct)))
    assert np.array_equal(cs.view(np.uint32), ct.view(np.uint32))
