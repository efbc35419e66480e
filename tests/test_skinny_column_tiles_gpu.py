"""Products of few rows whose workgroups take two or four column tiles, in one piece and in slabs of parts of k: against 64 bits, and slabs against the whole bit for bit."""
import ctypes as C

import numpy as np
import pytest

from layered_util import attention, config, delta, dense, layer

pytestmark = pytest.mark.gpu


def product(gpu, x, w, most, f32):
    out, n = np.full((8, len(x), len(w)), np.nan, np.float32), C.c_int(0)
    p = lambda t: t.ctypes.data_as(C.c_void_p)
    gpu.check(gpu.lib().tk_mi355x_gemm_image(0, f32, len(x), len(w), x.shape[1], most, p(x), p(w), p(out), C.byref(n)))
    s = out[0]
    for i in range(1, n.value):
        s = s + out[i]
    return s, n.value


def operands(rows, N, K, f32):
    rng = np.random.default_rng(rows + N + K)
    x, w = rng.normal(0, 1, (rows, K)).astype(np.float32), (rng.normal(0, 1, (N, K)) * K ** -0.5).astype(np.float32)
    if not f32:  # what the kernel multiplies: bf16
        x, w = ((t.view(np.uint32) + 0x7fff + ((t.view(np.uint32) >> 16) & 1) & 0xffff0000).view(np.float32) for t in (x, w))
    return x, w


# a last workgroup of one column tile, of one to three of four; rows of one to four tiles, also not filled; sums of K products in f32: sqrt(K) roundings of 2^-24 beside chains of K / 16
@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("N,K", [(6144, 160), (6160, 352), (16368, 96), (24576, 96), (24592, 160), (24608, 96), (24624, 64), (33000, 96)])
@pytest.mark.parametrize("rows", [1, 17, 33, 60])
def test_column_tiles_of_a_workgroup(gpu, rows, N, K, f32):
    x, w = operands(rows, N, K, f32)
    got, n = product(gpu, x, w, 1, f32)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    bound = K * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T)
    assert n == 1 and np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("f32,K", [(0, 4096), (0, 4160), (1, 2048), (1, 2064)])
@pytest.mark.parametrize("rows,N", [(17, 2064), (32, 4096), (33, 2080), (49, 4080), (64, 3000)])
def test_slabs_of_two_column_tiles_add_up_to_the_whole(gpu, rows, N, f32, K):
    x, w = operands(rows, N, K, f32)
    whole, one = product(gpu, x, w, 1, f32)
    parts, n = product(gpu, x, w, 8, f32)
    assert one == 1 and n == 5 and np.array_equal(parts.view(np.uint32), whole.view(np.uint32))


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("N", [2064, 6160, 24576, 28672, 32000, 33000])
def test_a_rows_sums_are_those_of_a_step_of_fewer_rows(gpu, N, f32):
    """bit for bit, within one depth of the loads (up to 32 rows, up to 64), which is also the order of k"""
    x, w = operands(64, N, 528 if f32 else 1056, f32)
    for few, more in ((1, 17), (16, 32), (33, 64)):
        a, b = product(gpu, x[:few], w, 1, f32)[0], product(gpu, x[:more], w, 1, f32)[0]
        assert np.array_equal(a.view(np.uint32), b[:few].view(np.uint32)), (few, more)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_a_sequences_logits_are_those_of_a_step_of_fewer(gpu, dtype):
    """the same for gate and up, 24 608 columns together"""
    m = gpu.LlmModel(config=config(1056, 96, [layer(attention(4, 2, 64, 64, 32, 70, 2), delta(4, 2, 64, 64, 4), dense(12304))]), dtype=dtype, seed=9)
    got = [gpu.LlmSession(m, 32, 8).forward_rows(range(n), [0] * n, range(n), range(n))[0] for n in (16, 17, 32)]
    assert np.array_equal(got[0], got[2][:16]) and np.array_equal(got[1], got[2][:17])
