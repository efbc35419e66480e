"""SiLU, GELU and sigmoid as the kernels evaluate them (fewer instructions than the host's forms, the same values): bit for bit what the oracle's library gives,
where the forms part: the clamps of exp, the sigmoid's subnormal end, denominators of every exponent, zeros, subnormals, infinities and NaN."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O


def inputs():
    rng = np.random.default_rng(3)
    edges = np.array([0.0, -0.0, 1.0, -1.0, 43.5, 44.0, 44.5, 86.9, 87.0, 87.3365, 87.34, 87.99, 88.0, 88.01, 88.7, 100.0, 1e4, 1e30, 3.4e38, 1e-30, 1e-38, 1e-45, np.inf, np.nan], np.float32)
    near = (edges[8:15].view(np.int32)[:, None] + np.arange(-40, 41, dtype=np.int32)).reshape(-1).view(np.float32)  # steps of one unit around the clamps
    bits = rng.integers(0, 1 << 32, 6000, np.uint64).astype(np.uint32).view(np.float32)  # every exponent
    x = np.concatenate([edges, -edges, near, -near, bits, rng.uniform(-90, 90, 8000).astype(np.float32), rng.normal(0, 2, 6000).astype(np.float32)])
    return np.concatenate([x, np.zeros(-len(x) % 64, np.float32)])


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 5, 6, 9, 10])
@pytest.mark.parametrize("act", [1, 2, 3])
def test_activations_of_the_kernels_are_the_hosts(gpu, act, form):
    x, L, f32 = inputs(), O.lib(), np.float32
    a = np.zeros((len(x), 4), f32)
    a[:, 0] = x
    a[np.isinf(x), 0] = 0.0  # an infinity would meet the row's zeros in the product
    w = np.zeros((16, 4), f32)
    w[:, 0] = 1.0
    c = np.zeros((len(x), 16), f32)
    p = lambda t: t.ctypes.data_as(C.POINTER(C.c_float))
    gpu.check(gpu.lib().tk_mi355x_gemm_f32(0, form, len(x), 16, 4, 4, 4, p(a), p(w), None, None, act, None, p(c)))
    with np.errstate(all="ignore"):
        v = a[:, 0] + f32(0.0)  # the chain starts from +0
        if act == 1:
            want = np.array([L.orc_siluf(float(t)) for t in v], f32)
        elif act == 2:
            want = np.array([L.orc_geluf(float(t)) for t in v], f32)
        else:
            want = f32(1.0) / (f32(1.0) + np.array([L.orc_expf(float(-t)) for t in v], f32))
    for n in (0, 7, 15):
        same = (c[:, n].view(np.uint32) == want.view(np.uint32)) | (np.isnan(c[:, n]) & np.isnan(want))
        assert same.all(), [(float(v[i]), float(c[i, n]), float(want[i])) for i in np.flatnonzero(~same)[:5]]


@pytest.mark.gpu
def test_f16_rounding_of_the_kernels_is_the_host_arithmetic(gpu):
    """every 16-bit result's neighbourhood: halfway points and one unit to either side, subnormals, overflow, infinities, NaN of both signs"""
    half = np.arange(0, 0x7C01, dtype=np.uint16).view(np.float16).astype(np.float32)
    half[-1] = 65536.0  # the value that infinity stands for in the spacing of the last finite ones
    mid = ((half[:-1].astype(np.float64) + half[1:]) / 2).astype(np.float32)  # exact
    near = [(t.view(np.int32) + d).view(np.float32) for t in (half, mid) for d in (-1, 0, 1)]
    bits = np.random.default_rng(8).integers(0, 1 << 32, 1 << 18, np.uint64).astype(np.uint32).view(np.float32)
    x = np.concatenate(near + [-t for t in near] + [bits, np.array([0x7F800000, 0xFF800000, 0x7FC00000, 0xFFC00000, 0x7F800001, 0xFFBFFFFF, 0, 0x80000000, 1, 0x80000001], np.uint32).view(np.float32)])
    got = np.zeros(len(x), np.uint16)
    gpu.check(gpu.lib().tk_mi355x_f32_to_f16(0, x.ctypes.data_as(C.POINTER(C.c_float)), len(x), got.ctypes.data_as(C.POINTER(C.c_uint16))))
    with np.errstate(all="ignore"):
        want = x.astype(np.float16).view(np.uint16)
    nan = np.isnan(x)
    want[nan] = np.where(np.signbit(x[nan]), 0xFE00, 0x7E00)
    bad = np.flatnonzero(got != want)
    assert len(bad) == 0, [(hex(int(x.view(np.uint32)[i])), hex(int(got[i])), hex(int(want[i]))) for i in bad[:5]]
