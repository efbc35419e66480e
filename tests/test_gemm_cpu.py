"""Which blocks a matrix product is cut into: the choice is made on the host, so it is held here; the kernels themselves are in the GPU tests."""
import ctypes as C

import pytest

import trackiellm_amd as tk
from layered_util import LARGE_PRODUCTS


def image_form(f32, rows, n, k, swiglu=0, experts=0, top=0, slabs=1):
    form = (C.c_int * 4)()
    assert tk.lib().tk_mi355x_gemm_image_form(f32, rows, n, k, swiglu, experts, top, slabs, form) == 0
    return tuple(form)


@pytest.mark.parametrize("rows,n,k,swiglu,slabs,want", [
    (2047, 7552, 4096, 0, 1, (256, 256, 2, 1)),
    (1303, 7552, 4096, 0, 1, (128, 128, 2, 1)),   # 256 x 256: 180 blocks, one round of 940 us; three rounds of a quarter each: 715
    (1303, 6192, 2080, 0, 1, (128, 64, 3, 1)),    # 318 us, 256 x 256 480
    (2047, 3072, 2048, 0, 1, (128, 64, 3, 1)),    # 202 us, 256 x 128 257
    (900, 4096, 14336, 0, 1, (128, 128, 4, 1)),
    (900, 28672, 4096, 1, 1, (128, 128, 2, 1)),   # 1656 us, 256 x 256 1886
    (256, 3072, 2048, 0, 8, (128, 64, 3, 8)),     # as many parts as 128 x 128 blocks leave room for: the error, not the time
    (900, 2048, 8192, 0, 2, (128, 128, 4, 2)),
])
def test_blocks_of_float32_products(rows, n, k, swiglu, slabs, want):
    """the choice is that of measured times: an f32 MFMA takes sixteen times as long as a bf16 one for the same k, so rounds half empty cost more than anything else"""
    assert image_form(1, rows, n, k, swiglu, slabs=slabs) == want


@pytest.mark.parametrize("rows,n,k,swiglu,want", [
    (1750, 28672, 4096, 1, (256, 256, 2, 1)), (2047, 4096, 14336, 0, (256, 128, 3, 1)), (1100, 28672, 4096, 1, (128, 128, 2, 1)),
    (1750, 2048, 8192, 0, (128, 128, 4, 1)), (600, 2048, 8192, 0, (128, 64, 3, 1)), (200, 4096, 14336, 0, (128, 32, 4, 1)), (2047, 1024, 512, 0, (128, 64, 3, 1)), (1100, 2048, 512, 0, (128, 128, 4, 1)), (64, 4096, 4096, 0, (64, 0, 0, 1)),
])
def test_blocks_of_bf16_products(rows, n, k, swiglu, want):
    assert image_form(0, rows, n, k, swiglu) == want


@pytest.mark.parametrize("f32", [0, 1])
def test_sizes_of_the_large_products_reach_every_form(f32):
    """the sizes that the GPU test takes (q, k, v in one product, then out, gate with up, down)"""
    plain, swiglu = set(), set()
    for width, ff, rows in LARGE_PRODUCTS:
        slabs = min(8, 2048 // rows)
        plain |= {image_form(f32, rows, 3 * width, width)[:3], image_form(f32, rows, width, width, slabs=slabs)[:3], image_form(f32, rows, width, ff, slabs=slabs)[:3]}
        swiglu.add(image_form(f32, rows, 2 * ((ff + 15) // 16 * 16), width, 1)[:3])
    forms = {(256, 256, 2), (256, 128, 3), (128, 128, 2), (128, 128, 4), (128, 64, 3)}
    assert swiglu == forms and plain == forms | {(128, 32, 4)}


@pytest.mark.parametrize("f32,rows,n,k,swiglu,experts,top,want", [
    (1, 2047, 1024, 2048, 0, 8, 2, (128, 32, 4, 1)),    # 182 us, 128 x 128 242
    (1, 1200, 512, 256, 1, 6, 3, (128, 64, 3, 1)),      # 31 blocks of 34 are live: 248 of 272 workgroups, one round.  13.5 us, 128 x 128 20.5
    (0, 1200, 1024, 2048, 0, 8, 2, (128, 128, 4, 1)),
    (0, 2047, 2048, 2048, 1, 64, 8, (128, 128, 2, 1)),
])
def test_blocks_of_experts(f32, rows, n, k, swiglu, experts, top, want):
    """row blocks come from the router; how many there will be is estimated"""
    assert image_form(f32, rows, n, k, swiglu, experts, top) == want


def f32_form(m, n, k, pad=0, batch=1, conv=None):
    form, block = C.c_int(), (C.c_int * 2)()
    ld = k + pad
    rc = tk.lib().tk_mi355x_gemm_f32_form(m, n, k, ld, k if conv else ld, batch, conv and (C.c_int * 9)(*conv), C.byref(form), block)
    assert rc == 0
    return form.value, tuple(block)


def conv3(c, side, stride, images):
    out = (side - 1) // stride + 1
    return images * out * out, 9 * c, (c, side, side, c, 3, stride, 1, out, out)


@pytest.mark.parametrize("m,n,k,pad,batch,block", [
    # side by side, short or unaligned: 0.55 - 0.75 of the speed where the 16 x 16 x 4 forms took them
    (255, 201, 400, 0, 48, (64, 64)), (1500, 80, 27, 1, 48, (64, 64)), (100, 1500, 64, 0, 48, (64, 64)), (102400, 80, 64, 0, 1, (128, 96)), (102400, 80, 64, 1, 1, (128, 96)),
    (25600, 96, 27, 1, 1, (128, 128)), (1500, 16, 27, 1, 1, (128, 32)), (6400, 384, 27, 1, 1, (128, 128)), (255, 1500, 64, 0, 48, (64, 64)),
    (400, 256, 1152, 0, 1, (32, 32)), (1, 1, 4608, 0, 1, (32, 32)), (1500, 201, 1152, 1, 6, (64, 80)), (33, 384, 400, 0, 6, (32, 32)),
])
def test_blocks_of_exact_products(m, n, k, pad, batch, block):
    assert f32_form(m, n, k, pad, batch)[1] == block


@pytest.mark.parametrize("c,side,stride,images,n,block", [
    (16, 160, 1, 1, 16, (64, 16)), (128, 20, 1, 1, 128, (32, 32)), (64, 80, 1, 1, 80, (64, 16)), (512, 112, 1, 1, 64, (64, 32)), (32, 160, 2, 32, 64, (128, 64)), (80, 80, 1, 32, 80, (64, 80)),
    (64, 40, 1, 8, 128, (64, 64)), (256, 20, 1, 32, 64, (64, 64)), (128, 80, 1, 8, 80, (128, 80)),
])
def test_blocks_of_convolutions(c, side, stride, images, n, block):
    m, k, conv = conv3(c, side, stride, images)
    assert f32_form(m, n, k, conv=conv)[1] == block


def test_block_hooks_refuse_bad_sizes():
    f = (C.c_int * 4)()
    for args in ((0, 0, 16, 64, 0, 0, 0, 1), (0, 8, 0, 64, 0, 0, 0, 1), (0, 8, 16, 0, 0, 0, 0, 1), (0, 8, 16, 64, 0, 4, 0, 1), (0, 8, 16, 64, 0, 4, 5, 1)):
        assert tk.lib().tk_mi355x_gemm_image_form(*args, f) != 0
    assert tk.lib().tk_mi355x_gemm_image_form(0, 8, 16, 64, 0, 0, 0, 1, None) != 0
