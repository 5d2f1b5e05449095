"""Convolutions of few channels run over patch rows (the KW taps of an image row side by side); byte matrices of every edge
length are turned round between NCHW and NHWC."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce
from test_gpu_conv import run_conv

pytestmark = pytest.mark.gpu

# (src, weights, stride, padding, dilation): image rows shorter than one 16-byte piece, of exactly one, padding wider than a
# piece, window rows of 16 bytes and one more, windows that leave the row on both sides, steps over what the window covers
FEW = [
    ((2, 5, 4, 3), (8, 3, 3, 3), (1, 1), (1, 1, 1, 1), (1, 1)),       # 12-byte rows
    ((1, 7, 16, 1), (5, 5, 5, 1), (1, 1), (2, 2, 2, 2), (1, 1)),      # 16-byte rows, 5 bytes of 16
    ((1, 6, 9, 4), (16, 3, 7, 4), (2, 1), (6, 1, 6, 1), (1, 1)),      # padding of 24 bytes
    ((2, 9, 40, 2), (33, 2, 8, 2), (3, 2), (0, 0, 4, 1), (1, 1)),     # exactly 16 bytes, no padding on the left
    ((1, 11, 23, 1), (70, 3, 17, 1), (1, 1), (8, 1, 8, 1), (1, 1)),   # 17 bytes of 32
    ((3, 33, 31, 3), (64, 7, 7, 3), (2, 2), (3, 3, 3, 3), (1, 1)),
    ((1, 12, 20, 5), (96, 5, 5, 5), (4, 1), (2, 2, 2, 2), (1, 2)),    # dilated down the image
    ((2, 8, 150, 8), (24, 3, 5, 8), (2, 2), (2, 1, 2, 1), (1, 1)),    # several workgroups per row
    ((2, 14, 15, 4), (64, 5, 5, 4), (1, 1), (2, 2, 2, 2), (1, 1)),    # the copy would double: channels padded
    ((2, 14, 15, 4), (65, 5, 5, 4), (1, 1), (2, 2, 2, 2), (1, 1)),    # ... and does, where it saves the pipelined kernel K steps
]


@pytest.mark.parametrize("case", range(len(FEW)))
@pytest.mark.parametrize("dt,w_dt,layout", [(np.uint8, np.int8, capi.NHWC), (np.int8, np.uint8, capi.NHWC), (np.uint8, np.uint8, capi.NCHW)])
def test_patch_rows(case, dt, w_dt, layout):
    _check(700 + case, *FEW[case], dt, w_dt, layout)


@pytest.mark.parametrize("C,H,W", [(16, 4, 4), (17, 5, 7), (31, 9, 15), (128, 8, 16), (129, 3, 43), (144, 16, 16), (272, 1, 16), (48, 1, 15)])
@pytest.mark.parametrize("OFM", [15, 16, 130])
def test_layout_conversion(C, H, W, OFM):
    _check(C + W + OFM, (3, H, W, C), (OFM, 1, 1, C), (1, 1), (0, 0, 0, 0), (1, 1), np.int8, np.int8, capi.NCHW)


@pytest.mark.parametrize("shape,wshape,kernel", [
    ((1, 255, 253, 3), (96, 5, 5, 3), "implicit_pp"),       # 16256 output rows: one column panel after the other does not pay yet
    ((1, 255, 255, 3), (96, 5, 5, 3), "implicit_narrow"),   # 16384
    ((2, 7, 9, 4), (256, 5, 5, 4), "implicit_pp"),
    ((2, 9, 9, 20), (64, 3, 3, 20), "implicit_narrow"),     # K = 192 by rows, 288 by taps: taps
    ((1, 181, 181, 20), (32, 3, 3, 20), "implicit_"),       # 8281 rows: rows
])
@pytest.mark.parametrize("dt,w_dt", [(np.int8, np.int8), (np.uint8, np.uint8)])
def test_patch_rows_follow_the_size(shape, wshape, kernel, dt, w_dt):
    k = wshape[1]
    name = _check(800 + shape[1], shape, wshape, (2, 2), (k // 2,) * 4, (1, 1), dt, w_dt, capi.NHWC)
    assert name.startswith(kernel), name


def test_a_step_too_long_for_patch_rows():
    """One output column and a step whose bytes pass 31 bits: the channels are padded instead"""
    _check(900, (2, 5, 6, 3), (24, 3, 3, 3), (800_000_000, 1), (1, 1, 1, 1), (1, 1), np.int8, np.int8, capi.NHWC)


def _check(seed, shape, wshape, stride, pad, dil, dt, w_dt, layout):
    rng = np.random.default_rng(seed)
    info, w_info = np.iinfo(dt), np.iinfo(w_dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(w_info.min, w_info.max + 1, size=wshape).astype(w_dt)
    zp, w_zp, ozp = (int(rng.integers(i.min + 60, i.max - 60)) for i in (info, w_info, info))
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    scales = rng.uniform(0.5, 2.0, size=wshape[0]) * 40.0 / ((wshape[1] * wshape[2] * wshape[3]) ** 0.5 * 74.0 * 74.0)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, scales, 1.0)
    announce("conv few channels / layouts", shape, wshape, stride, pad, dil, dt.__name__, w_dt.__name__, layout)
    got, name = run_conv(src, w, bias, zp, w_zp, mult, shift, ozp, info.min, info.max, stride, pad, dil, layout=layout)
    want = oracle.conv_nhwc_direct(src, w, bias, zp, w_zp, mult, shift, ozp, info.min, info.max, stride, pad, dil)
    np.testing.assert_array_equal(got, want)
    return name
