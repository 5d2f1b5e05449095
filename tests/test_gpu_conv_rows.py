"""Convolutions of few channels straight from the image: window rows of 1 to 32 bytes (one and two pieces, 1 to 4 k blocks), image rows
that start on any byte, bands that end inside an image, padding on every side and wider than a piece, strides, dilation down the image,
both signs, output channels around panels and stores of 16, 4 and 1 byte, per-tensor and per-channel constants with left shifts, and negative
multipliers, which take the general formula. Batches large enough that a workgroup's band is several output rows."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce
from test_gpu_conv import run_conv

pytestmark = pytest.mark.gpu

CASES = [
    ((2, 5, 4, 3), (8, 3, 3, 3), (1, 1), (1, 1, 1, 1), (1, 1)),
    ((1, 7, 17, 1), (5, 5, 5, 1), (1, 1), (2, 2, 2, 2), (1, 1)),
    ((3, 33, 31, 3), (64, 7, 7, 3), (2, 2), (3, 3, 3, 3), (1, 1)),
    ((2, 40, 41, 4), (96, 7, 7, 4), (1, 2), (3, 2, 3, 1), (1, 1)),
    ((1, 6, 9, 4), (16, 3, 7, 4), (2, 1), (6, 1, 6, 1), (1, 1)),
    ((2, 9, 40, 2), (33, 2, 8, 2), (3, 2), (0, 0, 4, 1), (1, 1)),
    ((1, 12, 20, 5), (66, 5, 5, 5), (4, 1), (2, 2, 2, 2), (1, 2)),
    ((5, 64, 65, 3), (24, 5, 5, 3), (2, 2), (2, 2, 2, 2), (1, 1)),
    ((1, 200, 201, 1), (128, 16, 3, 1), (1, 1), (1, 1, 8, 7), (1, 1)),
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("dt", [np.uint8, np.int8])
@pytest.mark.parametrize("how", ["per_channel", "per_tensor", "left_shift", "negative"])
def test_rows(case, dt, how):
    shape, wshape, stride, pad, dil = CASES[case]
    rng = np.random.default_rng(300 + case)
    info = np.iinfo(dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(-127, 128, size=wshape, dtype=np.int8)
    K = wshape[1] * wshape[2] * wshape[3]
    zp, ozp = (5, -7) if dt == np.int8 else (131, 9)
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    if how == "left_shift":
        mult, shift = [1 << 30], [-1]
    else:
        reals = rng.uniform(0.5, 2.0, size=1 if how == "per_tensor" else wshape[0]) * 40.0 / (K ** 0.5 * 74.0 * 74.0)
        mult, shift = oracle.calculate_quantized_multipliers(1.0, reals, 1.0)
        if how == "negative":
            mult = [-m if i % 3 == 0 else m for i, m in enumerate(mult)]
    for layout in (capi.NHWC, capi.NCHW) if how == "per_channel" else (capi.NHWC,):
        announce("conv rows", shape, wshape, stride, pad, dil, dt.__name__, how, layout)
        got, name = run_conv(src, w, bias, zp, 0, mult, shift, ozp, info.min, info.max, stride, pad, dil, layout=layout)
        assert name == "implicit_rows_32x64", name
        np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, zp, 0, mult, shift, ozp, info.min, info.max, stride, pad, dil))


# What a workgroup takes is several output rows where the batch leaves 512 workgroups all the same: (band, rows of the image's last band).
# 1 to 4 k blocks, one panel and two, bands of 2 to 16 rows, window rows off a dword
BANDS = [
    ((130, 11, 9, 3), (8, 3, 3, 3), (1, 1), (1, 1, 1, 1), 3, 2),
    ((64, 26, 22, 3), (96, 5, 5, 3), (2, 2), (2, 2, 2, 2), 4, 1),
    ((128, 21, 17, 4), (33, 5, 5, 4), (1, 2), (2, 2, 2, 2), 3, 2),
    ((300, 35, 32, 3), (5, 7, 7, 3), (1, 1), (3, 3, 3, 3), 16, 3),
    ((130, 15, 16, 3), (66, 7, 7, 3), (2, 2), (3, 3, 3, 3), 7, 1),
    ((257, 12, 70, 5), (16, 3, 5, 5), (2, 3), (0, 0, 0, 0), 3, 1),
]


@pytest.mark.parametrize("case", range(len(BANDS)))
@pytest.mark.parametrize("dt", [np.uint8, np.int8])
def test_bands_of_several_rows(case, dt):
    shape, wshape, stride, pad, band, last = BANDS[case]
    rng = np.random.default_rng(400 + case)
    info = np.iinfo(dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(-127, 128, size=wshape, dtype=np.int8)
    OH, OW = (shape[1] + 2 * pad[1] - wshape[1]) // stride[1] + 1, (shape[2] + 2 * pad[0] - wshape[2]) // stride[0] + 1
    panels = -(-wshape[0] // 64)
    # (conv_rows_plan: no more than 4 tiles of 32 pixels for each of 4 waves, at least 512 workgroups; the windows here are small)
    took = max(b for b in range(1, min(OH, -(-512 // OW)) + 1) if b == 1 or shape[0] * -(-OH // b) * panels >= 512)
    assert (took, OH - (-(-OH // took) - 1) * took) == (band, last)
    zp, ozp = (5, -7) if dt == np.int8 else (131, 9)
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    reals = rng.uniform(0.5, 2.0, size=wshape[0]) * 40.0 / ((wshape[1] * wshape[2] * wshape[3]) ** 0.5 * 74.0 * 74.0)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, reals, 1.0)
    announce("conv rows, bands", shape, wshape, stride, pad, dt.__name__)
    got, name = run_conv(src, w, bias, zp, 0, mult, shift, ozp, info.min, info.max, stride, pad)
    assert name == "implicit_rows_32x64", name
    np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, zp, 0, mult, shift, ozp, info.min, info.max, stride, pad, (1, 1)))
