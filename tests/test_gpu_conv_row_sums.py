"""Weights with an offset: the kernels of the implicit convolution take the row sums of the patches from the operand blocks
they multiply. One case per kernel form, with what can go wrong there: K that ends inside a step, channels padded to 16,
padded taps (the padding value counts), several panels of columns, K slices, the float destination."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, to_dev
from test_gpu_conv import run_conv

pytestmark = pytest.mark.gpu

# (src, weights, stride, padding, dilation, kernel the name of which starts with)
CASES = [
    ((2, 9, 11, 16), (24, 3, 3, 16), (1, 1), (1, 1, 1, 1), (1, 1), "implicit_narrow"),     # K = 144 of 192
    ((3, 12, 10, 24), (40, 3, 3, 24), (2, 1), (1, 0, 1, 2), (1, 1), "implicit_narrow"),    # 24 channels in 32, K = 288
    ((1, 17, 15, 40), (64, 5, 5, 40), (1, 2), (2, 2, 2, 2), (1, 1), "implicit_pp"),        # 40 in 48, K = 1200: past the narrow kernel
    ((2, 20, 20, 64), (200, 1, 1, 64), (1, 1), (0, 0, 0, 0), (1, 1), "implicit_narrow"),   # 4 panels
    ((2, 8, 8, 128), (64, 3, 3, 128), (1, 1), (1, 1, 1, 1), (1, 1), "implicit_narrow"),    # 6 batches of k blocks
    ((4, 56, 57, 64), (48, 3, 3, 64), (1, 1), (1, 1, 1, 1), (1, 1), "implicit_narrow"),    # images below the band form's
    ((32, 56, 56, 60), (33, 3, 3, 60), (1, 1), (1, 1, 1, 1), (1, 1), "implicit_band"),     # band, 60 channels in 64
    ((32, 56, 56, 64), (130, 1, 1, 64), (1, 1), (0, 0, 0, 0), (1, 1), "implicit_band"),    # band, 3 panels
    ((5, 13, 12, 32), (70, 3, 3, 32), (1, 1), (1, 1, 1, 1), (2, 1), "implicit_pp"),        # pipelined, K = 288 of 3 steps
    ((6, 28, 28, 136), (128, 3, 3, 136), (1, 1), (1, 1, 1, 1), (1, 1), "implicit_pp"),     # 136 in 144
    ((1, 7, 7, 512), (512, 3, 3, 512), (1, 1), (1, 1, 1, 1), (1, 1), "implicit_pp"),       # K slices
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("dt,w_dt", [(np.uint8, np.uint8), (np.int8, np.uint8), (np.uint8, np.int8)])
def test_row_sums_in_the_kernel(case, dt, w_dt):
    shape, wshape, stride, pad, dil, kernel = CASES[case]
    rng = np.random.default_rng(900 + case)
    info, w_info = np.iinfo(dt), np.iinfo(w_dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(w_info.min, w_info.max + 1, size=wshape).astype(w_dt)
    zp, w_zp, ozp = (int(rng.integers(i.min + 60, i.max - 60)) for i in (info, w_info, info))
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    K = wshape[1] * wshape[2] * wshape[3]
    per_channel = case % 2 == 1
    scales = rng.uniform(0.5, 2.0, size=wshape[0] if per_channel else 1) * 40.0 / (K ** 0.5 * 74.0 * 74.0)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, scales, 1.0)
    announce("conv row sums", shape, wshape, stride, pad, dil, dt.__name__, w_dt.__name__, zp, w_zp)
    got, name = run_conv(src, w, bias, zp, w_zp, mult, shift, ozp, info.min, info.max, stride, pad, dil)
    assert name.startswith(kernel), name
    # (large images: the first and the last one)
    rows = list(range(shape[0])) if shape[0] <= 6 else [0, shape[0] - 1]
    for n in rows:
        want = oracle.conv_nhwc_direct(src[n:n + 1], w, bias, zp, w_zp, mult, shift, ozp, info.min, info.max, stride, pad, dil)
        np.testing.assert_array_equal(got[n:n + 1], want)


@pytest.mark.parametrize("shape,OFM,k", [((1, 7, 7, 512), 512, 3), ((2, 9, 9, 48), 40, 3), ((32, 56, 56, 64), 64, 1), ((5, 13, 12, 32), 70, 3)])
def test_row_sums_with_a_float_destination(shape, OFM, k):
    """The float of the product and the float of the offset terms are rounded apart: K slices must not mix them."""
    rng = np.random.default_rng(sum(shape))
    B_, H, W, C = shape
    src = rng.integers(-128, 128, size=shape).astype(np.int8)
    w = rng.integers(-128, 128, size=(OFM, k, k, C)).astype(np.int8)
    p, zp, w_zp, scale = k // 2, 5, -7, 1e-4
    d = capi.conv_desc(B_, H, W, C, OFM, k, k, (1, 1), (p, p, p, p), (1, 1), capi.S8, capi.S8, capi.F32, -zp, -w_zp, zp, scale=scale)
    out = to_dev(np.zeros((B_, H, W, OFM), np.float32))
    cv = capi.Conv(d)
    cv.prepare(to_dev(w))
    cv.run(to_dev(src), out)
    got = out.cpu().numpy().reshape(B_, -1, OFM)
    announce("conv row sums f32", shape, OFM, k, cv.kernel_name)
    cv.close()
    wm = oracle.weights_reshape(w)
    for n in {0, B_ - 1}:
        cols = oracle.im2col_nhwc(src[n:n + 1], k, k, (1, 1), (p, p, p, p), (1, 1), zp)
        want = oracle.gemmlowp_f32(cols, wm, None, -zp, -w_zp, scale)
        np.testing.assert_array_equal(got[n].view(np.uint32), np.asarray(want).view(np.uint32))
