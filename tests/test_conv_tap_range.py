"""Images and dilations whose taps lie far from one another: the pipelined kernel works their offsets out in 24-bit factors."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi

RQ = capi.requant(1 << 30, 1, 0, -128, 127)

# (image, filter, stride, dilation, taken by the pipelined kernel)
CASES = [
    ((1, 4200, 4200, 16), (72, 5, 5, 16), (1, 1), (1040, 1040), True),    # the last row of taps 4160 x 4200 pixels down: 1.04 x 2^24
    ((1, 3, 524288, 32), (72, 3, 3, 32), (2048, 1), (1, 1), False),       # rows of 2^24 bytes
    ((1, 3, 524287, 32), (72, 3, 3, 32), (2048, 1), (1, 1), True),        # ... and of 32 less
]


def _desc(shape, wshape, stride, dil, rq=RQ):
    return capi.conv_desc(shape[0], shape[1], shape[2], shape[3], wshape[0], wshape[1], wshape[2], stride, (0, 0, 0, 0), dil, capi.S8, capi.S8,
                          capi.S8, 0, 0, 0, rq)


@pytest.mark.parametrize("shape,wshape,stride,dil,pipelined", CASES + [
    ((1, 1, 524288, 32), (72, 1, 3, 32), (2048, 1), (1, 1), True),        # one row of taps: how long an image row is does not count
    ((1, 20000000, 1, 16), (72, 5, 1, 16), (1, 4000), (1, 4194304), False)])  # dilated over 2^24 rows
def test_choice(shape, wshape, stride, dil, pipelined):
    conv = capi.Conv(_desc(shape, wshape, stride, dil))
    assert conv.kernel_name.startswith("implicit_pp_") == pipelined, conv.kernel_name
    conv.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,wshape,stride,dil,pipelined", CASES)
def test_result(shape, wshape, stride, dil, pipelined):
    from gpu_util import announce
    from test_gpu_conv import run_conv
    rng = np.random.default_rng(shape[2])
    src = rng.integers(-128, 128, size=shape, dtype=np.int8)
    w = rng.integers(-127, 128, size=wshape, dtype=np.int8)
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, [40.0 / ((wshape[1] * wshape[2] * shape[3]) ** 0.5 * 74.0 * 74.0)], 1.0)
    announce("conv tap range", shape, wshape, stride, dil)
    got, name = run_conv(src, w, bias, 3, 0, mult, shift, 5, -128, 127, stride, (0, 0, 0, 0), dil)
    assert name.startswith("implicit_pp_") == pipelined, name
    np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, 3, 0, mult, shift, 5, -128, 127, stride, (0, 0, 0, 0), dil))
