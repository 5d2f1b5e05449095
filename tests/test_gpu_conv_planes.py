"""NCHW destinations written by the pipelined kernel itself: planes of a multiple of 16, of 4 and of an odd number of pixels, tiles
that cross images and end inside one, output channels around a tile, both signs with and without a weights offset, and a negative
multiplier, which takes the general formula."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce
from test_gpu_conv import run_conv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,wshape,stride,pad", [
    ((3, 9, 7, 64), (70, 3, 3, 64), (1, 1), (1, 1, 1, 1)),
    ((2, 10, 10, 48), (130, 3, 3, 48), (1, 1), (1, 1, 1, 1)),
    ((5, 28, 28, 32), (96, 3, 3, 32), (1, 1), (1, 1, 1, 1)),
    ((9, 5, 5, 256), (65, 1, 1, 256), (1, 1), (0, 0, 0, 0)),
    ((32, 16, 16, 128), (128, 3, 3, 128), (1, 1), (1, 1, 1, 1)),
    ((7, 15, 13, 40), (200, 5, 5, 40), (2, 1), (2, 2, 2, 2))])
@pytest.mark.parametrize("dt,w_dt,negative", [(np.int8, np.int8, False), (np.uint8, np.uint8, False), (np.int8, np.int8, True)])
def test_planes(shape, wshape, stride, pad, dt, w_dt, negative):
    rng = np.random.default_rng(sum(shape) + sum(wshape))
    info, w_info = np.iinfo(dt), np.iinfo(w_dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(w_info.min, w_info.max + 1, size=wshape).astype(w_dt)
    zp, w_zp = (3, 0) if dt == np.int8 else (120, 131)
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    reals = rng.uniform(0.5, 2.0, size=wshape[0]) * 40.0 / ((wshape[1] * wshape[2] * shape[3]) ** 0.5 * 74.0 * 74.0)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, reals, 1.0)
    if negative:
        mult = [-m if i % 3 == 0 else m for i, m in enumerate(mult)]
    announce("conv planes", shape, wshape, dt.__name__, "negative", negative)
    got, name = run_conv(src, w, bias, zp, w_zp, mult, shift, 5, info.min, info.max, stride, pad, (1, 1), layout=capi.NCHW)
    assert name.startswith("implicit_pp") and "splitk" not in name, name
    np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, zp, w_zp, mult, shift, 5, info.min, info.max, stride, pad, (1, 1)))


def test_planes_take_no_second_destination():
    """A run whose kernel writes the planes itself holds no buffer of the destination's size in another layout (51 MB here)."""
    import torch
    rng = np.random.default_rng(77)
    conv = capi.Conv(capi.conv_desc(32, 56, 56, 16, 512, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), capi.S8, capi.S8, capi.S8, 0, 0, 0,
                                    capi.requant(1 << 30, 8, 0, -128, 127, False), layout=capi.NCHW))
    src = torch.from_numpy(rng.integers(-128, 128, size=(32, 16, 56, 56), dtype=np.int8)).cuda()
    w = torch.from_numpy(rng.integers(-128, 128, size=(512, 16, 1, 1), dtype=np.int8)).cuda()
    out = torch.zeros((32, 512, 56, 56), dtype=torch.int8, device="cuda")
    conv.prepare(w)
    torch.cuda.synchronize()
    announce("conv planes, memory of the first run")
    before = torch.cuda.mem_get_info()[0]
    conv.run(src, out)
    torch.cuda.synchronize()
    taken, name = before - torch.cuda.mem_get_info()[0], conv.kernel_name
    conv.close()
    assert name.startswith("implicit_pp") and "splitk" not in name, name
    assert taken < out.numel() // 2, taken
