"""The tiles whose waves all load and all multiply: sizes at the edges of a tile, of a K step and of the ring's depth (K of 1 to
NS + 2 steps, ending inside a step, a 16-byte column or on a boundary), both signs of A, every destination; and the
convolution's loader where taps lie outside the image for no, some and all lanes of a load."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, run_gemm
from test_gpu_conv import run_conv

pytestmark = pytest.mark.gpu

NAMES = ["pp_128x128x128_s3", "pp_128x64x128_s3", "pp_64x64x128_s3", "pp_64x64x128_s6", "pp_128x64x256_s3", "pp_128x128x128_s2",
         "pp_64x64x256_s2"]


@pytest.mark.parametrize("cfg", range(1, 8))
@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (63, 65, 128), (65, 64, 132), (128, 127, 256), (129, 129, 384), (64, 130, 500),
                                   (200, 96, 512), (127, 63, 768), (70, 40, 1020), (130, 257, 1536)])
def test_dense(cfg, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K + cfg)
    for dt in (np.uint8, np.int8):
        lo, hi = np.iinfo(dt).min, np.iinfo(dt).max
        A = rng.integers(lo, hi + 1, size=(M, K)).astype(dt)
        B = rng.integers(-128, 128, size=(K, N), dtype=np.int8)
        announce("ring tiles", NAMES[cfg - 1], (M, N, K), dt.__name__)
        ao, bo = -5, 9
        got, name = run_gemm(A, B, capi.EPI_S32, np.int32, ao, bo, path=capi.PATH_TILE + cfg, device=True, ldd=N + 3)
        if ((K + 127) // 128 * 128) % int(NAMES[cfg - 1].split("x")[2].split("_")[0]) == 0:
            assert name == NAMES[cfg - 1], name
        np.testing.assert_array_equal(got, oracle.gemmlowp_s32(A, B, ao, bo))
        bias = rng.integers(-20000, 20000, size=N, dtype=np.int32)
        mult, shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(0.5, 2.0, size=N) * 40.0 / (K ** 0.5 * 74.0 * 74.0), 1.0)
        for ldd in (N, (N + 15) // 16 * 16):
            got, _ = run_gemm(A, B, capi.EPI_FIXEDPOINT, dt, ao, bo, bias, mult, shift, 7, lo, hi, path=capi.PATH_TILE + cfg, device=True, ldd=ldd)
            np.testing.assert_array_equal(got, oracle.gemmlowp_fixedpoint(A, B, bias, ao, bo, mult, shift, 7, lo, hi, dt))
        if dt == np.int8:
            got, _ = run_gemm(A, B, capi.EPI_F32, np.float32, ao, bo, scale=3e-4, path=capi.PATH_TILE + cfg, device=True)
            np.testing.assert_array_equal(got.view(np.uint32), np.asarray(oracle.gemmlowp_f32(A, B, None, ao, bo, 3e-4)).view(np.uint32))


# (image, filter, stride, padding, dilation): no padding at all (every lane inside), a padding wider than a load's 8 pixels (none
# inside), odd ones; K of one step, ending inside a step, deeper than the ring; rows of both tile heights
@pytest.mark.parametrize("shape,wshape,stride,pad,dil", [
    ((3, 9, 11, 128), (70, 1, 1, 128), (1, 1), (0, 0, 0, 0), (1, 1)),
    ((2, 20, 21, 64), (130, 3, 3, 64), (1, 1), (0, 0, 0, 0), (1, 1)),
    ((2, 5, 6, 112), (72, 3, 3, 112), (1, 1), (12, 12, 12, 12), (3, 2)),
    ((1, 13, 40, 272), (90, 5, 5, 272), (2, 1), (2, 10, 1, 0), (1, 2)),
    ((40, 16, 15, 64), (200, 3, 3, 64), (1, 1), (1, 1, 1, 1), (1, 1)),
    ((9, 30, 31, 144), (128, 3, 3, 144), (1, 1), (1, 1, 1, 1), (1, 1))])
@pytest.mark.parametrize("dt,w_dt", [(np.int8, np.int8), (np.uint8, np.uint8)])
def test_convolution(shape, wshape, stride, pad, dil, dt, w_dt):
    rng = np.random.default_rng(sum(shape) + sum(wshape))
    info, w_info = np.iinfo(dt), np.iinfo(w_dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(w_info.min, w_info.max + 1, size=wshape).astype(w_dt)
    zp, w_zp = (3, 0) if dt == np.int8 else (120, 131)
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, [40.0 / ((wshape[1] * wshape[2] * shape[3]) ** 0.5 * 74.0 * 74.0)], 1.0)
    announce("ring tiles, convolution", shape, wshape, dt.__name__)
    got, name = run_conv(src, w, bias, zp, w_zp, mult, shift, 5, info.min, info.max, stride, pad, dil)
    assert name.startswith("implicit_"), name
    np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, zp, w_zp, mult, shift, 5, info.min, info.max, stride, pad, dil))
