"""The short form of the requantisation at the ends of what it takes and one past them: shifts of 2 and 22 (1 and 23 go to the general form),
multipliers of 2^30 and 2^31 - 1, result offsets of 511 and 512, and values over the whole range of 32 bits, which the bias brings (A is
zero). In the tiles of the pipelined kernel, the narrow and the band kernel and the one of few channels."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, run_gemm, to_dev, torch_dev

pytestmark = pytest.mark.gpu

SHIFTS = [(2, 2), (22, 22), (2, 22), (1, 22), (2, 23), (0, 31), (-3, 5)]


def _columns(N, shifts, seed):
    rng = np.random.default_rng(seed + 1000)
    edges = [-(1 << 31), (1 << 31) - 1, -(1 << 30), 1 << 30, -1, 0, 1, 3, -2]
    bias = rng.integers(-(1 << 31), 1 << 31, size=N)
    for s in range(2, 24):
        edges += [(1 << s) - 1, 1 << s, -(1 << s), -(1 << s) - 1, 3 << s, -(3 << s) - 1]
    small = rng.integers(-(1 << 31), 1 << 31, size=N) >> rng.integers(0, 31, size=N)
    bias = np.where(rng.random(N) < 0.3, bias, small)
    bias[:len(edges)] = np.clip(edges[:N], -(1 << 31), (1 << 31) - 1)
    mult = np.where(rng.random(N) < 0.3, 1 << 30, np.where(rng.random(N) < 0.4, (1 << 31) - 1, rng.integers(1 << 30, 1 << 31, size=N)))
    shift = rng.integers(shifts[0], shifts[1] + 1, size=N)
    shift[rng.integers(0, N, size=4)] = shifts[0]
    shift[rng.integers(0, N, size=4)] = shifts[1]
    return bias.astype(np.int32), mult.astype(np.int32), shift.astype(np.int32)


@pytest.mark.parametrize("shifts", SHIFTS)
@pytest.mark.parametrize("offset,dtype,lo,hi", [(0, np.int8, -128, 127), (511, np.uint8, 0, 255), (-511, np.int8, -128, 127), (512, np.uint8, 3, 200),
                                                (-3, np.int8, -20, 30)])
def test_tiles(shifts, offset, dtype, lo, hi):
    M, N, K = 70, 320, 64
    A, B = np.zeros((M, K), np.int8), np.ones((K, N), np.int8)
    bias, mult, shift = _columns(N, shifts, offset + shifts[1])
    want = oracle.gemmlowp_fixedpoint(A, B, bias, 0, 0, mult, shift, offset, lo, hi, dtype)
    for path in (capi.PATH_TILE + 0, capi.PATH_TILE + 3):
        announce("requant range", shifts, offset, path)
        got, _ = run_gemm(A, B, capi.EPI_FIXEDPOINT, dtype, 0, 0, bias, mult, shift, offset, lo, hi, path=path, device=True)
        np.testing.assert_array_equal(got, want)


# (narrow: few pixels, band: more than 4 tiles of 32 pixels per compute unit, rows: 3 channels)
@pytest.mark.parametrize("shifts", SHIFTS)
@pytest.mark.parametrize("batch,hw,C,k,kernel", [(1, 9, 64, 1, "narrow"), (3, 112, 64, 1, "band"), (1, 9, 3, 3, "rows")])
def test_convolutions(shifts, batch, hw, C, k, kernel):
    N = 64
    for offset in (7, -511, 512):
        announce("requant range, convolution", shifts, offset, kernel)
        bias, mult, shift = _columns(N, shifts, offset)
        rq = capi.requant(0, 0, offset, -128, 127, True)
        conv = capi.Conv(capi.conv_desc(batch, hw, hw, C, N, k, k, rq=rq))
        oh, ow = conv.out_dims()
        torch = torch_dev()
        src, w = torch.zeros((batch, hw, hw, C), dtype=torch.int8, device="cuda"), torch.ones((N, k, k, C), dtype=torch.int8, device="cuda")
        dst = torch.full((batch, oh, ow, N), 77, dtype=torch.int8, device="cuda")
        keep = [to_dev(x) for x in (bias, mult, shift)]
        conv.prepare(w, *keep)
        conv.run(src, dst)
        torch.cuda.synchronize()
        assert kernel in conv.kernel_name
        row = oracle.gemmlowp_fixedpoint(np.zeros((1, 16), np.int8), np.ones((16, N), np.int8), bias, 0, 0, mult, shift, offset, -128, 127, np.int8)
        np.testing.assert_array_equal(dst.cpu().numpy().reshape(-1, N), np.broadcast_to(row, (batch * oh * ow, N)))
        conv.close()
