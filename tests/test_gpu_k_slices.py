"""K slices that do not divide K: the last slice holds what is left of K, which may end inside a K step. Dense products (rows
dword aligned and not, both signs of A with the row sums taken per slice, every destination) and the convolution."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, run_gemm, to_dev, torch_dev
from test_gpu_conv import run_conv
from test_gpu_prepare_order import _Graph

pytestmark = pytest.mark.gpu

# (M, N, K): 2 to 30 slices; K of one value past a slice, one short of it, odd, a multiple of 4 only
SHAPES = [(70, 40, 2049), (100, 96, 4096 + 16), (65, 33, 10588), (190, 130, 3000), (130, 64, 7167), (254, 200, 5104)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dt", [np.uint8, np.int8])
def test_dense(M, N, K, dt):
    rng = np.random.default_rng(M + N + K)
    lo, hi = np.iinfo(dt).min, np.iinfo(dt).max
    A = rng.integers(lo, hi + 1, size=(M, K)).astype(dt)
    B = rng.integers(lo, hi + 1, size=(K, N)).astype(dt)
    ao, bo = -5, 9
    exact = (A.astype(np.float64) + ao) @ (B.astype(np.float64) + bo)
    announce("k slices", (M, N, K), dt.__name__)
    got, name = run_gemm(A, B, capi.EPI_S32, np.int32, ao, bo, device=True)
    assert "_splitk" in name, name
    np.testing.assert_array_equal(got, exact.astype(np.int64).astype(np.int32))
    bias = rng.integers(-20000, 20000, size=N, dtype=np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(0.5, 2.0, size=N) * 40.0 / (K ** 0.5 * 74.0 * 74.0), 1.0)
    got, name = run_gemm(A, B, capi.EPI_FIXEDPOINT, dt, -128 if lo == 0 else 3, -120 if lo == 0 else 0, bias, mult, shift, 7, lo, hi, device=True)
    assert "_splitk" in name, name
    np.testing.assert_array_equal(got, oracle.gemmlowp_fixedpoint(A, B, bias, -128 if lo == 0 else 3, -120 if lo == 0 else 0, mult, shift, 7, lo, hi, dt))
    if dt == np.int8:
        got, name = run_gemm(A, B, capi.EPI_F32, np.float32, ao, bo, scale=1e-4, device=True)
        np.testing.assert_array_equal(got.view(np.uint32), np.asarray(oracle.gemmlowp_f32(A, B, None, ao, bo, 1e-4)).view(np.uint32))


@pytest.mark.parametrize("shape,OFM,k", [((2, 9, 10, 304), 24, 5), ((1, 14, 14, 336), 130, 3), ((3, 7, 7, 432), 56, 5),
                                         ((2, 9, 10, 300), 24, 5), ((1, 14, 14, 330), 130, 3)])  # channels padded to 304 and 336
@pytest.mark.parametrize("dt,w_dt", [(np.int8, np.int8), (np.uint8, np.uint8)])
def test_convolution(shape, OFM, k, dt, w_dt):
    rng = np.random.default_rng(sum(shape) + OFM)
    info, w_info = np.iinfo(dt), np.iinfo(w_dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(w_info.min, w_info.max + 1, size=(OFM, k, k, shape[3])).astype(w_dt)
    zp, w_zp = (3, 0) if dt == np.int8 else (120, 131)
    bias = rng.integers(-3000, 3000, size=OFM).astype(np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, [40.0 / ((k * k * shape[3]) ** 0.5 * 74.0 * 74.0)], 1.0)
    p = k // 2
    announce("k slices, convolution", shape, OFM, k, dt.__name__)
    got, name = run_conv(src, w, bias, zp, w_zp, mult, shift, 5, info.min, info.max, (1, 1), (p, p, p, p))
    assert "_splitk" in name, name
    np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, zp, w_zp, mult, shift, 5, info.min, info.max, (1, 1), (p, p, p, p)))


def test_float_slices_with_an_offset_need_no_workspace_in_the_run():
    """Their row terms come from a pass over A (the planes must not mix them into the product), into a vector that prepare has
    made: a first run is recorded, and run_noalloc is not refused while the workspace is in use on another stream."""
    torch = torch_dev()
    M, N, K = 190, 130, 3008
    rng = np.random.default_rng(40)
    A, B = (rng.integers(-128, 128, size=s).astype(np.int8) for s in ((M, K), (K, N)))
    want = np.asarray(oracle.gemmlowp_f32(A, B, None, -5, 9, 1e-4)).view(np.uint32)
    busy = capi.Gemm(1024, 1024, 4000, capi.S8, capi.S8, capi.S32, capi.EPI_S32, 3, 4, lda=4003)  # (a padded copy of A)
    A_busy, B_busy = (torch.zeros(s, dtype=torch.int8, device="cuda") for s in ((1024, 4003), (4000, 1024)))
    D_busy = torch.zeros((1024, 1024), dtype=torch.int32, device="cuda")
    busy.prepare(B_busy)
    g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.F32, capi.EPI_F32, -5, 9, scale=1e-4)
    Ad, Bd = to_dev(A), to_dev(B)
    Dd = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    g.prepare(Bd)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    announce("float slices, workspace")
    graph = _Graph(lambda s: g.run(Ad, Dd, None, s), s2)
    assert "_splitk" in g.kernel_name, g.kernel_name
    for _ in range(2):
        graph.launch(s2)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(Dd.cpu().numpy().view(np.uint32), want)
        Dd.zero_()
        torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        torch.cuda._sleep(50_000_000)
    busy.run_noalloc(A_busy, D_busy, stream=s1.cuda_stream)
    g.run_noalloc(Ad, Dd, stream=s2.cuda_stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(Dd.cpu().numpy().view(np.uint32), want)
    graph.close()
    g.close()
    busy.close()
