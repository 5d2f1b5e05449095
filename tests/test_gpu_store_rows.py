"""Destinations whose rows are aligned to 16, 4 or 1 elements, with tiles inside and on the edges of the matrix: 8-bit, 32-bit and
half results of the pipelined kernel's tiles, of its K slices and of the streaming kernel's forms. Halves are the float results
rounded to nearest even."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, run_gemm

pytestmark = pytest.mark.gpu

PATHS = [capi.PATH_TILE + 0, capi.PATH_TILE + 1, capi.PATH_TILE + 3, capi.PATH_TILE + 5, capi.PATH_TILE + 6]


@pytest.mark.parametrize("path", PATHS)
@pytest.mark.parametrize("M,N,K", [(130, 64, 128), (257, 129, 260), (64, 131, 400), (300, 258, 132)])
def test_pipelined(path, M, N, K):
    rng = np.random.default_rng(M + N + K + path)
    A, B = (rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((M, K), (K, N)))
    bias = rng.integers(-20000, 20000, size=N, dtype=np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(0.5, 2.0, size=N) * 40.0 / (K ** 0.5 * 74.0 * 74.0), 1.0)
    want8 = oracle.gemmlowp_fixedpoint(A, B, bias, 3, 0, mult, shift, 7, -128, 127, np.int8)
    want32, wantf = oracle.gemmlowp_s32(A, B, -5, 9), np.asarray(oracle.gemmlowp_f32(A, B, None, 0, 0, 3e-4))
    for ldd in (N, (N + 3) // 4 * 4, (N + 15) // 16 * 16, N + 1):
        announce("store rows", path, (M, N, K), "ldd", ldd)
        how = dict(path=path, device=True, ldd=ldd)
        got, _ = run_gemm(A, B, capi.EPI_FIXEDPOINT, np.int8, 3, 0, bias, mult, shift, 7, -128, 127, **how)
        np.testing.assert_array_equal(got, want8)
        got, _ = run_gemm(A, B, capi.EPI_S32, np.int32, -5, 9, **how)
        np.testing.assert_array_equal(got, want32)
        got, _ = run_gemm(A, B, capi.EPI_F32, np.float32, scale=3e-4, **how)
        np.testing.assert_array_equal(got.view(np.uint32), wantf.view(np.uint32))
        got, _ = run_gemm(A, B, capi.EPI_F32, np.float16, scale=3e-4, **how)
        np.testing.assert_array_equal(got.view(np.uint16), wantf.astype(np.float16).view(np.uint16))


# tiles on the right edge with 1 to 3, 4 to 15 and 16 or more columns left, whose last pieces move back to the end of the row; rows that start on
# any element, as the caller's own row stride or as the previous row ends
@pytest.mark.parametrize("N", [2, 5, 17, 30, 63, 70, 77, 93, 141, 255])
@pytest.mark.parametrize("path,M", [(capi.PATH_TILE + 0, 257), (capi.PATH_TILE + 3, 70), (capi.PATH_TILE + 6, 129)])
def test_right_edge(path, M, N):
    K = 132
    rng = np.random.default_rng(M + N)
    A, B = (rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((2, M, K), (K, N)))
    bias = rng.integers(-20000, 20000, size=N, dtype=np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(0.5, 2.0, size=N) * 40.0 / (K ** 0.5 * 74.0 * 74.0), 1.0)
    for ldd in (N, N + 1, (N + 15) // 16 * 16):
        announce("right edge", path, (M, N, K), "ldd", ldd)
        how = dict(path=path, device=True, ldd=ldd)
        got8, _ = run_gemm(A, B, capi.EPI_FIXEDPOINT, np.int8, 3, 0, bias, mult, shift, 7, -128, 127, **how)
        got32, _ = run_gemm(A, B, capi.EPI_S32, np.int32, -5, 9, **how)
        gotf, _ = run_gemm(A, B, capi.EPI_F32, np.float32, scale=3e-4, **how)
        goth, _ = run_gemm(A, B, capi.EPI_F32, np.float16, scale=3e-4, **how)
        for z in range(2):
            np.testing.assert_array_equal(got8[z], oracle.gemmlowp_fixedpoint(A[z], B, bias, 3, 0, mult, shift, 7, -128, 127, np.int8))
            np.testing.assert_array_equal(got32[z], oracle.gemmlowp_s32(A[z], B, -5, 9))
            wantf = np.asarray(oracle.gemmlowp_f32(A[z], B, None, 0, 0, 3e-4))
            np.testing.assert_array_equal(gotf[z].view(np.uint32), wantf.view(np.uint32))
            np.testing.assert_array_equal(goth[z].view(np.uint16), wantf.astype(np.float16).view(np.uint16))


# streaming forms (staged, per step, stage-once of 8, 16, 32 and 64 rows, deep K, a batch on the grid), slices, rows on any byte
@pytest.mark.parametrize("batch,M,N,K", [(1, 5, 70, 200), (1, 8, 4099, 256), (1, 16, 300, 1024), (1, 30, 129, 640), (1, 60, 65, 512),
                                         (1, 8, 33, 9000), (1, 8, 48, 8320), (3, 7, 29, 64), (1, 100, 64, 4096), (1, 70, 61, 513)])
def test_half(batch, M, N, K):
    rng = np.random.default_rng(batch + M + N + K)
    A, B = (rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((batch, M, K), (batch, K, N)))
    bias = rng.normal(size=N).astype(np.float32)
    for ldd in (N, N + 1):
        announce("store rows, half", (batch, M, N, K), "ldd", ldd)
        got, _ = run_gemm(A, B, capi.EPI_F32, np.float16, scale=3e-4, bias_f32=bias, act=(-6.0, 6.0), device=True, ldd=ldd)
        for z in range(batch):
            want = np.asarray(oracle.gemmlowp_f32(A[z], B[z], bias, 0, 0, 3e-4, -6.0, 6.0)).astype(np.float16)
            np.testing.assert_array_equal(got[z].view(np.uint16), want.view(np.uint16))
