"""Rounding into half rows of every length: 8 elements per thread with rows that end anywhere in them, more columns than one
workgroup covers, destination rows and batch entries on any element, previous halfs added or not."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, run_gemm

pytestmark = pytest.mark.gpu


# one element per thread below 262144 elements, 8 from there on
SIZES = [(batch, M, N, pad) for N in (1, 7, 8, 9, 129, 257, 2049) for batch, M, pad in ((1, 1, 0), (1, 70, 1), (3, 5, 2))]
SIZES += [(1, 262144, 1, 0), (1, 37500, 7, 1), (1, 32768, 8, 0), (4, 8000, 9, 3), (1, 17500, 15, 0), (1, 16384, 16, 0), (3, 700, 129, 1),
          (2, 70, 2047, 0), (1, 128, 2048, 0), (1, 130, 2057, 5)]


@pytest.mark.parametrize("batch,M,N,pad", SIZES)
def test_half_rows(batch, M, N, pad):
    rng = np.random.default_rng(N * 1000 + M)
    K, scale = 32, 0.01
    A = rng.integers(-128, 128, size=(batch, M, K), dtype=np.int8)
    B = rng.integers(-128, 128, size=(batch, K, N), dtype=np.int8)
    prev = rng.normal(0, 3, size=(batch, M, N)).astype(np.float16)
    for was, act, flags in ((None, (-np.inf, np.inf), 0), (prev, (0.0, 6.0), capi.GEMM_ACCUMULATE)):
        announce("half rows", (batch, M, N), "pad", pad, "accumulate", flags != 0)
        got, _ = run_gemm(A, B, capi.EPI_F32, np.float16, -3, 7, scale=scale, act=act, device=True, ldd=N + pad, prev=was, flags=flags)
        for b in range(batch):
            want = oracle.gemmlowp_f16(A[b], B[b], None, -3, 7, scale, *act, prev=None if was is None else was[b])
            np.testing.assert_array_equal(got[b].view(np.uint16), want.view(np.uint16))
