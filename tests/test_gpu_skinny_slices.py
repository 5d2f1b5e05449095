"""The stage-once kernels with a K that ends inside a 64-byte block (whole 16-byte pieces), and with K in slices whose last
workgroup finishes: each run repeated, since a run leaves the counters as it found them."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, run_gemm, to_dev, torch_dev

pytestmark = pytest.mark.gpu


def _operands(M, N, K, a_dt):
    rng = np.random.default_rng(M + N + K)
    info = np.iinfo(a_dt)
    A = rng.integers(info.min, info.max + 1, size=(M, K)).astype(a_dt)
    B = rng.integers(-128, 128, size=(K, N), dtype=np.int8)
    bias = rng.integers(-3000, 3000, size=N, dtype=np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(0.5, 2.0, size=N) * 40.0 / (K ** 0.5 * 74.0 * 74.0), 1.0)
    return A, B, bias, mult, shift


def _all_outputs(A, B, bias, mult, shift, form):
    a_dt = A.dtype.type
    lo, hi, off = (-128, 127, -7) if a_dt == np.int8 else (0, 255, 121)
    N, K = B.shape[1], B.shape[0]
    got, name = run_gemm(A, B, capi.EPI_S32, np.int32, -5, 9, device=True, path=capi.PATH_SKINNY, ldd=N + 3)
    assert name.startswith(form), name
    np.testing.assert_array_equal(got, oracle.gemmlowp_s32(A, B, -5, 9))
    got, _ = run_gemm(A, B, capi.EPI_FIXEDPOINT, a_dt, -5, 0, bias, mult, shift, off, lo, hi, device=True, path=capi.PATH_SKINNY)
    np.testing.assert_array_equal(got, oracle.gemmlowp_fixedpoint(A, B, bias, -5, 0, mult, shift, off, lo, hi, a_dt))
    if a_dt == np.int8:
        got, _ = run_gemm(A, B, capi.EPI_F32, np.float32, -5, 9, scale=1e-4, device=True, path=capi.PATH_SKINNY, lda=K + 16)
        np.testing.assert_array_equal(got.view(np.uint32), np.asarray(oracle.gemmlowp_f32(A, B, None, -5, 9, 1e-4)).view(np.uint32))


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(40, 16), (300, 1040), (1000, 2064), (4100, 4080), (60, 3264)])
def test_k_of_whole_pieces(M, N, K):
    announce("whole pieces", (M, N, K))
    _all_outputs(*_operands(M, N, K, np.uint8 if K % 32 else np.int8), form="skinny_once")


@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("N,K", [(40, 8208), (700, 11056), (40, 16368)])
def test_deep_k_of_whole_pieces(M, N, K):
    announce("whole pieces, deep", (M, N, K))
    _all_outputs(*_operands(M, N, K, np.int8), form="skinny_deepk")


# 9 to 16 rows: from 8193 on; 17 to 32 rows: from 4097 on. One and several column groups per workgroup, a ragged last group, slices
# of unequal length, and (8200 columns) more than one round of workgroups
@pytest.mark.parametrize("M,N,K", [(9, 40, 8208), (16, 2000, 12128), (16, 4100, 8256), (17, 40, 4112), (32, 1472, 5424), (25, 3264, 11072),
                                   (32, 8200, 4176), (20, 300, 16400)])
@pytest.mark.parametrize("a_dt", [np.int8, np.uint8])
def test_k_slices(M, N, K, a_dt):
    announce("skinny slices", (M, N, K), a_dt.__name__)
    operands = _operands(M, N, K, a_dt)
    _all_outputs(*operands, form="skinny_slices")
    torch = torch_dev()
    A, B = operands[:2]
    want = oracle.gemmlowp_s32(A, B, 3, 0)
    code = capi.U8 if a_dt == np.uint8 else capi.S8
    g = capi.Gemm(M, N, K, code, capi.S8, capi.S32, capi.EPI_S32, 3, 0, path=capi.PATH_SKINNY)
    Ad, Bd, D = to_dev(A), to_dev(B), torch.zeros((M, N), dtype=torch.int32, device="cuda")
    for _ in range(2):
        g.prepare(Bd)
        for _ in range(3):
            D.zero_()
            g.run(Ad, D)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(D.cpu().numpy(), want)
    g.close()
