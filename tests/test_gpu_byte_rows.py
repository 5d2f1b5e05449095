"""Rows of A that start on any byte, and row sums that stop inside a 16-byte column, without a pass in front: base addresses and row
strides of every remainder modulo 4, K of 1 to 7 steps ending on every kind of place, batches whose entries start on any byte, K
slices, few rows, both signs, every destination. A lies at the very end of its allocation, and what surrounds its rows is not zero."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import CODE, announce, run_gemm, torch_dev

pytestmark = pytest.mark.gpu


def run_at(A, B, off, lda, a_bs, ao, bo, dst, **how):
    """A [batch][M][K] at byte `off` of a buffer that ends with A's last byte -> (result, kernel name)"""
    torch = torch_dev()
    batch, M, K = A.shape
    N = B.shape[1]
    size = off + (batch - 1) * a_bs + (M - 1) * lda + K
    flat = np.random.default_rng(off + lda).integers(0, 256, size=size, dtype=np.uint8)
    for z in range(batch):
        for i in range(M):
            at = off + z * a_bs + i * lda
            flat[at:at + K] = A[z, i].view(np.uint8)
    buf = torch.from_numpy(flat).cuda()
    g = capi.Gemm(M, N, K, CODE[A.dtype], CODE[B.dtype], dst, how.pop("epilogue"), ao, bo, batch=batch, lda=lda, a_batch_stride=a_bs, **how)
    g.prepare(torch.from_numpy(B).cuda())
    D = torch.full((batch, M, N), 77, dtype=torch.int32 if dst == capi.S32 else torch.float32, device="cuda")
    g.run(buf[off:], D)
    torch.cuda.synchronize()
    name = g.kernel_name
    g.close()
    return D.cpu().numpy(), name


@pytest.mark.parametrize("M,N,K", [(1, 5, 16), (3, 111, 233), (64, 65, 127), (65, 64, 128), (70, 130, 129), (129, 63, 386), (66, 70, 515), (100, 40, 643), (63, 17, 900)])
@pytest.mark.parametrize("dt", [np.uint8, np.int8])
def test_every_alignment(M, N, K, dt):
    rng = np.random.default_rng(M + N + K)
    info = np.iinfo(dt)
    for batch, off, pad in ((1, 0, 1), (1, 3, 0), (1, 2, 3), (2, 1, 2), (3, 2, 5)):
        lda = K + pad
        a_bs = M * lda + 1
        A = rng.integers(info.min, info.max + 1, size=(batch, M, K)).astype(dt)
        B = rng.integers(info.min, info.max + 1, size=(K, N)).astype(dt)
        announce("byte rows", (batch, M, N, K), "off", off, "lda", lda, dt.__name__)
        got, name = run_at(A, B, off, lda, a_bs, -5, 9, capi.S32, epilogue=capi.EPI_S32)
        for z in range(batch):
            np.testing.assert_array_equal(got[z], oracle.gemmlowp_s32(A[z], B, -5, 9))
        if dt == np.uint8:
            continue
        got, name = run_at(A, B, off, lda, a_bs, 0, 0, capi.F32, epilogue=capi.EPI_F32, scale=3e-4)
        for z in range(batch):
            np.testing.assert_array_equal(got[z].view(np.uint32), np.asarray(oracle.gemmlowp_f32(A[z], B, None, 0, 0, 3e-4)).view(np.uint32))
        if M > 64 and (lda | a_bs * (batch > 1)) % 4 != 0:
            assert name.endswith("_bytes"), name


@pytest.mark.parametrize("M,N,K", [(70, 130, 132), (200, 96, 500), (100, 64, 20), (90, 33, 1004), (5, 40, 36)])
def test_sums_that_stop_inside_a_column(M, N, K):
    """Dword-aligned rows and a B offset with K no multiple of 16"""
    rng = np.random.default_rng(M * K + N)
    A = rng.integers(0, 256, size=(M, K), dtype=np.uint8)
    B = rng.integers(0, 256, size=(K, N), dtype=np.uint8)
    bias = rng.integers(-20000, 20000, size=N, dtype=np.int32)
    mult, shift = oracle.calculate_quantized_multiplier(float(40.0 / (K ** 0.5 * 74.0 * 74.0)))
    announce("byte rows, sums", (M, N, K))
    got, name = run_gemm(A, B, capi.EPI_FIXEDPOINT, np.uint8, -120, -131, bias, [mult], [shift], 7, 0, 255, device=True)
    assert name.endswith("_bytes"), name
    np.testing.assert_array_equal(got, oracle.gemmlowp_fixedpoint(A, B, bias, -120, -131, [mult], [shift], 7, 0, 255, np.uint8))


def test_slices():
    rng = np.random.default_rng(9)
    for M, N, K in ((70, 60, 5001), (130, 40, 7167)):
        for dt in (np.uint8, np.int8):
            info = np.iinfo(dt)
            A = rng.integers(info.min, info.max + 1, size=(1, M, K)).astype(dt)
            B = rng.integers(info.min, info.max + 1, size=(K, N)).astype(dt)
            announce("byte rows, slices", (M, N, K), dt.__name__)
            got, name = run_at(A, B, 1, K, M * K, -5, 9, capi.S32, epilogue=capi.EPI_S32)
            assert "_splitk" in name, name
            np.testing.assert_array_equal(got[0], oracle.gemmlowp_s32(A[0], B, -5, 9))
