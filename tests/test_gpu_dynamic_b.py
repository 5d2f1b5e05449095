"""B that changes between runs: prepare() on a handle that is already prepared packs all batch entries in one launch and, on the
default stream, only enqueues. Sizes around the packing kernel's tile (64 columns x 128 of K) and its K runs, both operand orders, both packed
layouts; and a run on another stream, plain and under graph capture, behind a prepare that has not been waited for."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, to_dev, torch_dev
from test_gpu_prepare_order import _Graph

pytestmark = pytest.mark.gpu


# (batch, M, N, K, transposed, interleave): M <= 32 takes the streaming kernel's layout
SHAPES = [(1, 1, 1, 1, False, 0), (3, 40, 63, 127, False, 0), (2, 40, 65, 129, False, 0), (5, 9, 71, 128, False, 0),
          (1, 40, 9, 4100, False, 0), (2, 7, 300, 2051, False, 0), (1, 40, 130, 260, False, 4), (3, 40, 63, 130, True, 0),
          (2, 9, 257, 191, True, 0), (1, 40, 66, 132, True, 3)]


@pytest.mark.parametrize("batch,M,N,K,transposed,kf", SHAPES)
@pytest.mark.parametrize("dt", [np.uint8, np.int8])
def test_new_b_for_every_run(batch, M, N, K, transposed, kf, dt):
    rng = np.random.default_rng(M * 1000 + N + K)
    lo, hi = np.iinfo(dt).min, np.iinfo(dt).max + 1
    code = capi.U8 if dt == np.uint8 else capi.S8
    ao, bo = -131, 7
    pad = 5  # ldb > N: rows of B start on any byte
    g = capi.Gemm(M, N, K, code, code, capi.S32, capi.EPI_S32, ao, bo, batch=batch, b_batched=batch > 1,
                  ldb=(K if transposed else N) + pad, b_transposed=transposed, b_k_interleave=kf)
    for step in range(3):
        announce("dynamic b", (batch, M, N, K), transposed, kf, dt.__name__, "step", step)
        A = rng.integers(lo, hi, size=(batch, M, K)).astype(dt)
        B = rng.integers(lo, hi, size=(batch, K, N)).astype(dt)
        Bm = B if not kf else np.stack([b.reshape(K // kf, kf, N).transpose(1, 0, 2).reshape(K, N) for b in B])
        Bm = Bm.transpose(0, 2, 1) if transposed else Bm
        Bh = np.full(Bm.shape[:2] + (Bm.shape[2] + pad,), 99, dtype=dt)
        Bh[:, :, :Bm.shape[2]] = Bm
        Ad, Bd = to_dev(A), to_dev(Bh)
        Dd = to_dev(np.full((batch, M, N), 77, np.int32))
        g.prepare(Bd)
        g.run(Ad, Dd)
        got = Dd.cpu().numpy()
        for z in range(batch):
            np.testing.assert_array_equal(got[z], oracle.gemmlowp_s32(A[z], B[z], ao, bo))
    g.close()


@pytest.mark.parametrize("per_channel", [False, True])
def test_new_b_and_bias_with_requantisation_then_new_offsets(per_channel):
    rng = np.random.default_rng(11)
    M, N, K = 70, 130, 200
    mult, shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(1e-4, 1e-3, size=N if per_channel else 1), 1.0)
    rq = capi.requant(0 if per_channel else mult[0], 0 if per_channel else shift[0], 3, -128, 127, per_channel)
    g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S8, capi.EPI_FIXEDPOINT, -3, 2, rq)
    vecs = [to_dev(np.asarray(v, np.int32)) for v in (mult, shift)] if per_channel else [None, None]
    for step in range(3):
        A = rng.integers(-128, 128, size=(M, K)).astype(np.int8)
        B = rng.integers(-128, 128, size=(K, N)).astype(np.int8)
        bias = rng.integers(-2000, 2000, size=N).astype(np.int32)
        Ad, Bd, bd, Dd = to_dev(A), to_dev(B), to_dev(bias), to_dev(np.zeros((M, N), np.int8))
        g.prepare(Bd, bd, *vecs)
        for ao, bo in [(-3, 2), (9, -4)] if step == 2 else [(-3, 2)]:
            if (ao, bo) != (-3, 2):  # the sums and the bias of the last prepare still count
                bd.zero_()
                g.update_quant(ao, bo, rq)
            g.run(Ad, Dd)
            np.testing.assert_array_equal(Dd.cpu().numpy(), oracle.gemmlowp_fixedpoint(A, B, bias, ao, bo, mult, shift, 3, -128, 127, np.int8))
    g.close()


@pytest.mark.parametrize("captured", [False, True])
def test_run_on_another_stream_waits_for_the_prepare(captured):
    torch = torch_dev()
    rng = np.random.default_rng(5)
    M, N, K = 64, 2048, 4096
    A = rng.integers(-128, 128, size=(M, K)).astype(np.int8)
    Bs = [rng.integers(-128, 128, size=(K, N)).astype(np.int8) for _ in range(2)]
    g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S32, capi.EPI_S32)
    Ad, Bd = to_dev(A), [to_dev(b) for b in Bs]
    Dd = torch.zeros((M, N), dtype=torch.int32, device="cuda")
    here, other, third = torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    g.prepare(Bd[0], stream=here.cuda_stream)
    g.run(Ad, Dd, None, other.cuda_stream)
    torch.cuda.synchronize()
    want = A.astype(np.float64) @ Bs[0].astype(np.float64)
    np.testing.assert_array_equal(Dd.cpu().numpy(), want.astype(np.int32))
    announce("another stream, captured", captured)
    with torch.cuda.stream(here):
        torch.cuda._sleep(20_000_000)  # what is in front of the prepare takes some milliseconds
    g.prepare(Bd[1], stream=here.cuda_stream)
    if captured:
        # (not torch.cuda.graph, which synchronises the device first: the prepare would be over)
        graph = _Graph(lambda s: g.run(Ad, Dd, None, s), other)
        graph.launch(third)
    else:
        g.run(Ad, Dd, None, other.cuda_stream)
    torch.cuda.synchronize()
    want = A.astype(np.float64) @ Bs[1].astype(np.float64)
    np.testing.assert_array_equal(Dd.cpu().numpy(), want.astype(np.int32))
    if captured:
        graph.close()
    g.close()


def test_more_batch_entries_than_one_packing_launch_takes():
    """32768 entries are packed at a time. What is left over is one entry, which alone would be packed in several runs of K: the
    workspace of the column sums belongs to the count of the large parts."""
    batch, M, N, K = 32769, 2, 16, 200
    rng = np.random.default_rng(12)
    A = rng.integers(-128, 128, size=(batch, M, K)).astype(np.int8)
    B = rng.integers(-128, 128, size=(batch, K, N)).astype(np.int8)
    announce("many batch entries", batch)
    g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S32, capi.EPI_S32, 3, 0, batch=batch, b_batched=True)
    Ad, Bd = to_dev(A), to_dev(B)
    for _ in range(2):
        Dd = to_dev(np.full((batch, M, N), 77, np.int32))
        g.prepare(Bd)
        g.run(Ad, Dd)
        np.testing.assert_array_equal(Dd.cpu().numpy(), np.matmul(A.astype(np.float32) + 3, B.astype(np.float32)).astype(np.int32))
    g.close()
