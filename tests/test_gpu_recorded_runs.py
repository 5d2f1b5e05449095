"""Runs that are recorded into a graph may not allocate: what they need has to be there from the prepare, updates and runs before them,
also where those took another kernel."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, to_dev, torch_dev
from test_gpu_prepare_order import _Graph

pytestmark = pytest.mark.gpu


def test_a_convolution_whose_update_takes_it_off_the_image():
    """Few channels run straight from the image until the weights have an offset; then over patch rows, in a buffer of their own."""
    torch = torch_dev()
    rng = np.random.default_rng(51)
    src = rng.integers(0, 256, size=(2, 30, 33, 3), dtype=np.uint8)
    w = rng.integers(-128, 128, size=(24, 5, 5, 3), dtype=np.int8)
    bias = rng.integers(-3000, 3000, size=24).astype(np.int32)
    m, s = oracle.calculate_quantized_multipliers(1.0, [40.0 / (75 ** 0.5 * 74.0 * 74.0)], 1.0)
    rq = capi.requant(int(m[0]), int(s[0]), 9, 0, 255, False)
    conv = capi.Conv(capi.conv_desc(2, 30, 33, 3, 24, 5, 5, (1, 1), (2, 2, 2, 2), (1, 1), capi.U8, capi.S8, capi.U8, -131, 0, 131, rq))
    sd, wd, bd = to_dev(src), to_dev(w), to_dev(bias)
    out = torch.zeros((2, 30, 33, 24), dtype=torch.uint8, device="cuda")
    side = torch.cuda.Stream()

    def check(w_zp):
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), oracle.conv_nhwc_direct(src, w, bias, 131, w_zp, m, s, 9, 0, 255, (1, 1), (2, 2, 2, 2), (1, 1)))
        out.zero_()
        torch.cuda.synchronize()
    announce("recorded run behind an update")
    conv.prepare(wd, bd)
    conv.run(sd, out)
    assert conv.kernel_name == "implicit_rows_32x64", conv.kernel_name
    check(0)
    for w_zp in (7, 0, -3):
        conv.update_quant(-131, -w_zp, 131, rq)
        graph = _Graph(lambda stream: conv.run(sd, out, stream), side)
        assert (conv.kernel_name == "implicit_rows_32x64") == (w_zp == 0), conv.kernel_name
        for _ in range(2):
            graph.launch(side)
            check(w_zp)
        graph.close()
    conv.close()


def test_rows_of_another_alignment():
    """Sums of rows whose K ends inside a 16-byte column: inside the kernel for rows on any byte, by a pass into a vector of the handle's
    where the rows start on dwords (1500 x 40 x 2052: the copy that the first would need is what makes the difference)."""
    torch = torch_dev()
    M, N, K = 1500, 40, 2052
    rng = np.random.default_rng(52)
    A, B = rng.integers(-128, 128, size=(M, K), dtype=np.int8), rng.integers(-128, 128, size=(K, N), dtype=np.int8)
    want = oracle.gemmlowp_s32(A, B, -3, 5)
    buf = torch.zeros(M * K + 1, dtype=torch.int8, device="cuda")
    buf[1:] = to_dev(A).flatten()
    odd, even = buf[1:], to_dev(A)
    D = torch.zeros((M, N), dtype=torch.int32, device="cuda")
    g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S32, capi.EPI_S32, -3, 5)
    g.prepare(to_dev(B))
    announce("recorded run on rows of another alignment", M, N, K)
    g.run(odd, D)
    torch.cuda.synchronize()
    first = g.kernel_name
    np.testing.assert_array_equal(D.cpu().numpy(), want)
    side = torch.cuda.Stream()
    graph = _Graph(lambda stream: g.run(even, D, None, stream), side)
    assert first.endswith("_bytes") and not g.kernel_name.endswith("_bytes"), (first, g.kernel_name)
    for _ in range(2):
        D.zero_()
        torch.cuda.synchronize()
        graph.launch(side)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(D.cpu().numpy(), want)
    graph.close()
    g.close()
