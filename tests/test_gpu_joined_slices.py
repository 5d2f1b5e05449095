"""K slices that the last workgroup of a tile joins, each with a place of its own (up to 5) and added up in one (more): a run leaves
counters and sums as it found them, so runs repeat, also on other operands, and behind another prepare."""
import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, to_dev, torch_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,few", [(130, 70, 3008, False), (592, 182, 3856, True), (65, 33, 10592, False), (256, 256, 8192, False), (64, 64, 16384, False)])
@pytest.mark.parametrize("b_off", [0, 9])
def test_runs_repeat(M, N, K, few, b_off):
    torch = torch_dev()
    rng = np.random.default_rng(M + N + K)
    As = [rng.integers(-128, 128, size=(M, K), dtype=np.int8) for _ in range(2)]
    B = rng.integers(-128, 128, size=(K, N), dtype=np.int8)
    wants = [oracle.gemmlowp_s32(A, B, -3, b_off) for A in As]
    g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S32, capi.EPI_S32, -3, b_off, path=capi.PATH_MFMA)
    Ad, Bd, D = [to_dev(A) for A in As], to_dev(B), torch.zeros((M, N), dtype=torch.int32, device="cuda")
    announce("joined slices", (M, N, K), b_off)
    for _ in range(2):
        g.prepare(Bd)
        for i in (0, 1, 0):
            D.zero_()
            g.run(Ad[i], D)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(D.cpu().numpy(), wants[i])
    slices = int(g.kernel_name.split("_splitk")[1])
    assert slices > 1 and (slices <= 5) == few, g.kernel_name
    g.close()
