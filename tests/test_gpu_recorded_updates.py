"""update_quant() and prepare() under graph capture: what they write goes into the graph and has not happened yet, and launching
the graph repeats it. Calls outside the graph may take nothing that it writes for known. Both per-tensor forms: the vectors of
the streaming kernel (M = 64) and the digested ones of the pipelined kernel (M = 130)."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, to_dev, torch_dev
from test_gpu_prepare_order import _Graph

pytestmark = pytest.mark.gpu

N, K = 96, 512
SCALES = (2e-4, 7e-4)


class _Case:
    def __init__(self, M, seed):
        rng = np.random.default_rng(seed)
        self.M, self.torch = M, torch_dev()
        self.A = rng.integers(-128, 128, size=(M, K)).astype(np.int8)
        self.B = rng.integers(-128, 128, size=(K, N)).astype(np.int8)
        self.bias = rng.integers(-2000, 2000, size=N).astype(np.int32)
        self.q = [oracle.calculate_quantized_multipliers(1.0, [s], 1.0) for s in SCALES]
        self.offsets, self.lo = (3, -20), (-128, -40)
        self.rq = [capi.requant(q[0][0], q[1][0], o, lo, 127, False) for q, o, lo in zip(self.q, self.offsets, self.lo)]
        self.g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S8, capi.EPI_FIXEDPOINT, -3, 2, self.rq[0])
        self.Ad, self.Bd, self.bd = to_dev(self.A), to_dev(self.B), to_dev(self.bias)
        self.Dd = self.torch.zeros((M, N), dtype=self.torch.int8, device="cuda")
        self.side = self.torch.cuda.Stream()

    def update(self, which, stream=0):
        self.g.update_quant(-3, 2, self.rq[which], stream=stream)

    def run(self, stream=0):
        self.g.run(self.Ad, self.Dd, None, stream)

    def check(self, which):
        self.torch.cuda.synchronize()
        q = self.q[which]
        want = oracle.gemmlowp_fixedpoint(self.A, self.B, self.bias, -3, 2, *q, self.offsets[which], self.lo[which], 127, np.int8)
        np.testing.assert_array_equal(self.Dd.cpu().numpy(), want)
        self.Dd.zero_()
        self.torch.cuda.synchronize()


@pytest.mark.parametrize("M", [64, 130])
def test_an_update_that_was_only_recorded(M):
    c = _Case(M, 31)
    announce("recorded update", M)
    c.g.prepare(c.Bd, c.bd)
    graph = _Graph(lambda s: c.update(1, s), c.side)
    c.update(1)
    c.run()
    c.check(1)
    graph.close()
    c.g.close()


@pytest.mark.parametrize("M", [64, 130])
def test_a_graph_writes_what_its_run_needs(M):
    """Recorded while the handle held the very same values; the eager calls between the launches use others."""
    c = _Case(M, 32)
    announce("graph with its own update", M)
    c.g.prepare(c.Bd, c.bd)
    c.run()  # (the workspace of the row sums is there)
    c.check(0)

    def record(s):
        c.update(0, s)
        c.run(s)

    graph = _Graph(record, c.side)
    for _ in range(3):
        c.update(1)
        c.run()
        c.check(1)
        graph.launch(c.side)
        c.side.synchronize()
        c.check(0)
        c.update(1)  # again: the graph has written its own values since
        c.run()
        c.check(1)
    graph.close()
    c.g.close()


def _first_prepare_recorded(M):
    """It cannot wait for its work there and fails; nothing of it has happened, and the handle is as unprepared as before."""
    c = _Case(M, 33)
    announce("recorded prepare", M)
    hip, graph, at = capi.lib(), ctypes.c_void_p(), ctypes.c_void_p(c.side.cuda_stream)
    assert hip.hipStreamBeginCapture(at, 2) == 0  # relaxed: memory may be allocated
    try:
        with pytest.raises(RuntimeError):
            c.g.prepare(c.Bd, c.bd, stream=c.side.cuda_stream)
    finally:
        assert hip.hipStreamEndCapture(at, ctypes.byref(graph)) != 0
        hip.hipGetLastError()
    with pytest.raises(RuntimeError):
        c.run()
    c.g.prepare(c.Bd, c.bd)
    c.run()
    c.check(0)
    c.g.close()


def test_a_first_prepare_that_was_only_recorded():
    """In a process of its own: the stream with the broken capture stays unusable, and torch hands its streams out again."""
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(here), here, os.environ.get("PYTHONPATH", "")]))
    code = "import test_gpu_recorded_updates as t; t._first_prepare_recorded(64); t._first_prepare_recorded(130)"
    r = subprocess.run([sys.executable, "-c", code], env=env, timeout=100, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
