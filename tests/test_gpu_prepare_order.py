"""A repeated prepare() on the default stream returns while its work is still running. Everything that reads or writes what it writes
comes behind it: the prepare is held up by some milliseconds of other work in front of it, and what follows on another stream
has to see the new B."""
import ctypes

import numpy as np
import pytest

import oracle
from computelibrary_amd import capi
from gpu_util import announce, to_dev, torch_dev

pytestmark = pytest.mark.gpu

M, N, K = 64, 512, 1024


class _Changing:
    """A handle that is prepared with a first B, operands on the device, the stream of the prepares and two others"""

    def __init__(self, seed, per_channel=False, side=False):
        torch = self.torch = torch_dev()
        rng = np.random.default_rng(seed)
        self.A = rng.integers(-128, 128, size=(M, K)).astype(np.int8)
        self.Bs = [rng.integers(-128, 128, size=(K, N)).astype(np.int8) for _ in range(2)]
        self.bias = rng.integers(-2000, 2000, size=N).astype(np.int32)
        self.mult, self.shift = oracle.calculate_quantized_multipliers(1.0, rng.uniform(2e-4, 6e-4, size=N if per_channel else 1), 1.0)
        self.rq = capi.requant(0 if per_channel else self.mult[0], 0 if per_channel else self.shift[0], 3, -128, 127, per_channel)
        self.g = capi.Gemm(M, N, K, capi.S8, capi.S8, capi.S8, capi.EPI_FIXEDPOINT, -3, 2, self.rq)
        self.vecs = [to_dev(np.asarray(v, np.int32)) for v in (self.mult, self.shift)] if per_channel else [None, None]
        self.Ad, self.Bd, self.bd = to_dev(self.A), [to_dev(b) for b in self.Bs], to_dev(self.bias)
        self.Dd = torch.zeros((M, N), dtype=torch.int8, device="cuda")
        self.here = torch.cuda.Stream() if side else torch.cuda.default_stream()
        self.other, self.third = (torch.cuda.Stream() for _ in range(2))
        self.prepare(0)
        self.g.run(self.Ad, self.Dd, None, self.other.cuda_stream)
        self.check(0)

    def prepare(self, which):
        self.g.prepare(self.Bd[which], self.bd, *self.vecs, stream=self.here.cuda_stream)

    def prepare_held_up(self, which):
        self.torch.cuda.synchronize()
        with self.torch.cuda.stream(self.here):
            self.torch.cuda._sleep(20_000_000)
        self.prepare(which)

    def check(self, which, a_offset=-3, b_offset=2):
        self.torch.cuda.synchronize()
        want = oracle.gemmlowp_fixedpoint(self.A, self.Bs[which], self.bias, a_offset, b_offset, self.mult, self.shift, 3, -128, 127, np.int8)
        np.testing.assert_array_equal(self.Dd.cpu().numpy(), want)


@pytest.mark.parametrize("side", [False, True])
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("runs_on", ["here", "other", "third"])
def test_new_offsets_behind_a_prepare(per_channel, runs_on, side):
    c = _Changing(21, per_channel, side)
    announce("new offsets behind a prepare", per_channel, runs_on)
    c.prepare_held_up(1)
    c.g.update_quant(9, -4, c.rq, stream=c.other.cuda_stream)
    c.g.run(c.Ad, c.Dd, None, getattr(c, runs_on).cuda_stream)
    c.check(1, 9, -4)
    c.g.run(c.Ad, c.Dd, None, c.other.cuda_stream)  # what the update left stays
    c.check(1, 9, -4)
    c.g.close()


class _Graph:
    """A graph recorded on a stream with the HIP runtime's own calls: begun without the device synchronisation that
    torch.cuda.graph starts with, and always ended, whatever is raised while it is open"""

    def __init__(self, record, stream):
        self.hip, self.exe = capi.lib(), ctypes.c_void_p()  # (the library's own dependency answers)
        graph, at = ctypes.c_void_p(), ctypes.c_void_p(stream.cuda_stream)
        assert self.hip.hipStreamBeginCapture(at, 1) == 0  # errors of this thread only
        try:
            record(stream.cuda_stream)
        finally:
            end = self.hip.hipStreamEndCapture(at, ctypes.byref(graph))
        assert end == 0 and self.hip.hipGraphInstantiate(ctypes.byref(self.exe), graph, None, None, ctypes.c_size_t(0)) == 0
        self.hip.hipGraphDestroy(graph)

    def launch(self, stream):
        assert self.hip.hipGraphLaunch(self.exe, ctypes.c_void_p(stream.cuda_stream)) == 0

    def close(self):
        self.hip.hipGraphExecDestroy(self.exe)


@pytest.mark.parametrize("side,captured_on", [(False, "other"), (True, "other"), (True, "here")])
def test_run_recorded_behind_a_prepare(side, captured_on):
    """The graph may be launched on any stream, also where it was recorded on the stream of the prepare: the prepare has to be
    over when the recorded call returns."""
    c = _Changing(22, side=side)
    announce("run recorded behind a prepare", side, captured_on)
    c.prepare_held_up(1)
    graph = _Graph(lambda s: c.g.run(c.Ad, c.Dd, None, s), getattr(c, captured_on))
    for _ in range(3):
        graph.launch(c.third)
        c.third.synchronize()
        c.check(1)
        c.Dd.zero_()
    graph.close()
    c.g.close()


def test_graph_recorded_before_a_prepare():
    """Nothing of the library is called when a graph is launched: a prepare behind a recorded run is over when it returns."""
    c = _Changing(23)
    announce("graph recorded before a prepare")
    graph = _Graph(lambda s: c.g.run(c.Ad, c.Dd, None, s), c.other)
    for which in (1, 0, 1):
        c.prepare_held_up(which)
        graph.launch(c.third)
        c.third.synchronize()
        c.check(which)
        c.Dd.zero_()
    graph.close()
    c.g.close()
