"""Convolutions whose input window lies in LDS: every division that the plan gives covers the output, keeps inside the LDS and the
tables that the kernel indexes (checked on the host over the rule's range), and the kernel against the oracle: both layouts, channels in
pieces of 16 and 8 bytes and planes with any number of them, tiles that end inside an image and inside a row, waves that share K and
that share the pixels, several panels, weights with an offset, the general requantisation, updates, graphs and unaligned tensors."""
import os
import subprocess

import numpy as np
import pytest

import oracle
from computelibrary_amd import capi

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "computelibrary_amd", "csrc")

SWEEP = r"""
#include "conv_window_plan.hpp"
#include <cstdio>
using namespace mi355;
struct G { int H, W, C, KH, KW, OH, OW, stride_x, stride_y, pad_left, pad_top, dil_x, dil_y; };
int main()
{
    long taken = 0, split = 0;
    const int size[] = {1, 3, 4, 7, 8, 14, 15, 28, 33, 56, 112, 115, 224, 260, 300, 513, 1100};
    for (int W : size) for (int H : {1, 5, 14, 30, 112, 225}) for (int C = 5; C < 2100; C = C < 72 ? C + 3 : C * 4 / 3 + 1) for (int KH : {1, 2, 3, 5, 9}) for (int KW : {1, 3, 5, 8})
    for (int sx : {1, 2, 3, 4}) for (int sy : {1, 2}) for (int dx : {1, 2}) for (int pad : {0, 1})
    {
        G g{H, W, C, KH, KW, 0, 0, sx, sy, pad * (KW / 2), pad * (KH / 2), dx, 1};
        const int h = H + 2 * g.pad_top - KH, w = W + 2 * g.pad_left - ((KW - 1) * dx + 1);
        if (h < 0 || w < 0) continue;
        g.OH = h / sy + 1, g.OW = w / sx + 1;
        for (int batch : {1, 37}) for (int N : {1, 64, 70, 500}) for (int planes = 0; planes < 2; ++planes) for (int sums = 0; sums < 2; ++sums)
        {
            WindowPlan p;
            if (!conv_window_plan(g, batch, N, planes, sums, 256, p)) continue;
            ++taken, split += p.tx > 1;
            const int     most = conv_window_pixels(p.rs, p.wk), cpr = (C + 15) / 16, per_x = planes ? (p.wc + 3) / 4 : cpr * (C % 16 ? 2 : 1);
            const int64_t K = conv_window_k(g), nkb = (K + 63) / 64, row = planes ? (int64_t)per_x * cpr : (int64_t)per_x * p.wc;
            int64_t       last = 0; // the furthest entry of the table that a wave reads
            for (int wk = 0; wk < p.wk; ++wk) { const int64_t ns = (nkb - wk + p.wk - 1) / p.wk; last = std::max(last, std::max<int64_t>(ns, 1) * p.wk * 4 + wk * 4 + 3); }
            const int64_t box = p.wk == 1 ? 0 : (int64_t)WINDOW_WAVES * p.rs * 1024 * (p.wk == 4 ? 3 : 2) / 2;
            const int64_t out = planes ? (int64_t)WINDOW_PANEL * (most + 16) : (int64_t)most * WINDOW_OPITCH;
            const bool ok = C >= 8 && (planes ? W >= 4 : C % 8 == 0) && p.th * p.tw <= most && (p.tx == 1 || p.th == 1) && p.tx * p.tw >= g.OW && (p.tx - 1) * p.tw < g.OW &&
                            p.ty * p.th >= g.OH && (p.ty - 1) * p.th < g.OH && p.u >= cpr && p.lds <= WINDOW_MOST_LDS && (int64_t)p.wr * p.wc * p.u * 16 <= p.win_bytes &&
                            p.tab_bytes >= (last + 1) * 4 && p.xch_bytes >= box && p.xch_bytes >= out && p.panels * WINDOW_PANEL >= N && p.ppw <= p.panels &&
                            p.wr > (p.th - 1) * sy + (KH - 1) && p.wc > (p.tw - 1) * sx + (KW - 1) * dx &&
                            p.win_bytes + p.xch_bytes + p.tab_bytes + 4 * WINDOW_PANEL * 4 + most * 4 + (sums ? (int64_t)p.wr * p.wc * 4 : 0) <= p.lds &&
                            // (quotients by reciprocals are exact while x * d stays below 2^32)
                            (row + 512) * std::max(row, (int64_t)per_x) < ((int64_t)1 << 32) && (int64_t)most * p.tw < ((int64_t)1 << 32) && (K / 16 + 16) * cpr < ((int64_t)1 << 32) && most <= 512;
            if (!ok)
            {
                std::printf("%d x %d x %d x %d -> %d, %d x %d stride %d %d dil %d pad %d planes %d sums %d: rs %d wk %d ppw %d tile %d x %d of %d x %d lds %ld\n", batch, H, W, C, N, KH, KW, sx, sy, dx,
                            pad, planes, sums, p.rs, p.wk, p.ppw, p.th, p.tw, p.ty, p.tx, (long)p.lds);
                return 1;
            }
        }
    }
    std::printf("%ld %ld\n", taken, split);
    return 0;
}
"""


def test_every_division_fits(tmp_path):
    src, exe = tmp_path / "sweep.cpp", tmp_path / "sweep"
    src.write_text(SWEEP)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), str(src)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
    taken, split = map(int, r.stdout.split())
    assert taken > 200000 and split > 10000


def _case(shape, wshape, stride, pad, dil=(1, 1), dt=np.int8, w_dt=np.int8, layout=capi.NHWC, mults=None, seed=0):
    from gpu_util import announce
    from test_gpu_conv import run_conv
    rng = np.random.default_rng(sum(shape) + sum(wshape) + seed)
    info, w_info = np.iinfo(dt), np.iinfo(w_dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(w_info.min, w_info.max + 1, size=wshape).astype(w_dt)
    zp, ozp = (5, -7) if dt == np.int8 else (131, 9)
    w_zp = 0 if w_dt == np.int8 else 126
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    reals = rng.uniform(0.5, 2.0, size=wshape[0]) * 40.0 / ((wshape[1] * wshape[2] * wshape[3]) ** 0.5 * 74.0 * 74.0)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, reals, 1.0)
    if mults == "negative":
        mult = [-m if i % 3 == 0 else m for i, m in enumerate(mult)]
    elif mults == "left":
        mult, shift = [m >> 12 if i % 2 else m for i, m in enumerate(mult)], [-1 if i % 2 else s for i, s in enumerate(shift)]
    announce("conv window", shape, wshape, stride, pad, dil, dt.__name__, w_dt.__name__, layout, mults)
    got, name = run_conv(src, w, bias, zp, w_zp, mult, shift, ozp, info.min, info.max, stride, pad, dil, layout=layout)
    want = oracle.conv_nhwc_direct(src, w, bias, zp, w_zp, mult, shift, ozp, info.min, info.max, stride, pad, dil)
    assert 0.05 < ((want > info.min) & (want < info.max)).mean()
    assert "window" in name, name
    np.testing.assert_array_equal(got, want)


NHWC = [
    ((2, 14, 14, 256), (256, 3, 3, 256), (1, 1), (1, 1, 1, 1), (1, 1)),   # pieces of 16 bytes, 4 panels
    ((3, 13, 11, 40), (70, 3, 3, 40), (1, 1), (1, 1, 1, 1), (1, 1)),      # pieces of 8, 40 channels in 48, a second panel of 6 columns
    ((2, 9, 10, 8), (130, 5, 5, 8), (1, 1), (2, 2, 2, 2), (1, 1)),        # 8 in 16
    ((1, 16, 17, 88), (100, 3, 3, 88), (2, 1), (1, 0, 2, 1), (1, 1)),     # steps of two, uneven padding
    ((2, 12, 13, 56), (33, 3, 3, 56), (1, 2), (2, 2, 2, 2), (2, 1)),      # dilated
    ((1, 3, 300, 72), (8, 1, 3, 72), (1, 1), (1, 0, 1, 0), (1, 1)),       # rows in pieces, 8 columns
    ((1, 5, 5, 1000), (90, 1, 1, 1000), (1, 1), (0, 0, 0, 0), (1, 1)),    # deep K, few pixels
    ((7, 7, 7, 488), (200, 3, 3, 488), (1, 1), (1, 1, 1, 1), (1, 1)),
    ((1, 1, 1, 24), (5, 1, 1, 24), (1, 1), (0, 0, 0, 0), (1, 1)),         # one pixel, one piece of K short of 64
]
NCHW = [
    ((2, 28, 28, 128), (128, 3, 3, 128), (1, 1), (1, 1, 1, 1), (1, 1)),
    ((3, 7, 7, 33), (40, 3, 3, 33), (1, 1), (1, 1, 1, 1), (1, 1)),        # rows of 7 bytes, 33 channels in 48
    ((2, 6, 4, 16), (17, 3, 3, 16), (1, 1), (1, 1, 1, 1), (1, 1)),        # the narrowest rows
    ((2, 19, 22, 70), (3, 5, 5, 70), (2, 2), (2, 2, 2, 2), (1, 1)),       # 3 columns
    ((1, 4, 290, 20), (70, 3, 3, 20), (1, 1), (1, 1, 1, 1), (1, 1)),      # rows in pieces
    ((2, 9, 9, 100), (64, 3, 3, 100), (3, 1), (0, 3, 4, 1), (1, 2)),
    ((5, 2, 9, 48), (200, 1, 1, 48), (1, 1), (0, 0, 0, 0), (1, 1)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(NHWC)))
@pytest.mark.parametrize("dt,w_dt", [(np.int8, np.int8), (np.uint8, np.uint8), (np.uint8, np.int8)])
def test_pixels(case, dt, w_dt):
    _case(*NHWC[case], dt, w_dt)


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(NCHW)))
@pytest.mark.parametrize("dt,w_dt", [(np.int8, np.int8), (np.uint8, np.uint8), (np.int8, np.uint8)])
def test_planes(case, dt, w_dt):
    _case(*NCHW[case], dt, w_dt, capi.NCHW)


@pytest.mark.gpu
@pytest.mark.parametrize("mults", ["negative", "left"])
@pytest.mark.parametrize("layout", [capi.NHWC, capi.NCHW])
def test_general_requantisation(mults, layout):
    _case((2, 12, 13, 40), (70, 3, 3, 40), (1, 1), (1, 1, 1, 1), layout=layout, mults=mults)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [capi.NHWC, capi.NCHW])
def test_updates_unaligned_tensors_and_graphs(layout):
    """An update that brings a weights offset (another division: the sums take room) and one that leaves the stage for the integer
    multiplier (another kernel, whose buffers the recorded run finds), tensors on any byte, replays of a recorded run."""
    from gpu_util import announce, to_dev, torch_dev
    from test_gpu_prepare_order import _Graph
    torch = torch_dev()
    rng = np.random.default_rng(5)
    B_, H, W, C, N = 3, 11, 12, 24, 72
    src, w = rng.integers(0, 256, size=(B_, H, W, C)).astype(np.uint8), rng.integers(0, 256, size=(N, 3, 3, C)).astype(np.uint8)
    bias = rng.integers(-3000, 3000, size=N).astype(np.int32)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, [40.0 / (216 ** 0.5 * 74.0 * 74.0)], 1.0)
    rq = capi.requant(mult[0], shift[0], 9, 0, 255, False)
    nchw = layout == capi.NCHW
    turn = (lambda x: np.ascontiguousarray(x.transpose(0, 3, 1, 2))) if nchw else (lambda x: x)
    conv = capi.Conv(capi.conv_desc(B_, H, W, C, N, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), capi.U8, capi.U8, capi.U8, -131, -128, 131, rq, 0, layout))
    conv.prepare(to_dev(turn(w)), to_dev(bias))
    # both tensors one byte into their buffers
    sbuf = torch.zeros(src.size + 16, dtype=torch.uint8, device="cuda")
    dbuf = torch.zeros(B_ * H * W * N + 16, dtype=torch.uint8, device="cuda")
    sbuf[1:1 + src.size] = to_dev(turn(src).reshape(-1))
    s, d = sbuf[1:1 + src.size], dbuf[1:1 + B_ * H * W * N]
    side = torch.cuda.Stream()

    def check(w_zp, want=None):
        torch.cuda.synchronize()
        got = d.cpu().numpy().reshape((B_, N, H, W) if nchw else (B_, H, W, N))
        if want is None:
            want = oracle.conv_nhwc_direct(src, w, bias, 131, w_zp, mult, shift, 9, 0, 255, (1, 1), (1, 1, 1, 1), (1, 1))
        np.testing.assert_array_equal(got.transpose(0, 2, 3, 1) if nchw else got, want)
        d.zero_()
        torch.cuda.synchronize()

    announce("conv window, updates", layout)
    conv.run(s, d)
    assert "window" in conv.kernel_name
    check(128)
    for w_zp in (120, 128, 135):
        conv.update_quant(-131, -w_zp, 131, rq)
        conv.run(s, d)
        assert "window" in conv.kernel_name
        check(w_zp)
        graph = _Graph(lambda st: conv.run(s, d, st), side)
        for _ in range(3):
            graph.launch(side)
            check(w_zp)
        graph.close()
    # the integer multiplier: not this kernel's; the first run of another one is recorded
    conv.update_quant(-131, -120, 131, capi.requant(3, 9, 11, 0, 255, False, capi.STAGE_SCALE))
    graph = _Graph(lambda st: conv.run(s, d, st), side)
    assert "window" not in conv.kernel_name
    acc = np.zeros((B_, H, W, N), np.int64)
    padded = np.full((B_, H + 2, W + 2, C), 131, np.int64)
    padded[:, 1:-1, 1:-1] = src
    for ky in range(3):
        for kx in range(3):
            acc += (padded[:, ky:ky + H, kx:kx + W] - 131) @ (w[:, ky, kx].astype(np.int64) - 120).T
    want = np.clip(((acc + bias + 11) * 3) >> 9, 0, 255)
    for _ in range(2):
        graph.launch(side)
        check(120, want)
    graph.close()
    conv.close()
