"""Few channels straight from the image: every convolution that the rule takes has a launch (checked on the host over the rule's whole
range), bands of several rows that do and do not divide the image, and windows near the limit."""
import os
import subprocess

import numpy as np
import pytest

import oracle
from computelibrary_amd import capi

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "computelibrary_amd", "csrc")

SWEEP = r"""
#include "conv_rows_plan.hpp"
#include <cstdio>
struct G { int H, W, C, KH, KW, OH, OW, stride_x, stride_y, pad_left, pad_top, dil_x, dil_y; };
int main()
{
    long taken = 0, banded = 0;
    for (int C = 1; C <= 8; ++C) for (int KW = 1; KW <= 17; ++KW) for (int KH = 1; KH <= 16; KH += KH < 8 ? 1 : 4)
    for (int sx = 1; sx <= 4; ++sx) for (int sy = 1; sy <= 4; ++sy) for (int dy = 1; dy <= 3; dy += 2)
    for (int W = 8; W <= 4096; W += W < 256 ? 13 : 61) for (int H = 7; H <= 1024; H = H * 5 / 2)
    {
        G g{H, W, C, KH, KW, (H + 2 * (KH / 2) - (KH - 1) * dy - 1) / sy + 1, (W + 2 * (KW / 2) - KW) / sx + 1, sx, sy, KW / 2, KH / 2, 1, dy};
        if (H + 2 * (KH / 2) < (KH - 1) * dy + 1 || W + 2 * (KW / 2) < KW || !mi355::conv_rows_applies(g)) continue;
        for (int batch = 1; batch <= 300; batch *= 17) for (int panels = 1; panels <= 2; ++panels)
        {
            mi355::RowsPlan p;
            ++taken;
            const bool ok = mi355::conv_rows_plan(g, batch, panels, p);
            if (!ok || p.band < 1 || p.band > g.OH || p.nkb < 1 || p.nkb > 4 || p.lds > 65536 || (long)p.bands * p.band < g.OH || (long)(p.bands - 1) * p.band >= g.OH ||
                // the last pixel's pieces and one dword lie inside the window
                (g.OW - 1) * sx * C + (p.pieces - 1) * 16 + 20 > p.pitch || (p.band - 1) * sy + (KH - 1) * dy >= p.win_rows)
            { std::printf("C %d KW %d KH %d stride %d %d dil %d W %d H %d batch %d panels %d: %d lds %ld\n", C, KW, KH, sx, sy, dy, W, H, batch, panels, ok, (long)p.lds); return 1; }
            banded += p.band > 1;
        }
    }
    std::printf("%ld %ld\n", taken, banded);
    return 0;
}
"""


def test_what_the_rule_takes_can_be_launched(tmp_path):
    src, exe = tmp_path / "sweep.cpp", tmp_path / "sweep"
    src.write_text(SWEEP)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), str(src)])
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
    taken, banded = map(int, r.stdout.split())
    assert taken > 100000 and banded > 10000


def _check(shape, wshape, stride, pad, dt=np.uint8, mult_sign=1, layout=capi.NHWC, seed=0):
    from gpu_util import announce
    from test_gpu_conv import run_conv
    rng = np.random.default_rng(sum(shape) + sum(wshape) + seed)
    info = np.iinfo(dt)
    src = rng.integers(info.min, info.max + 1, size=shape).astype(dt)
    w = rng.integers(-127, 128, size=wshape, dtype=np.int8)
    bias = rng.integers(-3000, 3000, size=wshape[0]).astype(np.int32)
    zp, ozp = (5, -7) if dt == np.int8 else (131, 9)
    reals = rng.uniform(0.5, 2.0, size=wshape[0]) * 40.0 / ((wshape[1] * wshape[2] * wshape[3]) ** 0.5 * 74.0 * 74.0)
    mult, shift = oracle.calculate_quantized_multipliers(1.0, reals, 1.0)
    mult = [m * mult_sign if i % 3 == 0 else m for i, m in enumerate(mult)]
    announce("conv rows plan", shape, wshape, stride, pad, dt.__name__, mult_sign, layout)
    got, name = run_conv(src, w, bias, zp, 0, mult, shift, ozp, info.min, info.max, stride, pad, (1, 1), layout=layout)
    assert name == "implicit_rows_32x64", name
    np.testing.assert_array_equal(got, oracle.conv_nhwc_direct(src, w, bias, zp, 0, mult, shift, ozp, info.min, info.max, stride, pad, (1, 1)))


# windows that the limit of 40 KiB admits and the rest of the LDS does not, under 3 and 4 blocks of K
@pytest.mark.gpu
@pytest.mark.parametrize("shape,wshape,stride,pad", [
    ((128, 49, 581, 4), (32, 5, 5, 4), (4, 4), (2, 2, 2, 2)),
    ((128, 25, 1057, 3), (16, 7, 7, 3), (4, 4), (3, 3, 3, 3))])
def test_window_near_the_limit(shape, wshape, stride, pad):
    _check(shape, wshape, stride, pad)


# the panels of a large destination side by side: two of them, bands not a multiple of 8, a last band that is shorter
@pytest.mark.gpu
@pytest.mark.parametrize("shape,wshape,layout", [
    ((5, 233, 230, 3), (96, 3, 3, 3), capi.NHWC),
    ((3, 301, 299, 3), (112, 4, 4, 3), capi.NCHW),
    ((4, 250, 253, 4), (80, 7, 7, 4), capi.NHWC)])
def test_panels_side_by_side(shape, wshape, layout):
    _check(shape, wshape, (1, 1), (wshape[1] // 2,) * 4, np.int8, layout=layout)
