// Which convolutions gemm_window.hip takes and how a launch divides them. Plain C++, in one place: what the rule accepts is what the
// launch can run. G: a geometry with ConvGeom's members, of the caller's channels.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

namespace mi355
{
constexpr int WINDOW_WAVES = 8;        // per workgroup: two share the columns, the others K or the pixels
constexpr int WINDOW_PANEL = 64;       // output channels of a workgroup at a time
constexpr int WINDOW_MOST_LDS = 160 * 1024;
constexpr int WINDOW_OPITCH = 80;      // LDS bytes of a pixel's row of results

struct WindowPlan
{
    int     rs = 0, wk = 0;     // blocks of 16 pixels per wave; waves that share K (the others share the pixels)
    int     th = 0, tw = 0;     // output rows and columns of a workgroup's tile
    int     ty = 0, tx = 0;     // ... tiles down and across an image
    int     u = 0;              // 16-byte pieces of LDS per window pixel
    int     wr = 0, wc = 0;     // window rows and columns
    int     panels = 0, ppw = 0; // panels of output channels, and how many of them a workgroup takes one after the other
    int64_t win_bytes = 0, tab_bytes = 0, xch_bytes = 0, lds = 0;
    double  us = 0;
};

// Pixels of a tile: rs blocks of 16 per wave, wk waves on the same ones
inline int conv_window_pixels(int rs, int wk)
{
    return rs * 16 * (WINDOW_WAVES / 2 / wk);
}

// K of the packed weights: whole taps of cp channels (C rounded up to 16)
template <typename G>
int64_t conv_window_k(const G &c)
{
    return (int64_t)c.KH * c.KW * ((c.C + 15) / 16 * 16);
}

// One division of a convolution; false where it does not fit
template <typename G>
bool conv_window_try(const G &c, int batch, int N, bool planes, bool sums, int rs, int wk, int ppw, int cus, WindowPlan &p)
{
    const int most = conv_window_pixels(rs, wk);
    p.rs = rs, p.wk = wk, p.ppw = ppw;
    p.tx = (c.OW + most - 1) / most, p.tw = (c.OW + p.tx - 1) / p.tx;
    p.th = std::min<int>(c.OH, p.tx > 1 ? 1 : most / c.OW);
    p.ty = (c.OH + p.th - 1) / p.th, p.th = (c.OH + p.ty - 1) / p.ty;
    const int64_t wr = (int64_t)(p.th - 1) * c.stride_y + (int64_t)(c.KH - 1) * c.dil_y + 1;
    const int64_t wc = (int64_t)(p.tw - 1) * c.stride_x + (int64_t)(c.KW - 1) * c.dil_x + 1;
    const int64_t cpr = (c.C + 15) / 16, K = conv_window_k(c);
    // 16 pixels at a window step of stride_x, 4 pieces of each: free of bank conflicts where stride_x * u is 2 modulo 4 (see NARROW_PAD_PIECES);
    // at even steps an odd u is the nearest to that
    int64_t u = cpr;
    while (c.stride_x % 2 != 0 ? u % 4 != 2 : u % 2 != 1)
        ++u;
    if (wr * wc > (1 << 16) || wr * wc * u > (1 << 14) || K > (1 << 16))
        return false;
    p.wr = (int)wr, p.wc = (int)wc, p.u = (int)u;
    p.panels    = (N + WINDOW_PANEL - 1) / WINDOW_PANEL;
    p.win_bytes = (wr * wc * u * 16 + 1023) & ~(int64_t)1023;
    p.tab_bytes = ((K + 63) / 64 + 2 * wk) * 16;
    const int64_t out = planes ? (int64_t)WINDOW_PANEL * (most + 16) : (int64_t)most * WINDOW_OPITCH;
    p.xch_bytes = std::max<int64_t>(wk == 1 ? 0 : WINDOW_WAVES * 1024 * rs * (wk == 4 ? 3 : 2) / 2, out);
    p.lds       = p.win_bytes + p.tab_bytes + p.xch_bytes + 4 * WINDOW_PANEL * 4 + most * 4 + (sums ? ((wr * wc * 4 + 15) & ~(int64_t)15) : 0);
    if (p.lds > WINDOW_MOST_LDS)
        return false;
    const int64_t tiles = (int64_t)batch * p.ty * p.tx, groups = (p.panels + ppw - 1) / ppw, wgs = tiles * groups;
    if (wgs > INT32_MAX / 2)
        return false;
    // The price, in microseconds, fitted to 1500 timings (169 convolutions, every division; 8 % mean error, the choice 1 % slower than the best
    // division on average): what a round of workgroups costs (two per compute unit where the LDS holds them), and per workgroup on a
    // compute unit its matrix instructions, the KiB of its window and its output pixels.
    const double nkb = std::ceil(K / 64.0), ns = std::ceil(nkb / wk), per = (double)p.panels / (double)groups;
    const double full = std::ceil((double)wgs / cus), rounds = std::ceil((double)wgs / ((double)cus * std::min<int64_t>(2, WINDOW_MOST_LDS / p.lds)));
    const double mfma = rs * 2 * ns * 16 * (WINDOW_WAVES / 4) / 2100.0, win = (double)wr * wc * cpr / 64.0, pixels = most / 64.0;
    p.us = 1.75 + rounds * (1.62 + 1.34 * (per - 1) + 0.041 * ns * per + (planes ? 0.43 : 0.0)) +
           full * (0.71 + 0.25 * (per - 1) + 0.99 * mfma * per + (planes ? 0.058 : 0.045) * win + (planes ? 0.19 : 0.098) * pixels * per);
    return true;
}

// C a multiple of 8 (any with planes, rows of at least 4 pixels), and the cheapest of the divisions that fit
template <typename G>
bool conv_window_plan(const G &c, int batch, int N, bool planes, bool sums, int cus, WindowPlan &best)
{
    if (batch < 1 || N < 1 || c.C < 8 || (planes ? c.W < 4 : c.C % 8 != 0) || (int64_t)c.H * c.W * c.C >= (1 << 30) || (int64_t)c.OH * c.OW >= (1 << 24))
        return false;
    bool found = false;
    for (int wk : {1, 2, 4})
        for (int rs : {2, 4})
            for (int ppw : {1, 2})
            {
                WindowPlan p;
                if ((ppw == 1 || (N > WINDOW_PANEL && wk * rs != 16 && !(wk == 4 || (wk == 1 && rs == 2)))) &&
                    conv_window_try(c, batch, N, planes, sums, rs, wk, ppw, cus, p) && (!found || p.us < best.us))
                    best = p, found = true;
            }
    return found;
}

// What the other kernels take for the same convolution, in microseconds. K: of their weights; tiles_us: the price of the pipelined kernel's tiles; narrow: the narrow
// kernel runs it; copied: its channels are padded in a pass in front; planes: the source is transposed in front, and behind the narrow kernel the
// result. Fitted to the same 169 convolutions (9 and 11 % mean error).
template <typename G>
double conv_other_us(const G &c, int batch, int N, int K, bool planes, bool sums, bool copied, bool narrow, double tiles_us, int cus)
{
    const double M = (double)batch * c.OH * c.OW, cp = (c.C + 15) / 16 * 16.0, panels = std::ceil(N / 64.0);
    const double src = (double)batch * c.H * c.W * c.C * 1e-6, dst = M * N * 1e-6;
    double       us  = tiles_us * 0.85;
    if (narrow)
    {
        const double r = std::max(1.0, M / (128.0 * cus));
        const bool   band = !copied && c.C >= 64 && (c.C & (c.C - 1)) == 0 && M > 128.0 * cus; // (the form with the window in LDS: see halo_plan)
        us = (2.45 + r * panels * (1.0 + 0.46 * K / 192.0) + 0.16 * (panels - 1) + (sums ? 0.22 * r : 0.0)) * (band ? 0.87 : 1.0);
    }
    if (copied)
        us += (narrow ? 2.1 : 2.7) + 0.8 * src * cp / c.C;
    if (planes)
        us += narrow ? 6.5 + 0.78 * src + 0.23 * dst : 4.2 + 0.24 * src + 0.75 * dst;
    return us;
}

// Taken where it is cheaper by more than the prices are off: by a tenth; by a quarter from 40 us on (large matrices, where tiles of 128 x 128
// re-read less); by three tenths where K slices are the other choice, the price that is least sure
inline bool conv_window_pays(double window_us, double other_us, bool slices)
{
    return window_us < other_us * (slices ? 0.7 : other_us > 40 ? 0.75 : 0.9);
}
} // namespace mi355
