// Which convolutions gemm_rows.hip takes and how a launch divides them. Plain C++, in one place: what the rule accepts is what the
// launch can run. G: a geometry with ConvGeom's members, of the caller's channels.
#pragma once
#include <cstdint>

namespace mi355
{
constexpr int ROWS_WAVES = 4, ROWS_MAX_LDS = 64 * 1024; // (two workgroups per compute unit)
constexpr int ROWS_OPITCH = 80, ROWS_NPAR = 4;          // LDS bytes of a wave's row of 64 results; words of constants per column

struct RowsPlan
{
    int     pieces, nkb;                    // 16-byte pieces per window row (1 or 2), blocks of 64 of K = KH * pieces * 16
    int     band, bands, pitch, win_rows;   // output rows per workgroup, workgroups per image; LDS bytes per window row, window rows
    int64_t lds;
};

template <typename G>
int conv_rows_pieces(const G &c)
{
    const int64_t row = (int64_t)c.KW * c.C, pieces = (row + 15) / 16;
    return c.dil_x == 1 && pieces <= 2 && c.KH * pieces <= 16 ? (int)pieces : 0;
}
template <typename G>
int64_t conv_rows_window(const G &c, int rows)
{
    return (int64_t)(rows - 1) * c.stride_y + (int64_t)(c.KH - 1) * c.dil_y + 1;
}
// panel, constants, a wave's results
inline int64_t conv_rows_fixed_lds(int nkb)
{
    return 64 * (nkb * 64 + 32) + ROWS_NPAR * 256 + ROWS_WAVES * 32 * ROWS_OPITCH;
}

// The window of one output row takes at most 30 KiB (with the 29.5 KiB of conv_rows_fixed_lds(4) that is inside ROWS_MAX_LDS)
template <typename G>
bool conv_rows_applies(const G &c)
{
    const int pieces = conv_rows_pieces(c);
    if (pieces == 0)
        return false;
    const int64_t pitch = ((int64_t)(c.OW - 1) * c.stride_x) * c.C + pieces * 16 + 40; // at most (see below)
    return pitch <= 30 * 1024 && pitch * conv_rows_window(c, 1) <= 30 * 1024 && (int64_t)c.OH * c.OW < (1 << 24);
}

// As many output rows as give a wave about 4 tiles of 32 pixels, fewer where that leaves the chip without two workgroups per
// compute unit (512 in all), within 40 KiB of window and what the panel leaves of the LDS
template <typename G>
bool conv_rows_plan(const G &c, int batch, int panels, RowsPlan &p)
{
    if (!conv_rows_applies(c) || batch < 1 || panels < 1)
        return false;
    p.pieces = conv_rows_pieces(c);
    p.nkb    = (c.KH * p.pieces + 3) / 4;
    // the last pixel's pieces and the dword behind them end inside the window row
    p.pitch        = (((c.OW - 1) * c.stride_x * c.C + p.pieces * 16 + 8 + 15) & ~15) + 16;
    auto lds       = [&](int rows) { return conv_rows_fixed_lds(p.nkb) + conv_rows_window(c, rows) * p.pitch; };
    const int most = (ROWS_WAVES * 32 * 4 + c.OW - 1) / c.OW;
    p.band         = c.OH < most ? c.OH : most;
    while (p.band > 1 && (conv_rows_window(c, p.band) * p.pitch > 40 * 1024 || lds(p.band) > ROWS_MAX_LDS ||
                          (int64_t)batch * ((c.OH + p.band - 1) / p.band) * panels < 512))
        --p.band;
    p.bands = (c.OH + p.band - 1) / p.band, p.win_rows = (int)conv_rows_window(c, p.band), p.lds = lds(p.band);
    return p.lds <= ROWS_MAX_LDS && ((int64_t)batch * p.bands + 7) * panels <= INT32_MAX; // (workgroups)
}
} // namespace mi355
