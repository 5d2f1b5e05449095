// Convolution of few channels (a first layer: RGB), straight from the caller's NHWC image.
//
// The KW taps of an image row are KW * C consecutive bytes, at most 32 here. A workgroup takes a band of output rows of one image and a
// panel of up to 64 output channels: it copies the window of input rows under the band to LDS byte for byte (padding included, signs
// normalised), and a lane forms the 16 bytes of its (pixel, k) from the dwords that hold them, shifted into place: in the
// layout of patch rows (mi355_conv_create), K = KH pieces of 16 or 32 bytes, whose weights are packed the same way; what
// lies beyond KW * C in a piece are neighbouring pixels, which meet zero weights. The weights of the panel stay in registers.
//
// Against patch rows written out in memory and fetched by the narrow kernel (KH / stride times each) the image crosses the chip
// once: 32 x 224 x 224 x 3 -> 64, 7 x 7, stride 2: 9.4 us of copy and 30 of the narrow kernel, 20.6 in one launch, 18.4 with two vector instructions less per output; 29 x 85 x 85 x 3 -> 32:
// 10.2, 6.8; 2 x 93 x 93 x 3 -> 32, 5 x 5: 7.6, 4.7. What bounds it: the vector ALU, 5.75 instructions per output for the
// requantisation and about 60 per 32 pixels for the operands, at 3 waves per SIMD, then the output's bytes.
#include "conv_rows_plan.hpp"
#include "mfma_common.hpp"

namespace mi355
{
struct RowsArgs
{
    GemmArgs g;        // A: the image; conv: its geometry with the caller's channels; K: KH * piece bytes
    int32_t  pieces;   // 16-byte pieces per window row (1 or 2)
    int32_t  band, bands, pitch, win_rows; // output rows per workgroup, workgroups per image; LDS bytes per window row, window rows
    int32_t  row_bytes, left_bytes;        // bytes of an image row, of the padding in front of it
    int32_t  batch, panels;                // panels: 0 where they run one after the other
};

template <int NKB>
__global__ __launch_bounds__(ROWS_WAVES * 64) __attribute__((amdgpu_waves_per_eu(NKB <= 2 ? 4 : 3))) void conv_rows_kernel(RowsArgs a, uint32_t flip)
{
    constexpr int    BPITCH = NKB * 64 + 32, OPITCH = ROWS_OPITCH; // (a panel row 32 bytes past a multiple of 64: see NARROW_PAD_PIECES)
    constexpr int    NT = ROWS_WAVES * 64, NPAR = PAR_ROWS;
    static_assert(NPAR == ROWS_NPAR, "conv_rows_fixed_lds counts them");
    const GemmArgs  &g = a.g;
    const ConvGeom  &c = g.conv;
    const EpiParams &p = g.epi;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char    *panel = smem;                                   // 64 rows of BPITCH
    int32_t *par   = (int32_t *)(smem + 64 * BPITCH);        // [NPAR][64]
    char    *out   = smem + 64 * BPITCH + NPAR * 256;        // a wave's 32 x 64 results
    char    *win   = out + ROWS_WAVES * 32 * OPITCH;         // win_rows of a.pitch
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lh = lane >> 4;
    int wg = (int)blockIdx.x, n0 = (int)blockIdx.y * 64;
    if (a.panels > 1) // panels of one band side by side (see conv_rows_launch), 8 workgroups apart: on the same die
    {
        const int at = wg / (8 * a.panels), in = wg - at * 8 * a.panels;
        wg = at * 8 + (in & 7), n0 = (in >> 3) * 64;
        if (wg >= a.bands * a.batch)
            return;
    }
    const int n = wg / a.bands, band = wg - n * a.bands;
    const int oy0 = band * a.band, rows = min(a.band, c.OH - oy0), npix = rows * c.OW;
    const int qflag = p.qp_flag ? *p.qp_flag : 1;

    // the panel of weights: 64 rows of NKB * 64 bytes
    for (int i = tid; i < 64 * NKB * 4; i += NT)
    {
        const int r = i / (NKB * 4), q = i % (NKB * 4);
        *(v4i *)(panel + r * BPITCH + q * 16) = *(const v4i *)(g.Bp + (int64_t)(n0 + r) * g.Kp + q * 16);
    }
    if (p.qp_flag)
        for (int i = tid; i < PAR_LOADS * 64; i += NT)
            park_constant(par, i, 64, i < 64 ? p.colvec[n0 + i] : p.qp[(int64_t)(i / 64 - 1) * p.qp_stride + n0 + i % 64], p.result_offset);
    // the window, a dword per thread and step, four steps of loads at a time
    {
        const int      per_row = a.pitch / 4, total = a.win_rows * per_row;
        const int      iy0 = oy0 * c.stride_y - c.pad_top;
        const int8_t  *image = g.A + (int64_t)n * c.H * a.row_bytes;
        for (int i0 = tid; i0 < total; i0 += 4 * NT)
        {
            uint32_t lo[4], hi[4], keep[4], sh[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const int i = i0 + u * NT, r = i / per_row, x = (i - r * per_row) * 4 - a.left_bytes, iy = iy0 + r;
                lo[u] = hi[u] = keep[u] = sh[u] = 0;
                if (i < total && iy >= 0 && iy < c.H && x > -4 && x < a.row_bytes)
                {
                    // bytes x .. x + 3 of the row, those in [0, row_bytes) count; only dwords that hold one of them are read
                    const int8_t   *at = image + (int64_t)iy * a.row_bytes + max(x, 0);
                    const uint32_t  m  = (uint32_t)(uintptr_t)at & 3u;
                    const int       skip = max(-x, 0), left = min(a.row_bytes - max(x, 0), 4 - skip); // valid bytes from `at` on
                    const int8_t   *lp = at - m;
                    lo[u]   = *(const uint32_t *)lp;
                    hi[u]   = m + (uint32_t)left > 4u ? *(const uint32_t *)(lp + 4) : 0u;
                    sh[u]   = m | ((uint32_t)skip << 8);
                    keep[u] = (left >= 4 ? ~0u : (1u << (8 * left)) - 1u) << (8 * skip);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const int i = i0 + u * NT;
                if (i < total)
                {
                    const uint32_t v = __builtin_amdgcn_alignbyte(hi[u], lo[u], sh[u] & 3u) << (8 * (sh[u] >> 8));
                    *(uint32_t *)(win + (int64_t)i * 4) = ((v & keep[u]) | (c.pad_word & ~keep[u])) ^ flip;
                }
            }
        }
    }
    __syncthreads();

    v4i fb[NKB][4];
    int koff[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
    {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            fb[kb][q] = *(const v4i *)(panel + (q * 16 + lr) * BPITCH + (kb * 4 + lh) * 16);
        const int piece = kb * 4 + lh, ky = a.pieces == 2 ? piece >> 1 : piece;
        // (pieces beyond the last row meet zero weights: any bytes of the window do)
        koff[kb] = min(ky, c.KH - 1) * c.dil_y * a.pitch + (a.pieces == 2 ? (piece & 1) * 16 : 0);
    }
    const int     cols = min(g.N - n0, 64);
    char         *mine = out + wave * 32 * OPITCH;
    char         *D    = (char *)g.D + ((int64_t)n * c.OH + oy0) * c.OW * g.ldd + n0;
    const pk16_t  lo16 = {(int16_t)p.lo, (int16_t)p.lo}, hi16 = {(int16_t)p.hi, (int16_t)p.hi};
    for (int t = wave; t * 32 < npix; t += ROWS_WAVES)
    {
        v4i acc[2][4];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
        {
            const int   pix = min(t * 32 + rb * 16 + lr, npix - 1);
            const int   r = fast_div(pix, c.magic_OW), x = pix - r * c.OW;
            const int   at = r * c.stride_y * a.pitch + x * c.stride_x * c.C;
            const char *from = win + (at & ~3);
            const int   m    = at & 3;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                acc[rb][q] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
            {
                uint32_t w[5];
#pragma unroll
                for (int d = 0; d < 5; ++d)
                    w[d] = *(const uint32_t *)(from + koff[kb] + 4 * d);
                v4i fa;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    fa[d] = (int)__builtin_amdgcn_alignbyte(w[d + 1], w[d], (uint32_t)m);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[rb][q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[kb][q], fa, acc[rb][q], 0, 0, 0);
            }
        }
        // requantise into the wave's own 32 x 64 bytes of LDS (accumulator layout as in epilogue_store_t)
        auto each = [&](auto requant4)
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                if (q * 16 >= cols)
                    continue;
                const int col = q * 16 + 4 * lh;
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
                    *(uint32_t *)(mine + (rb * 16 + lr) * OPITCH + col) = requant4(acc[rb][q], col);
            }
        };
        auto one_by_one = [&](auto requant)
        {
            each([&](v4i v, int col) {
                int32_t o[4];
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    o[d] = requant(v[d], col + d);
                const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)o[1], (uint32_t)o[0], 0x0c0c0400u);
                const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)o[3], (uint32_t)o[2], 0x0c0c0400u);
                return __builtin_amdgcn_perm(p23, p01, 0x05040100u);
            });
        };
        if (qflag == 0 && p.qp_std)
            each([&](v4i v, int col) {
                const v4i cv = *(const v4i *)(par + PAR_CV * 64 + col);
                int32_t   x[4];
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    x[d] = (int32_t)((uint32_t)v[d] + (uint32_t)cv[d]);
                return std_requant4(x, *(const v4i *)(par + PAR_M * 64 + col), *(const v4i *)(par + PAR_SM1 * 64 + col),
                                    *(const v4i *)(par + PAR_ADD * 64 + col), lo16, hi16);
            });
        else if ((qflag & 1) == 0)
            one_by_one([&](int32_t v, int col) {
                return fast_requant((int32_t)((uint32_t)v + (uint32_t)par[PAR_CV * 64 + col]), par[PAR_M * 64 + col], par[PAR_SM1 * 64 + col],
                                    p.result_offset, p.lo, p.hi);
            });
        else
            one_by_one([&](int32_t v, int col) {
                int first = n0; // (hidden: the addresses of 16 columns in three vectors, kept over the loop, were 100 registers)
                asm volatile("" : "+s"(first));
                const int j = min(first + col, g.N - 1);
                return epi_fixedpoint(v, p.colvec[j], 0, p.mult ? p.mult[j] : p.mult_s, p.shift ? p.shift[j] : p.shift_s, p);
            });
        // ... and out, 16, 4 or 1 byte per lane
        auto leave = [&](auto bytes_c)
        {
            constexpr int W = decltype(bytes_c)::value, LPR = 64 / W, RPI = 64 / LPR;
#pragma unroll
            for (int it = 0; it < 32 / RPI; ++it)
            {
                const int r = it * RPI + lane / LPR, cc = (lane % LPR) * W, pix = t * 32 + r;
                if (pix >= npix || cc >= cols)
                    continue;
                char       *to = D + (int64_t)pix * g.ldd + cc;
                const char *at = mine + r * OPITCH + cc;
                if constexpr (W == 16)
                    __builtin_nontemporal_store(*(const v4i *)at, (v4i *)to); // (N % 16 == 0 where this form is taken)
                else if constexpr (W == 4)
                    *(int *)to = *(const int *)at;
                else
                    *to = *at;
            }
        };
        if (p.vec_store16 && g.N % 16 == 0)
            leave(std::integral_constant<int, 16>{});
        else if (p.vec_store && g.N % 4 == 0)
            leave(std::integral_constant<int, 4>{});
        else
            leave(std::integral_constant<int, 1>{});
    }
}

// conv: the caller's geometry, pad_word the raw padding byte replicated
int conv_rows_launch(bool flip_a, const GemmArgs &args, int batch, hipStream_t s)
{
    RowsArgs        a{};
    const ConvGeom &c      = args.conv;
    const int       panels = (args.N + 63) / 64;
    RowsPlan        p;
    if (args.N < 1 || !conv_rows_plan(c, batch, panels, p) || args.epi.rowsum_mul != 0 || args.epi.rowvec != nullptr || args.epi.stage != 0)
        return (int)hipErrorInvalidValue;
    if (args.Kp < p.nkb * 64 || round_up(args.N, PACK_N_ALIGN) < panels * 64)
        return (int)hipErrorInvalidValue;
    a.g      = args;
    a.pieces = p.pieces, a.band = p.band, a.bands = p.bands, a.pitch = p.pitch, a.win_rows = p.win_rows;
    a.row_bytes  = c.W * c.C;
    a.left_bytes = c.pad_left * c.C;
    // The panels of a band write different parts of the same lines. One panel after the other over the whole image batch, a large
    // destination's lines leave the caches in between and go out twice: in pieces of 16 bytes and from 24 MB on the panels
    // go side by side (16 x 186 x 189 x 3 -> 112, 5 x 5: 55.3 and 46.1 us, by patch rows 51.0; 30 x 192 x 192 x 3 -> 96, 3 x 3: 91.3, 80.0,
    // 88.2; not 2 x 408 x 408 x 4 -> 65, 3 x 3: 28.8, 33.7, nor 19 MB of 96 columns, 7 x 7: 18.7, 20.8; 128 columns: no difference)
    const bool side = panels > 1 && args.epi.vec_store16 && args.N % 16 == 0 && args.N % 64 != 0 && (int64_t)batch * c.OH * c.OW * args.N > 24000000;
    a.batch = batch, a.panels = side ? panels : 0;
    const dim3 grid(side ? (unsigned)(((int64_t)batch * p.bands + 7) / 8 * 8 * panels) : (unsigned)(batch * p.bands), side ? 1u : (unsigned)panels), block(ROWS_WAVES * 64);
    const uint32_t flip = flip_a ? 0x80808080u : 0u;
    switch (p.nkb)
    {
        case 1: conv_rows_kernel<1><<<grid, block, p.lds, s>>>(a, flip); break;
        case 2: conv_rows_kernel<2><<<grid, block, p.lds, s>>>(a, flip); break;
        case 3: conv_rows_kernel<3><<<grid, block, p.lds, s>>>(a, flip); break;
        case 4: conv_rows_kernel<4><<<grid, block, p.lds, s>>>(a, flip); break;
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}
} // namespace mi355
