// Convolution whose input window lies in LDS: the image crosses the vector memory path once instead of KH * KW times, in whatever layout
// the caller has it (NHWC, channels a multiple of 8; NCHW), and nothing but the weights moves in the K loop.
//
// A workgroup of 8 waves takes a tile of output pixels of one image (rows, or a piece of one) and a panel of 64 output channels, or two one
// after the other. It copies the window of input pixels under the tile to LDS, padding included, signs normalised, channels rounded up to 16, and
// works out where each 16-byte piece of K lies there (a table). From then on a wave needs no barrier: operand blocks of A are LDS reads
// at a pixel's address plus the table's offset, those of B come straight from memory to registers in operand order, 2 or 3 K blocks ahead. Two
// waves share the columns; the other four take parts of K (WK of them, added up through LDS behind the loop) or of the pixels. A weights offset
// needs one sum per window pixel, taken on the way in, and KH * KW additions per output pixel.
//
// Against the tiles that fetch every tap (and the passes in front of them: transposes of NCHW, channels padded to 16), us, before and now: 32 x 14 x 14 x
// 256 -> 256, 3 x 3, both operands with zero points 13.0 and 9.7; 32 x 28 x 28 x 128 -> 128, 3 x 3, NCHW 15.9 and 11.1; 16 x 26 x 26 x 72 -> 24, 5 x 5 stride 2
// 11.4 and 6.1; 3 x 42 x 45 x 216 -> 392, 3 x 3 stride 2, NCHW 18.8 and 9.4; 15 x 16 x 17 x 88 -> 112, 1 x 1, NCHW 13.5 and 5.7. What bounds it: latency, one phase
// behind the other with one or two workgroups per compute unit. Of the 9 us that a workgroup of the first takes, arguments are 0.6, the window 2.0,
// the K loop 4.0 (its matrix instructions 2.1), adding the halves up 1.2 and the results 1.0. 4 waves with tiles of 112 pixels were slower (10.2 us: a lone
// wave of a SIMD takes the LDS reads and the matrix instructions in turn), as was B four or eight blocks ahead with half the waves (9.1 and 9.1,
// NCHW 10.9 and 14.4), or loads straight to LDS, whose addresses cost as much and which unsigned pixels had to be passed over after (1.1 us).
#include "conv_window_plan.hpp"
#include "direct_lds.hpp"

#include <atomic>

namespace mi355
{
struct WindowArgs
{
    const int8_t  *src, *B;
    int8_t        *D;
    const int32_t *colvec, *qp, *qp_flag;
    int64_t        qp_stride;
    int32_t        H, W, C, OH, OW, sx, sy, pl, pt;
    int32_t        nblocks, groups, ppw, panels, th, tw, ty, tx, u, wr, wc;
    uint32_t       magic_groups, magic_per, magic_tx; // see ConvGeom::magic_*
    int32_t        row_len, rows_at_once; // loads of a window row, rows that the workgroup loads at a time
    uint32_t       magic_len, magic_x, flip, pad_word;
    int32_t        rowsum_mul, K, kbp; // K: KH * KW * (channels rounded up); kbp: 64-byte blocks of a packed column
    int32_t        KH, KW, dx, dy;
    uint32_t       magic_tw, magic_cpr, magic_KW;
    int32_t        result_offset, lo, hi, qp_std, N, ldd;
    int32_t        tab_off, par_off, rowv_off, psum_off, xch_off; // in LDS, behind the window
};
typedef int v2i_any __attribute__((ext_vector_type(2), aligned(1)));
typedef int v2i __attribute__((ext_vector_type(2)));

// 4 pixels (bytes) of 4 channels (words) -> 4 channels (bytes) of 4 pixels (words)
__device__ __forceinline__ void transpose4(const uint32_t (&d)[4], uint32_t (&o)[4])
{
    const uint32_t a = __builtin_amdgcn_perm(d[1], d[0], 0x05010400u), b = __builtin_amdgcn_perm(d[3], d[2], 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(d[1], d[0], 0x07030602u), e = __builtin_amdgcn_perm(d[3], d[2], 0x07030602u);
    o[0] = __builtin_amdgcn_perm(b, a, 0x05040100u), o[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    o[2] = __builtin_amdgcn_perm(e, c, 0x05040100u), o[3] = __builtin_amdgcn_perm(e, c, 0x07060302u);
}

// The arguments again from where the launch left them: what a phase of the kernel needs is then fetched there, in one batch, instead of being kept
// (and spilled: 100 to 160 scalars of them, and 2200 reads back) from the start
typedef const __attribute__((address_space(4))) WindowArgs *WindowArgsPtr;
__device__ __forceinline__ WindowArgsPtr window_args()
{
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return (WindowArgsPtr)p;
}
typedef const __attribute__((address_space(1))) int8_t  *global_i8;
typedef const __attribute__((address_space(1))) int32_t *global_i32;
typedef __attribute__((address_space(1))) char          *global_out;

enum : int
{
    WINDOW_PIECES16 = 0, // NHWC, C % 16 == 0: 16 bytes at a time, on any byte
    WINDOW_PIECES8  = 1, // NHWC, C % 8 == 0: 8 bytes
    WINDOW_PLANES   = 2  // NCHW: 16 channels by 4 pixels, transposed in registers
};

template <int RS, int WK, int MODE>
__global__ __launch_bounds__(WINDOW_WAVES * 64) __attribute__((amdgpu_waves_per_eu(4))) void conv_window_kernel(WindowArgs)
{
    using std::integral_constant;
    constexpr int  NT = WINDOW_WAVES * 64, QS = 2, D = RS > 2 ? 2 : 3, WP = WINDOW_WAVES / 2 / WK, NPIX = RS * 16 * WP;
    constexpr bool PLANES = MODE == WINDOW_PLANES;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lh = lane >> 4, wn = wave & 1, wk = (wave >> 1) % WK, wp = (wave >> 1) / WK;

    int       n, oy0, ox0, pan0, rows, cols, ns, kbp;
    v4i       fb[D][QS];
    global_i8 b_base;
    // B: this wave's two column blocks of a panel, K block kb (the image is padded to whole blocks of 256 columns)
    auto load_b = [&](int slot, int s)
    {
        const int kb = min(wk + s * WK, kbp - 1);
#pragma unroll
        for (int j = 0; j < QS; ++j)
            fb[slot][j] = *(const __attribute__((address_space(1))) v4i *)(b_base + (uint32_t)((j * kbp + kb) * 1024));
    };
    bool    sums;
    int     qflag;
    int32_t par_reg = 0;
    {
        // (one batch of scalar loads: see gemm_dma_kernel)
        WindowArgs          g;
        const WindowArgsPtr k = window_args();
        uintptr_t           u_src = (uintptr_t)k->src, u_b = (uintptr_t)k->B, u_cv = (uintptr_t)k->colvec, u_qp = (uintptr_t)k->qp, u_fl = (uintptr_t)k->qp_flag;
        g.qp_stride = k->qp_stride;
        g.H = k->H, g.W = k->W, g.C = k->C, g.OH = k->OH, g.OW = k->OW, g.sx = k->sx, g.sy = k->sy, g.pl = k->pl, g.pt = k->pt;
        g.nblocks = k->nblocks, g.groups = k->groups, g.ppw = k->ppw, g.th = k->th, g.tw = k->tw, g.ty = k->ty, g.tx = k->tx, g.u = k->u, g.wr = k->wr, g.wc = k->wc;
        g.magic_groups = k->magic_groups, g.magic_per = k->magic_per, g.magic_tx = k->magic_tx, g.row_len = k->row_len, g.rows_at_once = k->rows_at_once;
        g.magic_len = k->magic_len, g.magic_x = k->magic_x, g.flip = k->flip, g.pad_word = k->pad_word, g.rowsum_mul = k->rowsum_mul, g.K = k->K, g.kbp = k->kbp;
        asm volatile("" : "+s"(u_src), "+s"(u_b), "+s"(u_cv), "+s"(u_qp), "+s"(u_fl), "+s"(g.qp_stride), "+s"(g.H), "+s"(g.W), "+s"(g.C), "+s"(g.OH), "+s"(g.OW),
                     "+s"(g.sx), "+s"(g.sy), "+s"(g.pl), "+s"(g.pt), "+s"(g.nblocks), "+s"(g.groups), "+s"(g.ppw), "+s"(g.th), "+s"(g.tw), "+s"(g.ty), "+s"(g.tx));
        asm volatile("" : "+s"(g.u), "+s"(g.wr), "+s"(g.wc), "+s"(g.magic_groups), "+s"(g.magic_per), "+s"(g.magic_tx), "+s"(g.row_len), "+s"(g.rows_at_once),
                     "+s"(g.magic_len), "+s"(g.magic_x), "+s"(g.flip), "+s"(g.pad_word), "+s"(g.rowsum_mul), "+s"(g.K), "+s"(g.kbp));
        // the groups of panels of a tile one after the other on one die, whose L2 then holds the window
        int l = (int)blockIdx.x;
        if ((g.nblocks & 7) == 0)
            l = (l & 7) * (g.nblocks >> 3) + (l >> 3);
        const int tile = fast_div(l, g.magic_groups);
        n              = fast_div(tile, g.magic_per);
        const int in = tile - n * (g.ty * g.tx), by = fast_div(in, g.magic_tx), bx = in - by * g.tx;
        pan0 = (l - tile * g.groups) * g.ppw;
        oy0 = by * g.th, ox0 = bx * g.tw;
        rows = min(g.th, g.OH - oy0), cols = min(g.tw, g.OW - ox0);
        const int iy0 = oy0 * g.sy - g.pt, ix0 = ox0 * g.sx - g.pl;
        const int cpr = (g.C + 15) >> 4, nkb = (g.K + 63) >> 6;
        kbp    = g.kbp;
        ns     = (nkb - wk + WK - 1) / WK; // K blocks of this wave: wk, wk + WK ...
        b_base = (global_i8)u_b + (int64_t)(pan0 * 4 + wn * QS) * kbp * 1024 + lane * 16;
        sums   = g.rowsum_mul != 0;
        // the constants of the first panel, in front of everything that is waited for
        qflag = *(const __attribute__((address_space(4))) int32_t *)u_fl;
        if (tid < PAR_LOADS * 64)
            par_reg = tid < 64 ? ((global_i32)u_cv)[pan0 * WINDOW_PANEL + tid] : ((global_i32)u_qp)[(int64_t)(tid / 64 - 1) * g.qp_stride + pan0 * WINDOW_PANEL + tid % 64];
        int32_t *psum = nullptr;
        if (sums)
        {
            psum = (int32_t *)(smem + window_args()->psum_off);
            for (int i = tid; i < g.wr * g.wc; i += NT)
                psum[i] = 0;
            __syncthreads();
        }

        // ---- the window: a thread takes the same place of one row after the other ----
        const global_i8 img = (global_i8)u_src + (int64_t)n * (g.H * g.W * g.C);
        const int       rr = g.row_len <= NT ? fast_div(tid, g.magic_len) : 0;
        const int       row_pitch = g.wc * g.u * 16;
        if (rr < g.rows_at_once)
        {
            for (int j = tid - rr * g.row_len; j < g.row_len; j += NT)
            {
                if constexpr (!PLANES)
                {
                    constexpr int PB = MODE == WINDOW_PIECES16 ? 16 : 8;
                    using piece_t = std::conditional_t<PB == 16, v4i, v2i>;
                    using piece_any = std::conditional_t<PB == 16, v4i_any, v2i_any>;
                    const int      x = fast_div(j, g.magic_x), c = j - x * (cpr * (16 / PB)), ix = ix0 + x;
                    const bool     chan = PB == 16 || c * PB < g.C; // (added channels are zero, in the signed form)
                    const bool     okx = (unsigned)ix < (unsigned)g.W && chan;
                    const int      off = ix * g.C + c * PB, to = x * g.u * 16 + c * PB;
                    const uint32_t fill = chan ? g.pad_word ^ g.flip : 0u;
                    for (int r0 = rr; r0 < g.wr; r0 += 4 * g.rows_at_once)
                    {
                        piece_t v[4];
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                        {
                            const int r = r0 + t * g.rows_at_once, iy = iy0 + r;
                            v[t] = (piece_t)(int)fill;
                            if (okx && (unsigned)iy < (unsigned)g.H && r < g.wr)
                                v[t] = (piece_t)*(const __attribute__((address_space(1))) piece_any *)(img + (uint32_t)(iy * (g.W * g.C) + off)) ^ (int)g.flip;
                        }
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                        {
                            const int r = r0 + t * g.rows_at_once;
                            if (r < g.wr)
                            {
                                *(piece_t *)(smem + r * row_pitch + to) = v[t];
                                if (sums)
                                {
                                    int32_t sum = 0;
#pragma unroll
                                    for (int q = 0; q < PB / 4; ++q)
                                        sum = __builtin_amdgcn_sdot4(v[t][q], ONES4, sum, false);
                                    atomicAdd(psum + r * g.wc + x, sum);
                                }
                            }
                        }
                    }
                }
                else
                {
                    const int nq = (g.wc + 3) >> 2, gr = fast_div(j, g.magic_x), xq = j - gr * nq, ix = ix0 + xq * 4;
                    // the dword that holds the 4 pixels (inside the row: W >= 4), moved into place; what lies outside the row is padding
                    const int      from = min(max(ix, 0), g.W - 4), move = ix - from;
                    const uint32_t plane = (uint32_t)(g.H * g.W), pad = g.pad_word;
                    uint32_t       sel = 0;
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        sel |= ((unsigned)(ix + b) < (unsigned)g.W ? (uint32_t)(b + move) & 3u : 4u) << (8 * b);
                    const int       left_c = g.C - gr * 16; // channels of this piece that exist
                    const global_i8 p = img + (uint32_t)(gr * 16) * plane + (uint32_t)from;
                    for (int r = rr; r < g.wr; r += g.rows_at_once)
                    {
                        const int  iy = iy0 + r;
                        const bool in_y = (unsigned)iy < (unsigned)g.H;
                        const uint32_t at = (uint32_t)(min(max(iy, 0), g.H - 1) * g.W), s = in_y ? sel : 0x04040404u;
                        uint32_t   d[4][4], o[4][4];
#pragma unroll
                        for (int t = 0; t < 16; ++t)
                            d[t >> 2][t & 3] = (uint32_t)*(const __attribute__((address_space(1))) int_any *)(p + (at + (uint32_t)min(t, left_c - 1) * plane));
#pragma unroll
                        for (int t = 0; t < 16; ++t)
                            d[t >> 2][t & 3] = __builtin_amdgcn_perm(pad, d[t >> 2][t & 3], s) ^ g.flip;
                        if (left_c < 16) // (added channels are zero, in the signed form)
                        {
#pragma unroll
                            for (int t = 0; t < 16; ++t)
                                d[t >> 2][t & 3] = t < left_c ? d[t >> 2][t & 3] : 0u;
                        }
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            transpose4(d[t], o[t]);
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (xq * 4 + x < g.wc)
                            {
                                const v4i v = {(int)o[0][x], (int)o[1][x], (int)o[2][x], (int)o[3][x]};
                                *(v4i *)(smem + r * row_pitch + ((xq * 4 + x) * g.u + gr) * 16) = v;
                                if (sums)
                                    atomicAdd(psum + r * g.wc + xq * 4 + x, sum_bytes(v, 0));
                            }
                    }
                }
            }
        }
#pragma unroll
        for (int s = 0; s < D; ++s)
            load_b(s, s);

        // where the pieces of K lie in the window
        const WindowArgsPtr a = window_args();
        int32_t            *tab = (int32_t *)(smem + a->tab_off);
        for (int e = tid; e < (nkb + 2 * WK) * 4; e += NT)
        {
            const int tap = fast_div(e, a->magic_cpr), c0 = (e - tap * cpr) * 16, ky = fast_div(tap, a->magic_KW), kx = tap - ky * a->KW;
            tab[e] = e * 16 < a->K ? ((ky * a->dy * a->wc + kx * a->dx) * a->u) * 16 + c0 : 0;
        }
        if (tid < PAR_LOADS * 64)
            park_constant((int32_t *)(smem + a->par_off), tid, 64, par_reg, a->result_offset);
        __syncthreads();
        if (sums && tid < NPIX)
        {
            const int      p = min(tid, rows * a->tw - 1), py = fast_div(p, a->magic_tw), px = p - py * a->tw;
            const int32_t *from = psum + py * a->sy * a->wc + px * a->sx;
            int32_t        sum = 0;
            for (int ky = 0; ky < a->KH; ++ky)
                for (int kx = 0; kx < a->KW; ++kx)
                    sum += from[ky * a->dy * a->wc + kx * a->dx];
            ((int32_t *)(smem + a->rowv_off))[tid] = (int32_t)((uint32_t)a->rowsum_mul * (uint32_t)sum);
        }
    }

    const char    *pix[RS]; // the top-left tap of this lane's pixels
    const int32_t *tb;
    int            pan1, P;
    {
        const WindowArgsPtr a = window_args();
        P    = rows * a->tw; // (pixels of a tile narrower than tw are not stored)
        pan1 = min(a->panels, pan0 + a->ppw);
        tb   = (const int32_t *)(smem + a->tab_off) + wk * 4 + lh;
#pragma unroll
        for (int i = 0; i < RS; ++i)
        {
            const int p = min((wp * RS + i) * 16 + lr, P - 1), py = fast_div(p, a->magic_tw), px = p - py * a->tw;
            pix[i] = smem + (py * a->sy * a->wc + px * a->sx) * a->u * 16;
        }
    }
    for (int pan = pan0; pan < pan1; ++pan)
    {
        const int n0 = pan * WINDOW_PANEL;
        if (pan != pan0)
        {
            const WindowArgsPtr a = window_args();
            if (tid < PAR_LOADS * 64)
                park_constant((int32_t *)(smem + a->par_off), tid, 64,
                              tid < 64 ? ((global_i32)(uintptr_t)a->colvec)[n0 + tid] : ((global_i32)(uintptr_t)a->qp)[(int64_t)(tid / 64 - 1) * a->qp_stride + n0 + tid % 64],
                              a->result_offset);
        }
        v4i acc[RS][QS];
#pragma unroll
        for (int i = 0; i < RS; ++i)
#pragma unroll
            for (int j = 0; j < QS; ++j)
                acc[i][j] = (v4i){0, 0, 0, 0};
        v4i fa[2][RS];
        int off = tb[0], off_next = tb[WK * 4];
#pragma unroll
        for (int i = 0; i < RS; ++i)
            fa[0][i] = *(const v4i *)(pix[i] + off);
        // One K block: the matrix instructions of its operands, behind those of a block row the read of the next K block's
        auto block = [&](int s, auto slot_c)
        {
            constexpr int SLOT = decltype(slot_c)::value % D, CUR = decltype(slot_c)::value & 1;
            off      = off_next;
            off_next = tb[min(s + 2, ns) * (WK * 4)];
#pragma unroll
            for (int i = 0; i < RS; ++i)
            {
#pragma unroll
                for (int j = 0; j < QS; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[SLOT][j], fa[CUR][i], acc[i][j], 0, 0, 0);
                fa[CUR ^ 1][i] = *(const v4i *)(pix[i] + off);
                __builtin_amdgcn_sched_barrier(0);
            }
            load_b(SLOT, s + D);
            __builtin_amdgcn_sched_barrier(0);
        };
        // (2 D of them written out: the slots of B and the two sets of A come round together)
        int  s = 0;
        auto some = [&](auto first_c, auto check_c)
        {
            constexpr int  I = decltype(first_c)::value;
            constexpr bool CHECK = decltype(check_c)::value;
            if (!CHECK || s + I < ns)
                block(s + I, first_c);
            if (!CHECK || s + I + 1 < ns)
                block(s + I + 1, integral_constant<int, I + 1>{});
        };
        for (; s + 2 * D <= ns; s += 2 * D)
        {
            some(integral_constant<int, 0>{}, std::false_type{});
            some(integral_constant<int, 2>{}, std::false_type{});
            if constexpr (D == 3)
                some(integral_constant<int, 4>{}, std::false_type{});
        }
        some(integral_constant<int, 0>{}, std::true_type{});
        some(integral_constant<int, 2>{}, std::true_type{});
        if constexpr (D == 3)
            some(integral_constant<int, 4>{}, std::true_type{});
        // (behind a branch the compiler does not keep the distance between a matrix instruction and a read of its result)
        asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
        if (pan + 1 < pan1)
        {
            b_base += (uint32_t)(4 * kbp * 1024);
#pragma unroll
            for (int t = 0; t < D; ++t)
                load_b(t, t);
        }
        const WindowArgsPtr a = window_args();
        char *const         xch = smem + a->xch_off;

        // ---- the parts of K: of two waves each finishes one of the two column blocks, of four also half of the pixels ----
        constexpr int FR = WK == 4 ? RS / 2 : RS, FC = WK == 1 ? 2 : 1;
        static_assert(WK != 4 || RS % 2 == 0, "half of the pixels each");
        v4i fin[FR][FC];
        if constexpr (WK == 1)
        {
#pragma unroll
            for (int i = 0; i < RS; ++i)
#pragma unroll
                for (int j = 0; j < QS; ++j)
                    fin[i][j] = acc[i][j];
            __syncthreads(); // (the row terms)
        }
        else
        {
            constexpr int FAR = WK; // waves apart: the other half of K's parts
            v4i          *box = (v4i *)xch + wave * RS * 64 + lane, *from = (v4i *)xch + (wave ^ FAR) * RS * 64 + lane;
            v4i           sum[RS];
            const bool    high = (wk & (WK / 2)) != 0;
            if (high)
            {
#pragma unroll
                for (int i = 0; i < RS; ++i)
                    box[i * 64] = acc[i][0], sum[i] = acc[i][1];
            }
            else
            {
#pragma unroll
                for (int i = 0; i < RS; ++i)
                    box[i * 64] = acc[i][1], sum[i] = acc[i][0];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < RS; ++i)
                sum[i] += from[i * 64];
            if constexpr (WK == 2)
            {
#pragma unroll
                for (int i = 0; i < RS; ++i)
                    fin[i][0] = sum[i];
            }
            else
            {
                v4i *box2 = (v4i *)xch + (WINDOW_WAVES * RS + wave * FR) * 64 + lane, *from2 = (v4i *)xch + (WINDOW_WAVES * RS + (wave ^ 2) * FR) * 64 + lane;
                if (wk & 1)
                {
#pragma unroll
                    for (int i = 0; i < FR; ++i)
                        box2[i * 64] = sum[i], fin[i][0] = sum[FR + i];
                }
                else
                {
#pragma unroll
                    for (int i = 0; i < FR; ++i)
                        box2[i * 64] = sum[FR + i], fin[i][0] = sum[i];
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < FR; ++i)
                    fin[i][0] += from2[i * 64];
            }
            __syncthreads();
        }
        const int pix0 = (WK == 4 ? (wk & 1) * FR : wp * RS) * 16 + lr, col0 = wn * 32 + (WK == 1 ? 0 : WK == 2 ? wk : wk >> 1) * 16 + 4 * lh;
        // ---- requantised into LDS: pixels of 64 channels, or channels of NPIX pixels ----
        constexpr int CPITCH = NPIX + 16;
        int32_t       rv[FR];
#pragma unroll
        for (int i = 0; i < FR; ++i)
            rv[i] = 0;
        if (sums)
        {
#pragma unroll
            for (int i = 0; i < FR; ++i)
                rv[i] = ((const int32_t *)(smem + a->rowv_off))[pix0 + i * 16];
        }
        const int32_t *par = (const int32_t *)(smem + a->par_off);
        const int32_t  lo = a->lo, hi = a->hi, result_offset = a->result_offset;
        const pk16_t   lo16 = {(int16_t)lo, (int16_t)lo}, hi16 = {(int16_t)hi, (int16_t)hi};
        auto           each = [&](auto std_c)
        {
#pragma unroll
            for (int j = 0; j < FC; ++j)
            {
                const int c = col0 + j * 16;
                const v4i cv = *(const v4i *)(par + PAR_CV * 64 + c), m = *(const v4i *)(par + PAR_M * 64 + c);
                const v4i sm1 = *(const v4i *)(par + PAR_SM1 * 64 + c), add = *(const v4i *)(par + PAR_ADD * 64 + c);
#pragma unroll
                for (int i = 0; i < FR; ++i)
                {
                    int32_t  x[4];
                    uint32_t w = 0;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        x[t] = (int32_t)((uint32_t)fin[i][j][t] + (uint32_t)cv[t] + (uint32_t)rv[i]);
                    if constexpr (decltype(std_c)::value)
                        w = std_requant4(x, m, sm1, add, lo16, hi16);
                    else
                    {
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            w |= ((uint32_t)any_requant(x[t], m[t], sm1[t], result_offset, lo, hi) & 0xFFu) << (8 * t);
                    }
                    const int p = pix0 + i * 16;
                    if constexpr (PLANES)
                    {
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            xch[(c + t) * CPITCH + p] = (char)(w >> (8 * t));
                    }
                    else
                        *(uint32_t *)(xch + p * WINDOW_OPITCH + c) = w;
                }
            }
        };
        if (a->qp_std && qflag == 0)
            each(std::true_type{});
        else
            each(std::false_type{});
        __syncthreads();
        // ---- and out: W bytes per lane, on any byte; the last piece of a run moves back to end where the run does ----
        const int ncols = min(WINDOW_PANEL, a->N - n0);
        auto      piece = [&](const char *from, global_out to, auto bytes_c) // (LDS rows have 16 bytes to spare)
        {
            constexpr int   W = decltype(bytes_c)::value;
            const uint32_t  by = (uint32_t)(size_t)from & 3u;
            const uint32_t *w = (const uint32_t *)(from - by);
            if constexpr (W == 1)
                *to = *from;
            else if constexpr (W == 4)
                *(__attribute__((address_space(1))) int_any *)to = (int)__builtin_amdgcn_alignbyte(w[1], w[0], by);
            else
            {
                v4i v;
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    v[t] = (int)__builtin_amdgcn_alignbyte(w[t + 1], w[t], by);
                *(__attribute__((address_space(1))) v4i_any *)to = v;
            }
        };
        if constexpr (PLANES)
        {
            const bool       one = a->tx == 1; // rows follow one another: one run per channel
            const int        len = one ? P : cols, runs = one ? 1 : rows, plane = a->OH * a->OW;
            const global_out D0 = (global_out)(uintptr_t)a->D + ((int64_t)n * a->N + n0) * plane + (oy0 * a->OW + ox0);
            auto             leave = [&](auto bytes_c)
            {
                constexpr int  W = decltype(bytes_c)::value;
                const int      npc = (len + W - 1) / W, per = runs * npc, total = ncols * per;
                const uint32_t m_per = per == 1 ? 0u : 0xFFFFFFFFu / (uint32_t)per + 1u, m_npc = npc == 1 ? 0u : 0xFFFFFFFFu / (uint32_t)npc + 1u;
                for (int i = tid; i < total; i += NT)
                {
                    const int c = fast_div(i, m_per), t = i - c * per, r = fast_div(t, m_npc), at = min((t - r * npc) * W, len - W);
                    piece(xch + c * CPITCH + r * a->tw + at, D0 + ((int64_t)c * plane + r * a->OW + at), bytes_c);
                }
            };
            if (len >= 16)
                leave(integral_constant<int, 16>{});
            else if (len >= 4)
                leave(integral_constant<int, 4>{});
            else
                leave(integral_constant<int, 1>{});
        }
        else
        {
            const global_out D0 = (global_out)(uintptr_t)a->D + ((int64_t)(n * a->OH + oy0) * a->OW + ox0) * a->ldd + n0;
            auto             leave = [&](auto bytes_c)
            {
                constexpr int W = decltype(bytes_c)::value, LPP = 64 / W; // lanes per pixel
                for (int i = tid; i < P * LPP; i += NT)
                {
                    const int p = i / LPP, q = (i % LPP) * W, py = fast_div(p, a->magic_tw), px = p - py * a->tw;
                    if (q >= ncols || px >= cols)
                        continue;
                    const int at = min(q, ncols - W);
                    piece(xch + p * WINDOW_OPITCH + at, D0 + ((int64_t)(py * a->OW + px) * a->ldd + at), bytes_c);
                }
            };
            if (ncols >= 16)
                leave(integral_constant<int, 16>{});
            else if (ncols >= 4)
                leave(integral_constant<int, 4>{});
            else
                leave(integral_constant<int, 1>{});
        }
        if (pan + 1 < pan1)
            __syncthreads(); // (the next panel writes the constants and the exchange area)
    }
}

template <int MODE>
static const void *window_fn(int rs, int wk)
{
    switch (rs * 10 + wk)
    {
        case 21: return (const void *)conv_window_kernel<2, 1, MODE>;
        case 41: return (const void *)conv_window_kernel<4, 1, MODE>;
        case 22: return (const void *)conv_window_kernel<2, 2, MODE>;
        case 42: return (const void *)conv_window_kernel<4, 2, MODE>;
        case 24: return (const void *)conv_window_kernel<2, 4, MODE>;
        case 44: return (const void *)conv_window_kernel<4, 4, MODE>;
    }
    return nullptr;
}

// conv: the caller's geometry, pad_word the raw padding byte replicated; args.Bp: weights of taps of whole 16-byte pieces, packed in operand
// order with args.Kp bytes a column; rowsum_mul as for the other convolution kernels; planes != 0: NCHW on both sides
int conv_window_launch(const WindowPlan &p, bool flip_a, const GemmArgs &args, int batch, hipStream_t s)
{
    const ConvGeom &c  = args.conv;
    const EpiParams &e = args.epi;
    const int64_t K = conv_window_k(c);
    const bool planes = e.planes != 0;
    if (args.Kp % 64 != 0 || args.Kp < K || e.stage != 0 || e.rowvec != nullptr || e.accumulate || e.qp == nullptr || e.qp_flag == nullptr)
        return (int)hipErrorInvalidValue;
    auto magic = [](int64_t d) -> uint32_t { return d == 1 ? 0u : (uint32_t)(((uint64_t)1 << 32) / (uint64_t)d) + 1u; };
    const int  cpr = (c.C + 15) / 16, mode = planes ? WINDOW_PLANES : c.C % 16 == 0 ? WINDOW_PIECES16 : WINDOW_PIECES8;
    WindowArgs a{};
    a.src = args.A, a.B = args.Bp, a.D = (int8_t *)args.D;
    a.colvec = e.colvec, a.qp = e.qp, a.qp_flag = e.qp_flag, a.qp_stride = e.qp_stride;
    a.H = c.H, a.W = c.W, a.C = c.C, a.KH = c.KH, a.KW = c.KW, a.OH = c.OH, a.OW = c.OW, a.sx = c.stride_x, a.sy = c.stride_y;
    a.pl = c.pad_left, a.pt = c.pad_top, a.dx = c.dil_x, a.dy = c.dil_y;
    a.K = (int32_t)K, a.kbp = (int32_t)(args.Kp / 64), a.N = args.N, a.ldd = (int32_t)args.ldd;
    a.th = p.th, a.tw = p.tw, a.ty = p.ty, a.tx = p.tx, a.u = p.u, a.wr = p.wr, a.wc = p.wc;
    a.ppw = p.ppw, a.panels = p.panels, a.groups = (p.panels + p.ppw - 1) / p.ppw;
    a.nblocks = (int32_t)((int64_t)batch * p.ty * p.tx * a.groups);
    const int per_x = planes ? (p.wc + 3) / 4 : cpr * (mode == WINDOW_PIECES8 ? 2 : 1); // what a place in a row is divided by
    a.row_len       = planes ? per_x * cpr : per_x * p.wc;
    a.rows_at_once  = a.row_len <= WINDOW_WAVES * 64 ? WINDOW_WAVES * 64 / a.row_len : 1;
    a.magic_len = magic(a.row_len), a.magic_x = magic(per_x), a.magic_tw = magic(p.tw), a.magic_cpr = magic(cpr), a.magic_KW = magic(c.KW);
    a.magic_groups = magic(a.groups), a.magic_per = magic((int64_t)p.ty * p.tx), a.magic_tx = magic(p.tx);
    if ((int64_t)a.nblocks * std::max(a.groups, p.ty * p.tx) >= ((int64_t)1 << 32))
        return (int)hipErrorInvalidValue;
    a.flip = flip_a ? 0x80808080u : 0u, a.pad_word = c.pad_word;
    a.rowsum_mul = e.rowsum_mul, a.result_offset = e.result_offset, a.lo = e.lo, a.hi = e.hi, a.qp_std = e.qp_std;
    const int most = conv_window_pixels(p.rs, p.wk);
    a.xch_off = (int32_t)p.win_bytes, a.tab_off = a.xch_off + (int32_t)p.xch_bytes, a.par_off = a.tab_off + (int32_t)p.tab_bytes;
    a.rowv_off = a.par_off + PAR_ROWS * WINDOW_PANEL * 4, a.psum_off = a.rowv_off + most * 4;
    if (p.lds > WINDOW_MOST_LDS || (a.rowsum_mul != 0 && a.psum_off + (int64_t)p.wr * p.wc * 4 > p.lds))
        return (int)hipErrorInvalidValue;
    const void *fn = mode == WINDOW_PLANES ? window_fn<WINDOW_PLANES>(p.rs, p.wk) : mode == WINDOW_PIECES8 ? window_fn<WINDOW_PIECES8>(p.rs, p.wk) : window_fn<WINDOW_PIECES16>(p.rs, p.wk);
    if (fn == nullptr)
        return (int)hipErrorInvalidValue;
    static std::atomic<uint32_t> raised[3][5][5]; // (once per kernel and device)
    std::atomic<uint32_t>       &done = raised[mode][p.rs][p.wk];
    int                          dev  = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 32)
        return (int)hipErrorInvalidDevice;
    if ((done.load(std::memory_order_acquire) & (1u << dev)) == 0)
    {
        const hipError_t err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, WINDOW_MOST_LDS);
        if (err != hipSuccess)
            return (int)err;
        done.fetch_or(1u << dev, std::memory_order_release);
    }
    void *kargs[] = {&a};
    return (int)hipLaunchKernel(fn, dim3((unsigned)a.nblocks), dim3(WINDOW_WAVES * 64), kargs, (size_t)p.lds, s);
}
} // namespace mi355
