// Pieces shared by the matrix-core GEMM kernels: LDS swizzle, tile -> workgroup mapping, accumulator epilogue.
#pragma once
#include <type_traits>
#include "internal.hpp"

namespace mi355
{
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
// Four dwords, or four halves, at an address of any alignment that their elements have (v4i_any: on any byte): gfx950 stores them with one
// instruction all the same
typedef int      v4i_any __attribute__((ext_vector_type(4), aligned(1)));
typedef int      int_any __attribute__((aligned(1)));
typedef int      v4i_word __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 v4h_half __attribute__((ext_vector_type(4), aligned(2)));

// LDS tiles are rows of CPR 16-byte columns. Column c of row r is stored at column c ^ swz(r). The LDS serves a 16-byte
// access 16 lanes (256 bytes, all 64 banks) per clock: 16 consecutive rows reading the same logical column must land in
// 16 different 16-byte bank groups. 16/CPR rows share one 256-byte span, so rows r and r + 16/CPR (same position in the
// span) get different rotations; a staging write (consecutive columns of consecutive rows) is conflict free as well.
template <int CPR>
__device__ __forceinline__ int swz(int row)
{
    return (row / (16 / CPR)) & (CPR - 1);
}

// Tile -> workgroup mapping. Workgroups are handed to the 8 XCDs round-robin and each XCD has its own L2: give every
// XCD a contiguous run of logical tile ids, and walk the tile grid in groups of GM row panels so that a run covers a
// compact GM x (run/GM) patch whose A and B panels are shared inside one L2.
__device__ __forceinline__ void tile_coords(int bid, int nblocks, int tiles_m, int tiles_n, int &tm, int &tn)
{
    int l = bid;
    if ((nblocks & 7) == 0)
        l = (bid & 7) * (nblocks >> 3) + (bid >> 3);
    const int GM      = 4;
    const int per_grp = GM * tiles_n;
    const int grp     = l / per_grp;
    const int first   = grp * GM;
    const int gsize   = min(tiles_m - first, GM);
    const int in_grp  = l - grp * per_grp;
    tm                = first + in_grp % gsize;
    tn                = in_grp / gsize;
}

// The same for a batch of GEMMs launched as one 1-D grid of batch * tiles_m * tiles_n workgroups: the logical ids run
// batch-major, so an XCD's contiguous run covers whole batch entries (their A and B are then fetched into one L2 only).
__device__ __forceinline__ void tile_coords_batched(int bid, int nblocks, int tiles_m, int tiles_n, int &bz, int &tm,
                                                    int &tn)
{
    int l = bid;
    if ((nblocks & 7) == 0)
        l = (bid & 7) * (nblocks >> 3) + (bid >> 3);
    const int tpb = tiles_m * tiles_n;
    bz            = l / tpb;
    l -= bz * tpb;
    const int GM      = 4;
    const int per_grp = GM * tiles_n;
    const int grp     = l / per_grp;
    const int first   = grp * GM;
    const int gsize   = min(tiles_m - first, GM);
    const int in_grp  = l - grp * per_grp;
    tm                = first + in_grp % gsize;
    tn                = in_grp / gsize;
}

// The same map with the two run-time divisors replaced by multiplications with host-computed reciprocals (every wave of
// every block walks this dependent scalar chain before it can do anything else) and the group size, 1 to 4, by shifts.
__device__ __forceinline__ void tile_coords_batched_fast(int bid, int nblocks, int tiles_m, int tiles_n, uint32_t magic_tiles,
                                                         uint32_t magic_group, int &bz, int &tm, int &tn)
{
    int l = bid;
    if ((nblocks & 7) == 0)
        l = (bid & 7) * (nblocks >> 3) + (bid >> 3);
    const int tpb = tiles_m * tiles_n;
    bz            = nblocks == tpb ? 0 : (int)__umulhi((uint32_t)l, magic_tiles);
    l -= bz * tpb;
    const int per_grp = 4 * tiles_n;
    const int grp     = (int)__umulhi((uint32_t)l, magic_group);
    const int first   = grp * 4;
    const int gsize   = min(tiles_m - first, 4);
    const int in_grp  = l - grp * per_grp;
    // in_grp < 4 * tiles_n: x / 3 == (x * 0xAAAB) >> 17 holds for x < 2^16
    tn = gsize == 4 ? in_grp >> 2 : gsize == 2 ? in_grp >> 1 : gsize == 1 ? in_grp : (int)(((uint32_t)in_grp * 0xAAABu) >> 17);
    tm = first + in_grp - tn * gsize;
}

// Row sums of A taken inside the pipelined kernels: a lane holds the 16-byte column lane/16 of row lane%16 of every
// operand block of A it reads; sums[f] collects the bytes of block row f over the whole K loop (sdot4 with ones). The four
// lanes of a row are added up here, the padding the loader flipped along with the data (K steps beyond K hold zeros;
// a flipped zero counts -128) is taken out, and the sum is scaled: sums[f] becomes the per-row term of output row
// f*16 + lane%16, in every lane of that row - the layout the epilogues above take their row terms in.
template <int RS>
__device__ __forceinline__ void finish_row_sums(int32_t (&sums)[RS], int32_t mul, int32_t flipped_pad_bytes)
{
#pragma unroll
    for (int f = 0; f < RS; ++f)
    {
        int32_t v = sums[f];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        sums[f] = (int32_t)((uint32_t)mul * (uint32_t)(v + 128 * flipped_pad_bytes));
    }
}
constexpr int32_t ONES4 = 0x01010101;
__device__ __forceinline__ int32_t sum_bytes(v4i x, int32_t acc, v4i ones = (v4i){ONES4, ONES4, ONES4, ONES4})
{
#pragma unroll
    for (int t = 0; t < 4; ++t)
        acc = __builtin_amdgcn_sdot4(x[t], ones[t], acc, false);
    return acc;
}
// a one in each of the first n of 16 bytes (n of any sign and size): what sum_bytes counts of a piece that is partly
// padding
__device__ __forceinline__ v4i first_bytes(int n)
{
    v4i m;
#pragma unroll
    for (int t = 0; t < 4; ++t)
    {
        const int r = min(max(n - 4 * t, 0), 4);
        m[t]        = r == 0 ? 0 : (int)((uint32_t)ONES4 >> (8 * (4 - r)));
    }
    return m;
}
// The same for the 16 bytes at k of a convolution's patch (k < K): a pixel's channels beyond c_true are padding of the
// channel count, and k from K on is nothing. Padded taps count: they hold the padding value, as in the patch matrix.
__device__ __forceinline__ v4i patch_bytes(const ConvGeom &c, int k, int K)
{
    const int c0 = k - fast_div(k, c.magic_C) * c.C;
    return first_bytes(k < K ? c.c_true - c0 : 0);
}

// Accumulator (fm, fn, r) of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32 of its 32 x 32 block.
// (row0, col0) is the wave's top-left output coordinate.
template <int EPI, int FM, int FN>
__device__ __forceinline__ void epilogue_store(const v16i (&acc)[FM][FN], const GemmArgs &g, int row0, int col0, int lane,
                                               int bz)
{
    const int        lr = lane & 31, lh = lane >> 5;
    const EpiParams &p      = g.epi;
    const int32_t   *colvec = p.colvec + (int64_t)bz * p.colvec_batch_stride;
    const int32_t   *rowvec = p.rowvec ? p.rowvec + (int64_t)bz * p.rowvec_batch_stride : nullptr;
    char            *D      = (char *)g.D;
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
    {
        const int  j  = col0 + fn * 32 + lr;
        const bool vj = j < g.N;
        int32_t    cv = 0, mu = p.mult_s, sh = p.shift_s;
        float      bf = 0.f;
        if (vj)
        {
            cv = colvec[j];
            if (EPI == EPI_FIXEDPOINT && p.mult)
            {
                mu = p.mult[j];
                sh = p.shift[j];
            }
            if (EPI == EPI_F32 && p.bias_f32)
                bf = p.bias_f32[j];
        }
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
        {
#pragma unroll
            for (int r = 0; r < 16; ++r)
            {
                const int i = row0 + fm * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                if (vj && i < g.M)
                {
                    const int32_t rv  = rowvec ? rowvec[i] : 0;
                    const int32_t a   = acc[fm][fn][r];
                    const int64_t idx = (int64_t)bz * g.d_batch_stride + (int64_t)i * g.ldd + j;
                    if (EPI == EPI_S32)
                        ((int32_t *)D)[idx] = (int32_t)((uint32_t)a + (uint32_t)cv + (uint32_t)rv +
                                                        (p.accumulate ? (uint32_t)((int32_t *)D)[idx] : 0u));
                    else if (EPI == EPI_FIXEDPOINT)
                        ((int8_t *)D)[idx] = (int8_t)epi_fixedpoint(a, cv, rv, mu, sh, p);
                    else
                        ((float *)D)[idx] = epi_f32(a, (int32_t)((uint32_t)cv + (uint32_t)rv), bf, p.bias_f32 != nullptr,
                                                    p, p.accumulate ? ((float *)D)[idx] : 0.f);
                }
            }
        }
    }
}
// Accumulators of the pipelined kernel: 16 x 16 blocks produced by v_mfma_i32_16x16x64_i8 with the B panel as the first
// matrix operand, i.e. transposed. A wave's sub-tile is RS row slots of 16 rows by QS column slots of 16 columns; lane l
// holds, for every (rs, qs), output row rs*16 + l%16 and the 4 consecutive output columns qs*16 + 4*(l/16) + {0..3}
// in the 4 registers of acc[rs][qs]: per-column parameters are read as 16-byte vectors and 4 results leave in one store.
// (row0, col0) is the wave's top-left output coordinate.
template <int EPI, int RS, int QS, bool PLANES = false>
__device__ __forceinline__ void epilogue_store_t(const v4i (&acc)[RS][QS], const GemmArgs &g, int row0, int col0,
                                                 int lane, int bz, const int32_t *rvk = nullptr, bool use_rvk = false)
{
    const int        lr = lane & 15, lh = lane >> 4;
    const EpiParams &p      = g.epi;
    const int32_t   *colvec = p.colvec + (int64_t)bz * p.colvec_batch_stride;
    const int32_t   *rowvec = p.rowvec ? p.rowvec + (int64_t)bz * p.rowvec_batch_stride : nullptr;
    char            *D      = (char *)g.D;
    int32_t          rv[RS];
#pragma unroll
    for (int rs = 0; rs < RS; ++rs)
    {
        const int i = row0 + rs * 16 + lr;
        rv[rs]      = use_rvk ? rvk[rs] : ((rowvec && i < g.M) ? rowvec[i] : 0);
    }
#pragma unroll
    for (int qs = 0; qs < QS; ++qs)
    {
        const int j0 = col0 + qs * 16 + 4 * lh; // first of 4 consecutive columns; inside the padded vectors
        const v4i cv = *(const v4i *)(colvec + j0);
        v4i       mu = {p.mult_s, p.mult_s, p.mult_s, p.mult_s};
        v4i       sh = {p.shift_s, p.shift_s, p.shift_s, p.shift_s};
        float     bf[4] = {0.f, 0.f, 0.f, 0.f};
        if (EPI == EPI_FIXEDPOINT && p.mult)
        {
            mu = *(const v4i *)(p.mult + j0);
            sh = *(const v4i *)(p.shift + j0);
        }
        if (EPI == EPI_F32 && p.bias_f32)
        {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (j0 + t < g.N)
                    bf[t] = p.bias_f32[j0 + t];
        }
#pragma unroll
        for (int rs = 0; rs < RS; ++rs)
        {
            const int i = row0 + rs * 16 + lr;
            if (i >= g.M || j0 >= g.N)
                continue;
            const int64_t idx = (int64_t)bz * g.d_batch_stride + (int64_t)i * g.ldd + j0;
            const bool    vec = p.vec_store && (j0 + 3 < g.N);
            if (EPI == EPI_FIXEDPOINT)
            {
                uint32_t packed = 0;
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    packed |= ((uint32_t)epi_fixedpoint(acc[rs][qs][t], cv[t], rv[rs], mu[t], sh[t], p) & 0xFFu) << (8 * t);
                if (PLANES)
                {
                    const int n = fast_div(fast_div(i, g.conv.magic_OW), g.conv.magic_OH);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (j0 + t < g.N)
                            D[((int64_t)n * g.N + j0 + t) * p.planes + i - n * p.planes] = (char)(packed >> (8 * t));
                }
                else if (vec)
                    *(uint32_t *)(D + idx) = packed;
                else
                {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (j0 + t < g.N)
                            D[idx + t] = (char)(packed >> (8 * t));
                }
            }
            else if (EPI == EPI_S32)
            {
                v4i o, prev = {0, 0, 0, 0};
                if (p.accumulate)
                {
                    if (vec)
                        prev = *(const v4i *)((int32_t *)D + idx);
                    else
                    {
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            if (j0 + t < g.N)
                                prev[t] = ((int32_t *)D)[idx + t];
                    }
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    o[t] = (int32_t)((uint32_t)acc[rs][qs][t] + (uint32_t)cv[t] + (uint32_t)rv[rs] + (uint32_t)prev[t]);
                if (vec)
                    *(v4i *)((int32_t *)D + idx) = o;
                else
                {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (j0 + t < g.N)
                            ((int32_t *)D)[idx + t] = o[t];
                }
            }
            else
            {
                typedef float v4f __attribute__((ext_vector_type(4)));
                v4f o, prev = {0.f, 0.f, 0.f, 0.f};
                if (p.accumulate)
                {
                    if (vec)
                        prev = *(const v4f *)((float *)D + idx);
                    else
                    {
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            if (j0 + t < g.N)
                                prev[t] = ((float *)D)[idx + t];
                    }
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    o[t] = epi_f32(acc[rs][qs][t], (int32_t)((uint32_t)cv[t] + (uint32_t)rv[rs]), bf[t], p.bias_f32 != nullptr, p,
                                   prev[t]);
                if (vec)
                    *(v4f *)((float *)D + idx) = o;
                else
                {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (j0 + t < g.N)
                            ((float *)D)[idx + t] = o[t];
                }
            }
        }
    }
}
// FIXEDPOINT epilogue of the narrow kernels for multipliers >= 0, straight to the destination. The block's per-column constants were staged in LDS
// as par[PAR_ROWS][BN]; col_in_tile is the wave's first
// column inside the block tile. Same accumulator layout as epilogue_store_t.
template <int RS, int QS, int BN>
__device__ __forceinline__ void epilogue_store_fast(const v4i (&acc)[RS][QS], const GemmArgs &g, const int32_t *par,
                                                    int row0, int col0, int col_in_tile, int lane, int bz,
                                                    const int32_t *rvk = nullptr, bool use_rvk = false)
{
    const int        lr = lane & 15, lh = lane >> 4;
    const EpiParams &p      = g.epi;
    const int32_t   *rowvec = p.rowvec ? p.rowvec + (int64_t)bz * p.rowvec_batch_stride : nullptr;
    char            *D      = (char *)g.D;
    int32_t          rv[RS];
#pragma unroll
    for (int rs = 0; rs < RS; ++rs)
    {
        const int i = row0 + rs * 16 + lr;
        rv[rs]      = use_rvk ? rvk[rs] : ((rowvec && i < g.M) ? rowvec[i] : 0);
    }
#pragma unroll
    for (int qs = 0; qs < QS; ++qs)
    {
        const int c  = col_in_tile + qs * 16 + 4 * lh;
        const int j0 = col0 + qs * 16 + 4 * lh;
        const v4i cv = *(const v4i *)(par + PAR_CV * BN + c), mu = *(const v4i *)(par + PAR_M * BN + c);
        const v4i sm1 = *(const v4i *)(par + PAR_SM1 * BN + c);
#pragma unroll
        for (int rs = 0; rs < RS; ++rs)
        {
            const int i = row0 + rs * 16 + lr;
            int32_t   o[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
            {
                const int32_t v = (int32_t)((uint32_t)acc[rs][qs][t] + (uint32_t)cv[t] + (uint32_t)rv[rs]);
                o[t]            = fast_requant(v, mu[t], sm1[t], p.result_offset, p.lo, p.hi);
            }
            // low bytes of o[0..3] -> one dword
            const uint32_t p01    = __builtin_amdgcn_perm((uint32_t)o[1], (uint32_t)o[0], 0x0c0c0400u);
            const uint32_t p23    = __builtin_amdgcn_perm((uint32_t)o[3], (uint32_t)o[2], 0x0c0c0400u);
            const uint32_t packed = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
            if (i >= g.M || j0 >= g.N)
                continue;
            const int64_t idx = (int64_t)bz * g.d_batch_stride + (int64_t)i * g.ldd + j0;
            if (p.vec_store && (j0 + 3 < g.N))
                *(uint32_t *)(D + idx) = packed;
            else
            {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (j0 + t < g.N)
                        D[idx + t] = (char)(packed >> (8 * t));
            }
        }
    }
}
// FIXEDPOINT epilogue of the pipelined kernel for multipliers >= 0. The block's per-column constants were staged in LDS
// as par[PAR_ROWS][BN]; col_in_tile is the wave's first
// column inside the block tile; accumulator layout as in epilogue_store_t. The packed 8-bit results of the whole BM x BN block
// tile are first laid out in LDS (row pitch BN + 16 bytes: the 64 dword writes of a wave instruction - 16 rows by 4 dwords - then
// hit 64 different banks) and then written row by row, so a wave instruction writes pieces of rows end to end instead of
// 16 (or 4 times 1) bytes of 16 different rows. All NW consumer waves of the block call this together; `barrier` is executed
// once between the two phases by every wave of the block. stage must not overlap par. ROWV: a per-row term exists and is added.
// PLANES (a convolution): laid out column by column instead, and written as runs of a plane's pixels (EpiParams::planes).
template <bool STD, bool ROWV, int RS, int QS, int BM, int BN, int NW, bool PLANES = false, typename Barrier>
__device__ __forceinline__ void epilogue_store_staged(const v4i (&acc)[RS][QS], const GemmArgs &g, const int32_t *par,
                                                      char *stage, int m0, int n0, int row_in_tile, int col_in_tile,
                                                      int wave, int lane, int bz, Barrier barrier,
                                                      const int32_t *rvk = nullptr, bool use_rvk = false)
{
    constexpr int    PITCH = PLANES ? BM + 16 : BN + 16;
    const int        lr = lane & 15, lh = lane >> 4;
    const EpiParams &p      = g.epi;
    const int32_t   *rowvec = p.rowvec ? p.rowvec + (int64_t)bz * p.rowvec_batch_stride : nullptr;
    int32_t          rv[RS];
    const pk16_t     lo16 = {(int16_t)p.lo, (int16_t)p.lo}, hi16 = {(int16_t)p.hi, (int16_t)p.hi};
#pragma unroll
    for (int rs = 0; rs < RS; ++rs)
    {
        const int i = m0 + row_in_tile + rs * 16 + lr;
        rv[rs]      = !ROWV ? 0 : (use_rvk ? rvk[rs] : ((rowvec && i < g.M) ? rowvec[i] : 0));
    }
#pragma unroll
    for (int qs = 0; qs < QS; ++qs)
    {
        const int c  = col_in_tile + qs * 16 + 4 * lh;
        const v4i cv = *(const v4i *)(par + PAR_CV * BN + c), mu = *(const v4i *)(par + PAR_M * BN + c);
        const v4i sm1 = *(const v4i *)(par + PAR_SM1 * BN + c);
        v4i       add = {0, 0, 0, 0};
        if (STD)
            add = *(const v4i *)(par + PAR_ADD * BN + c);
#pragma unroll
        for (int rs = 0; rs < RS; ++rs)
        {
            int32_t v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
                v[t] = ROWV ? (int32_t)((uint32_t)acc[rs][qs][t] + (uint32_t)cv[t] + (uint32_t)rv[rs]) : (int32_t)((uint32_t)acc[rs][qs][t] + (uint32_t)cv[t]);
            if constexpr (STD && !PLANES)
                *(uint32_t *)(stage + (row_in_tile + rs * 16 + lr) * PITCH + c) = std_requant4(v, mu, sm1, add, lo16, hi16);
            else
            {
                int32_t o[4];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    o[t] = STD ? std_requant(v[t], mu[t], sm1[t], add[t], p.lo, p.hi) : fast_requant(v[t], mu[t], sm1[t], p.result_offset, p.lo, p.hi);
                if constexpr (PLANES)
                {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        stage[(c + t) * PITCH + row_in_tile + rs * 16 + lr] = (char)o[t];
                }
                else
                {
                    const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)o[1], (uint32_t)o[0], 0x0c0c0400u);
                    const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)o[3], (uint32_t)o[2], 0x0c0c0400u);
                    *(uint32_t *)(stage + (row_in_tile + rs * 16 + lr) * PITCH + c) = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
                }
            }
        }
    }
    barrier();
    if constexpr (PLANES)
    {
        char *D     = (char *)g.D;
        auto  leave = [&](auto bytes_c)
        {
            constexpr int W = decltype(bytes_c)::value, TOTAL = BM * BN / W;
#pragma unroll
            for (int it = 0; it < (TOTAL + NW * 64 - 1) / (NW * 64); ++it)
            {
                const int at = (it * NW + wave) * 64 + lane, c = at / (BM / W), r = at % (BM / W) * W;
                const int i = m0 + r, j = n0 + c;
                if (i >= g.M || j >= g.N || (TOTAL % (NW * 64) != 0 && c >= BN))
                    continue;
                // (pieces of W pixels do not cross images: W divides the plane, M and i)
                const int   n  = fast_div(fast_div(i, g.conv.magic_OW), g.conv.magic_OH);
                char       *to = D + ((int64_t)n * g.N + j) * p.planes + i - n * p.planes;
                const char *from = stage + c * PITCH + r;
                if constexpr (W == 16)
                    __builtin_nontemporal_store(*(const v4i *)from, (v4i *)to);
                else if constexpr (W == 4)
                    *(int *)to = *(const int *)from;
                else
                    *to = *from;
            }
        };
        if (p.planes % 16 == 0 && ((uintptr_t)D & 15) == 0)
            leave(std::integral_constant<int, 16>{});
        else if (p.planes % 4 == 0 && ((uintptr_t)D & 3) == 0)
            leave(std::integral_constant<int, 4>{});
        else
            leave(std::integral_constant<int, 1>{});
        return;
    }
    // 16 bytes per lane whatever the destination's alignment (a store of 16 bytes may start on any byte): a wave instruction writes
    // pieces of rows end to end. In a tile on the right edge the last piece of a row moves back to end where the row does; the bytes
    // it shares with the piece before it are written twice, with the same values. A byte or a dword per lane where rows are not
    // aligned to 16 made the stores as many instructions as the tile has bytes per lane: 2048 x 4095 x 512 12.1 us, now 9.0, 4000 x 1001
    // x 64 6.9 and 5.1, 2774 x 2406 x 227 14.2 and 10.8. Rows on 16 bytes go past the caches (a write is exactly the output then);
    // others share cache lines with the next tile's, which the L2 has to put together.
    char *D    = (char *)g.D + (int64_t)bz * g.d_batch_stride;
    const int ncols = min(BN, g.N - n0);
    auto  leave = [&](auto bytes_c, auto edge_c, auto nt_c)
    {
        constexpr int  W    = decltype(bytes_c)::value;
        constexpr bool EDGE = decltype(edge_c)::value;
        constexpr int LPR = BN / W > 64 ? 64 : BN / W; // lanes per output row (or per 64 bytes of it)
        constexpr int PARTS = BN / W / LPR, RPI = 64 / LPR; // ... rows per wave instruction
        const int     rr = lane / LPR;
#pragma unroll
        for (int it = 0; it < (BM + NW * RPI - 1) / (NW * RPI); ++it)
        {
            const int r = (it * NW + wave) * RPI + rr;
            const int i = m0 + r;
#pragma unroll
            for (int part = 0; part < PARTS; ++part)
            {
                const int cc = part * LPR * W + (lane % LPR) * W;
                if (i >= g.M || (EDGE && cc >= ncols) || (BM % (NW * RPI) != 0 && r >= BM))
                    continue;
                const int   c0   = EDGE ? min(cc, ncols - W) : cc;
                char       *to   = D + (int64_t)i * g.ldd + n0 + c0;
                const char *from = stage + r * PITCH + c0;
                if constexpr (W == 16)
                {
                    v4i val;
                    if constexpr (EDGE)
                    {
                        const int      *w  = (const int *)(stage + r * PITCH + (c0 & ~3)); // (a fifth dword: the pitch has 16 bytes to spare)
                        const uint32_t  by = (uint32_t)c0 & 3u;
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            val[t] = (int)__builtin_amdgcn_alignbyte((uint32_t)w[t + 1], (uint32_t)w[t], by);
                    }
                    else
                        val = *(const v4i *)from;
                    if constexpr (decltype(nt_c)::value)
                        __builtin_nontemporal_store(val, (v4i *)to);
                    else
                        *(v4i_any *)to = val;
                }
                else if constexpr (W == 4)
                {
                    const uint32_t *w = (const uint32_t *)(stage + r * PITCH + (c0 & ~3));
                    *(int_any *)to    = (int)__builtin_amdgcn_alignbyte(w[1], w[0], (uint32_t)c0 & 3u);
                }
                else
                    *to = *from;
            }
        }
    };
    using yes = std::true_type;
    using no  = std::false_type;
    if (ncols == BN && p.vec_store16)
        leave(std::integral_constant<int, 16>{}, no{}, yes{});
    else if (ncols == BN)
        leave(std::integral_constant<int, 16>{}, no{}, no{});
    else if (ncols >= 16)
        leave(std::integral_constant<int, 16>{}, yes{}, no{});
    else if (ncols >= 4)
        leave(std::integral_constant<int, 4>{}, yes{}, no{});
    else
        leave(std::integral_constant<int, 1>{}, yes{}, no{});
}
// S32 / F32 results of one wave's (RS*16) x (QS*16) sub-tile, 16 rows at a time through a wave-private LDS area
// (16 rows, pitch QS*64 + 16 bytes) so that they leave as 16 bytes per lane along whole row segments of QS*64 bytes
// instead of 16-byte pieces of 16 different rows. Needs no synchronisation with other waves. Halves (EpiParams::half_out) are rounded
// on the way out: as a pass of its own behind a float workspace that was 5.0 of 21 us at 512 x 4096 x 4096.
template <int EPI, int RS, int QS>
__device__ __forceinline__ void epilogue_store_wave32(const v4i (&acc)[RS][QS], const GemmArgs &g, char *stage, int row0,
                                                      int col0, int lane, int bz, const int32_t *rvk = nullptr, bool use_rvk = false)
{
    static_assert(EPI == EPI_S32 || EPI == EPI_F32, "32-bit outputs only");
    constexpr int    PITCH = QS * 64 + 16;
    constexpr int    LPR   = QS * 4;   // lanes per output row segment
    constexpr int    RPI   = 64 / LPR; // rows per wave instruction
    static_assert(LPR <= 64 && 16 % RPI == 0, "wave tile width");
    const int        lr = lane & 15, lh = lane >> 4;
    const EpiParams &p      = g.epi;
    const int32_t   *colvec = p.colvec + (int64_t)bz * p.colvec_batch_stride;
    const int32_t   *rowvec = p.rowvec ? p.rowvec + (int64_t)bz * p.rowvec_batch_stride : nullptr;
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    const bool       half   = EPI == EPI_F32 && p.half_out, nt = p.vec_store;
    const int        esz    = half ? 2 : 4;
    char            *D      = (char *)g.D + (int64_t)bz * g.d_batch_stride * esz;
    const int        rr = lane / LPR, cc = lane % LPR;
    // Everything the loop below needs from global memory is fetched before its first store goes out: a wait for a load
    // issued after a store also waits for that store to reach memory, and one such wait per block of 16 x 16 outputs
    // made the epilogue as slow as its slowest store, sixteen times over.
    v4i     cvq[QS];
    float   bfq[QS][4];
    int32_t rvs[RS];
    const bool has_bias = EPI == EPI_F32 && p.bias_f32 != nullptr;
#pragma unroll
    for (int qs = 0; qs < QS; ++qs)
    {
        const int j0 = col0 + qs * 16 + 4 * lh; // inside the padded vectors
        cvq[qs]      = *(const v4i *)(colvec + j0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            bfq[qs][t] = (has_bias && j0 + t < g.N) ? p.bias_f32[j0 + t] : 0.f;
    }
#pragma unroll
    for (int rs = 0; rs < RS; ++rs)
    {
        const int i = row0 + rs * 16 + lr;
        rvs[rs]     = use_rvk ? rvk[rs] : ((rowvec && i < g.M) ? rowvec[i] : 0);
    }
    // The conditions that are the same for the whole launch (bias, offsets, second clamp) and for the whole tile (inside
    // the matrix or on its edge) are decided once, here, and the loop over the outputs is instantiated for each answer:
    // tested per output they cost about 25 vector instructions each, and with two consumer waves per SIMD that, not the
    // stores, set the length of the epilogue. Inside the matrix a store is a running row pointer and nothing else.
    const bool interior = __builtin_amdgcn_readfirstlane(row0) + RS * 16 <= g.M && __builtin_amdgcn_readfirstlane(col0) + QS * 16 <= g.N;
    auto tile = [&](auto bias_c, auto offs_c, auto twice_c, auto inside_c)
    {
        constexpr bool BIAS = decltype(bias_c)::value, OFFS = decltype(offs_c)::value, TWICE = decltype(twice_c)::value;
        constexpr bool INSIDE = decltype(inside_c)::value;
        // This lane's 4 columns: on the right edge the last ones of a row move back to end where the row does, and share columns with
        // the ones before, which both write with the same values. Rows may start on any element (see v4i_word)
        const int     ncols = INSIDE ? QS * 16 : min(QS * 16, __builtin_amdgcn_readfirstlane(g.N - col0));
        const bool    few   = !INSIDE && ncols < 4, mine = cc * 4 < ncols;
        const int     c0    = INSIDE ? cc * 4 : max(min(cc * 4, ncols - 4), 0);
        char         *dp   = D + ((int64_t)(row0 + rr) * g.ldd + col0 + c0) * esz; // ... of the first row
        const int64_t step = (int64_t)RPI * g.ldd * esz;
        const float   scale = p.scale, lo = p.act_min, hi = p.act_max;
#pragma unroll
        for (int rs = 0; rs < RS; ++rs)
        {
            const int32_t rv = rvs[rs];
#pragma unroll
            for (int qs = 0; qs < QS; ++qs)
            {
                const v4i cv = cvq[qs];
                v4i       o;
#pragma unroll
                for (int t = 0; t < 4; ++t)
                {
                    const int32_t off = (int32_t)((uint32_t)cv[t] + (uint32_t)rv);
                    if (EPI == EPI_S32)
                        o[t] = (int32_t)((uint32_t)acc[rs][qs][t] + (uint32_t)off);
                    else
                        o[t] = __float_as_int(epi_f32_static<BIAS, OFFS, TWICE>(acc[rs][qs][t], off, bfq[qs][t], scale, lo, hi));
                }
                *(v4i *)(stage + lr * PITCH + (qs * 16 + 4 * lh) * 4) = o;
            }
            if (!few)
            {
                // (all reads, then all stores, with no condition between them but the edge's own. With halves and last pieces of under 4
                // columns tested at every store and all of it written out, the float kernel of 256 x 128 tiles was 2.4 times as long:
                // 30 x 450 x 1008 x 1408 38.4 us, then 34.3. Rows that are not aligned to 16 bytes share cache lines between tiles and are
                // left to the L2: 47 x 678 x 734 x 24 to float 37.2 us one element per lane, 36 past the caches, 25.6 like this; 25 x
                // 320 x 977 x 23 17.0, 14.5 and 13.3)
                v4i val[16 / RPI];
#pragma unroll
                for (int it = 0; it < 16 / RPI; ++it)
                {
                    const char *from = stage + (it * RPI + rr) * PITCH + c0 * 4;
                    val[it]          = INSIDE ? *(const v4i *)from : (v4i)*(const v4i_word *)from;
                }
                const int  rows = mine ? g.M - (row0 + rs * 16 + rr) : 0;
                auto       leave = [&](auto half_c, auto nt_c)
                {
                    constexpr bool NT = decltype(nt_c)::value;
#pragma unroll
                    for (int it = 0; it < 16 / RPI; ++it)
                    {
                        if (INSIDE || it * RPI < rows)
                        {
                            if constexpr (decltype(half_c)::value)
                            {
                                const v4h h = {(_Float16)__int_as_float(val[it][0]), (_Float16)__int_as_float(val[it][1]),
                                               (_Float16)__int_as_float(val[it][2]), (_Float16)__int_as_float(val[it][3])};
                                if constexpr (NT)
                                    __builtin_nontemporal_store(h, (v4h_half *)dp);
                                else
                                    *(v4h_half *)dp = h;
                            }
                            else if constexpr (NT)
                                __builtin_nontemporal_store(val[it], (v4i_word *)dp);
                            else
                                *(v4i_word *)dp = val[it];
                        }
                        dp += step;
                    }
                };
                if (nt)
                {
                    if (half)
                        leave(std::true_type{}, std::true_type{});
                    else
                        leave(std::false_type{}, std::true_type{});
                }
                else if (half)
                    leave(std::true_type{}, std::false_type{});
                else
                    leave(std::false_type{}, std::false_type{});
            }
            else
            {
                // under 4 columns: one element per lane
                const int at = lane / 4, c = lane % 4;
                const int val = *(const int *)(stage + at * PITCH + c * 4);
                if (c < ncols && row0 + rs * 16 + at < g.M)
                {
                    char *to = D + ((int64_t)(row0 + rs * 16 + at) * g.ldd + col0 + c) * esz;
                    if (half)
                        *(_Float16 *)to = (_Float16)__int_as_float(val);
                    else
                        *(int32_t *)to = val;
                }
            }
        }
    };
    using yes = std::true_type;
    using no  = std::false_type;
    auto edge_or_not = [&](auto bias_c, auto offs_c, auto twice_c)
    {
        if (interior)
            tile(bias_c, offs_c, twice_c, yes{});
        else
            tile(bias_c, offs_c, twice_c, no{});
    };
    if (EPI == EPI_S32)
        edge_or_not(no{}, no{}, no{});
    else if (!p.has_offsets)
    {
        if (has_bias)
            edge_or_not(yes{}, no{}, no{});
        else
            edge_or_not(no{}, no{}, no{});
    }
    else if (p.act_twice)
    {
        if (has_bias)
            edge_or_not(yes{}, yes{}, yes{});
        else
            edge_or_not(no{}, yes{}, yes{});
    }
    else
    {
        if (has_bias)
            edge_or_not(yes{}, yes{}, no{});
        else
            edge_or_not(no{}, yes{}, no{});
    }
}
} // namespace mi355
