// Bandwidth-bound helper kernels of the quantized-GEMM path: B packing + column sums (prepare time), the A pre-pass
// (row sums / padded copy), the stand-alone output stage, explicit im2col, and a one-thread-per-output GEMM used only
// for cross-checking the matrix-core kernels.
#include "internal.hpp"

#include <algorithm>

namespace mi355
{
typedef int v4i __attribute__((ext_vector_type(4)));

static inline int launch_status()
{
    return (int)hipGetLastError();
}

// sum of the four int8 lanes of a dword
__device__ __forceinline__ int32_t sum4_i8(int32_t w)
{
    return __builtin_amdgcn_sdot4(w, 0x01010101, 0, false);
}

__global__ void fill_i32_kernel(int32_t *p, int32_t v, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}
int fill_i32_launch(int32_t *p, int32_t v, int64_t n, hipStream_t s)
{
    if (n <= 0)
        return 0;
    fill_i32_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(p, v, n);
    return launch_status();
}

// ---- split K: the partial products of `splits` K slices (S32 planes of M rows of ldp words, `plane` words apart) summed
// and put through the epilogue the fused kernel would have applied. One thread per 4 consecutive columns of a row.
// Same arithmetic as epilogue_store_t: the sum of the slices is the accumulator of the whole K
// (what CpuGemmLowpOffsetContributionOutputStageKernel, src/cpu/kernels/CpuGemmLowpOffsetContributionOutputStageKernel.cpp:
// 830-940, is handed by the matrix multiply before it).
template <int EPI>
__global__ __launch_bounds__(256) void splitk_finish_kernel(const int32_t *__restrict__ parts, int64_t plane, int ldp, int splits,
                                                            GemmArgs g)
{
    typedef int   v4i __attribute__((ext_vector_type(4)));
    const EpiParams &p  = g.epi;
    const int        n4 = (g.N + 3) / 4;
    const int64_t    t  = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)g.M * n4)
        return;
    const int i = (int)(t / n4), j0 = (int)(t % n4) * 4;
    v4i       acc = {0, 0, 0, 0};
    // (columns from N on hold whatever the allocation held: never used below. Four loads at a time: few threads read many
    // planes, and one load after the other is all latency)
    const int32_t *from = parts + (int64_t)i * ldp + j0;
    int            sl   = 0;
    for (; sl + 4 <= splits; sl += 4, from += 4 * plane)
    {
        const v4i p0 = *(const v4i *)from, p1 = *(const v4i *)(from + plane), p2 = *(const v4i *)(from + 2 * plane),
                  p3 = *(const v4i *)(from + 3 * plane);
        acc += (p0 + p1) + (p2 + p3);
    }
    for (; sl < splits; ++sl, from += plane)
        acc += *(const v4i *)from;
    const int32_t rv  = p.rowvec ? p.rowvec[i] : 0;
    const int64_t idx = (int64_t)i * g.ldd + j0;
    const bool    vec = p.vec_store && j0 + 3 < g.N;
    char         *D   = (char *)g.D;
    v4i           o   = {0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < 4; ++c)
    {
        const int j = j0 + c;
        if (j >= g.N)
            continue;
        const int32_t cv = p.colvec[j];
        if (EPI == EPI_FIXEDPOINT)
            o[c] = epi_fixedpoint(acc[c], cv, rv, p.mult ? p.mult[j] : p.mult_s, p.shift ? p.shift[j] : p.shift_s, p);
        else if (EPI == EPI_S32)
            o[c] = (int32_t)((uint32_t)acc[c] + (uint32_t)cv + (uint32_t)rv + (p.accumulate ? (uint32_t)((int32_t *)D)[idx + c] : 0u));
        else
            o[c] = __float_as_int(epi_f32(acc[c], (int32_t)((uint32_t)cv + (uint32_t)rv), p.bias_f32 ? p.bias_f32[j] : 0.f,
                                          p.bias_f32 != nullptr, p, p.accumulate ? ((float *)D)[idx + c] : 0.f));
    }
    if (EPI == EPI_FIXEDPOINT)
    {
        if (vec)
            *(uint32_t *)(D + idx) = ((uint32_t)o[0] & 0xFFu) | (((uint32_t)o[1] & 0xFFu) << 8) | (((uint32_t)o[2] & 0xFFu) << 16) |
                                     (((uint32_t)o[3] & 0xFFu) << 24);
        else
            for (int c = 0; c < 4 && j0 + c < g.N; ++c)
                D[idx + c] = (char)o[c];
    }
    else if (EPI == EPI_F32 && p.half_out)
    {
        typedef _Float16 v4h __attribute__((ext_vector_type(4)));
        const v4h        h = {(_Float16)__int_as_float(o[0]), (_Float16)__int_as_float(o[1]), (_Float16)__int_as_float(o[2]),
                              (_Float16)__int_as_float(o[3])};
        if (vec)
            *(v4h *)((_Float16 *)D + idx) = h;
        else
            for (int c = 0; c < 4 && j0 + c < g.N; ++c)
                ((_Float16 *)D)[idx + c] = h[c];
    }
    else
    {
        if (vec)
            *(v4i *)((int32_t *)D + idx) = o;
        else
            for (int c = 0; c < 4 && j0 + c < g.N; ++c)
                ((int32_t *)D)[idx + c] = o[c];
    }
}
int splitk_finish_launch(int epi, const GemmArgs &g, const int32_t *parts, int64_t plane, int ldp, int splits, hipStream_t s)
{
    if (g.M < 1 || g.N < 1 || splits < 1 || ldp % 4 != 0 || plane % 4 != 0 || ((uintptr_t)parts & 15) != 0 || g.epi.colvec == nullptr)
        return (int)hipErrorInvalidValue;
    const int64_t  n = (int64_t)g.M * ((g.N + 3) / 4);
    const unsigned blocks = (unsigned)((n + 255) / 256);
    if (epi == EPI_FIXEDPOINT)
        splitk_finish_kernel<EPI_FIXEDPOINT><<<dim3(blocks), dim3(256), 0, s>>>(parts, plane, ldp, splits, g);
    else if (epi == EPI_S32)
        splitk_finish_kernel<EPI_S32><<<dim3(blocks), dim3(256), 0, s>>>(parts, plane, ldp, splits, g);
    else if (epi == EPI_F32)
        splitk_finish_kernel<EPI_F32><<<dim3(blocks), dim3(256), 0, s>>>(parts, plane, ldp, splits, g);
    else
        return (int)hipErrorInvalidValue;
    return launch_status();
}

// ---- P1: B[K][ldb] -> packed B (K contiguous, optional sign flip, zero padding) + column sums + the per-column term -----
// Replaces pretranspose_B_array (src/cpu/operators/internal/CpuGemmAssemblyDispatch.cpp:594-617) / CpuGemmTranspose1xWKernel and
// CpuGemmLowpMatrixBReductionKernel (src/cpu/kernels/CpuGemmLowpMatrixReductionKernel.cpp:273-446) in one pass over B.
// kf > 1 re-orders K on the way: packed row k = a*kf + b (b < kf) is source row b*(K/kf) + a, which is what
// CpuConvertFullyConnectedWeightsKernel does to weights trained in the other data layout
// (src/cpu/kernels/CpuConvertFullyConnectedWeightsKernel.cpp:60-66,118-121 with kf = its _factor2).
__device__ __forceinline__ int k_source(int k, int K, int kf)
{
    return kf > 1 ? (k % kf) * (K / kf) + k / kf : k;
}

// colvec[j] = a_off*colsum[j] + a_off*b_off*K (+ bias[j]); the per-column part of the offset contribution, folded with the
// bias like arm_gemm's col_bias (src/core/NEON/kernels/arm_gemm/quantized.cpp:963-968). bias_copy keeps the bias for a later
// change of the offsets.
__device__ __forceinline__ void finish_column(const ColumnFinish &f, int Np, int b, int j, int32_t sum)
{
    f.colsum[(int64_t)b * Np + j] = sum;
    if (j >= f.N)
        return;
    uint32_t v = f.a_off * (uint32_t)sum + f.a_off * f.b_off * f.K;
    if (f.bias)
    {
        const int32_t x = f.bias[j];
        v += (uint32_t)x;
        if (b == 0 && f.bias_copy != f.bias)
            f.bias_copy[j] = x;
    }
    f.colvec[(int64_t)b * Np + j] = (int32_t)v;
}

// Where piece kc / 16 (16 bytes along K) of column n goes: K-contiguous rows, or the 1 KiB blocks of 16 columns x 64 k in the
// lane order in which the 16x16x64 matrix instruction reads its B operand (lane l: column l % 16, bytes 16 * (l / 16) ..
// + 16 of the k block), one block after the other along K
template <bool SKINNY>
__device__ __forceinline__ int64_t packed_offset(int n, int kc, int Kp)
{
    if (SKINNY)
        return ((int64_t)(n >> 4) * (Kp >> 6) + (kc >> 6)) * 1024 + (((kc >> 4) & 3) * 16 + (n & 15)) * 16;
    return (int64_t)n * Kp + kc;
}

// A workgroup packs 64 columns x a run of 128-deep K tiles of one batch entry. A thread fetches 8 columns of 4 rows (any
// alignment: the hardware takes unaligned 8-byte loads), turns each 4 x 4 block of bytes round in registers (8 byte
// permutes) and the tile leaves through LDS as whole 128-byte rows (piece c of column n lies at c ^ (n / 8), so that the
// dword writes of a wave spread over the banks). All batch entries go out in one launch, and where a workgroup walks the
// whole K (splits = 1) it finishes its columns' sums itself: packing a new B is one launch. Bound by HBM (1 byte read and
// 1 written per element). One byte per lane and load, an LDS tile of bytes and one atomic per column and tile took 17.8 us
// at 4096 x 4096, plus a second pass of 18 us into the streaming kernel's order; this form 11.5 + 6 us (sums) in either
// order. 32 entries of 512 x 128, prepare and run together: 338 us as three launches per entry, 15.2 us now.
template <bool SKINNY>
__global__ __launch_bounds__(256) void pack_b_kernel(const uint8_t *__restrict__ B, int64_t ldb, int64_t b_bs, int K, int N, int Kp,
                                                     int Np, uint32_t flip4, int kf, int tiles_per_split, int8_t *__restrict__ out,
                                                     int32_t *__restrict__ partial, ColumnFinish f)
{
    __shared__ v4i     tile[64 * 8];
    __shared__ int32_t csum[64];
    const int          b = blockIdx.z, n0 = blockIdx.x * 64, tid = threadIdx.x;
    const int          nq = tid & 7, kq = tid >> 3, n = n0 + nq * 8;
    B += (int64_t)b * b_bs;
    out += (int64_t)b * Np * Kp;
    if (tid < 64)
        csum[tid] = 0;
    const int kt0 = blockIdx.y * tiles_per_split, kt1 = min(kt0 + tiles_per_split, Kp / 128);
    int       row[2], piece[2];
    int32_t   sum[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 2; ++j)
    {
        const int idx = tid + 256 * j, blk = idx >> 6, lane = idx & 63;
        row[j]   = SKINNY ? (blk >> 1) * 16 + (lane & 15) : idx >> 3;
        piece[j] = SKINNY ? (blk & 1) * 4 + (lane >> 4) : idx & 7;
    }
    for (int kt = kt0; kt < kt1; ++kt)
    {
        const int k0 = kt * 128;
        uint32_t  w[4][2];
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int k = k0 + kq * 4 + r;
            w[r][0] = 0, w[r][1] = 0;
            if (k >= K || n >= N)
                continue;
            const uint8_t *p = B + (int64_t)k_source(k, K, kf) * ldb + n;
            if (n + 8 <= N)
            {
                __builtin_memcpy(w[r], p, 8);
                w[r][0] ^= flip4, w[r][1] ^= flip4;
            }
            else
                for (int t = 0; t < N - n; ++t)
                    w[r][t >> 2] |= (uint32_t)(uint8_t)(p[t] ^ (uint8_t)flip4) << (8 * (t & 3));
        }
        if (kt > kt0)
            __syncthreads(); // the tile before this one has left LDS
        uint32_t *lds = (uint32_t *)tile + (nq * 8) * 32 + (((kq >> 2) ^ nq) << 2) + (kq & 3);
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            const uint32_t lo01 = __builtin_amdgcn_perm(w[1][h], w[0][h], 0x05010400), hi01 = __builtin_amdgcn_perm(w[1][h], w[0][h], 0x07030602);
            const uint32_t lo23 = __builtin_amdgcn_perm(w[3][h], w[2][h], 0x05010400), hi23 = __builtin_amdgcn_perm(w[3][h], w[2][h], 0x07030602);
            lds[(h * 4 + 0) * 32] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100);
            lds[(h * 4 + 1) * 32] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302);
            lds[(h * 4 + 2) * 32] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100);
            lds[(h * 4 + 3) * 32] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            const v4i v = tile[row[j] * 8 + (piece[j] ^ ((row[j] >> 3) & 7))];
            *(v4i *)(out + packed_offset<SKINNY>(n0 + row[j], k0 + piece[j] * 16, Kp)) = v;
            sum[j] += sum4_i8(v.x) + sum4_i8(v.y) + sum4_i8(v.z) + sum4_i8(v.w);
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
        atomicAdd(&csum[row[j]], sum[j]);
    __syncthreads();
    if (tid >= 64)
        return;
    if (partial)
        partial[((int64_t)b * gridDim.y + blockIdx.y) * Np + n0 + tid] = csum[tid];
    else
        finish_column(f, Np, b, n0 + tid, csum[tid]);
}

// sums the K runs of pack_b_kernel
__global__ __launch_bounds__(256) void colsum_finish_kernel(const int32_t *__restrict__ partial, int splits, int Np, ColumnFinish f)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (j >= Np)
        return;
    int32_t sum = 0;
    for (int i = 0; i < splits; ++i)
        sum += partial[((int64_t)b * splits + i) * Np + j];
    finish_column(f, Np, b, j, sum);
}

// K runs of a packing launch: about four workgroups per compute unit (4096 x 4096: 16 runs of 2 tiles), none of them empty
int pack_b_splits(int Kp, int Np, int nb)
{
    const int64_t columns = (int64_t)(Np / 64) * nb, tiles = Kp / 128;
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>(tiles, 1024 / columns)), per = (tiles + want - 1) / want;
    return (int)((tiles + per - 1) / per);
}

int pack_b_launch(const void *B, int64_t ldb, int64_t b_bs, int nb, int K, int N, int Kp, int Np, bool flip, int kf, bool skinny, int splits,
                  int8_t *out, int32_t *partial, const ColumnFinish &f, hipStream_t s)
{
    if (Np % 64 || Kp % 128 || Np < N || Kp < K || nb < 1 || nb > 65535 || (kf > 1 && K % kf != 0))
        return (int)hipErrorInvalidValue;
    const int tiles = Kp / 128;
    if (splits < 1 || splits > tiles || (splits > 1 && partial == nullptr))
        return (int)hipErrorInvalidValue;
    const int  per = (tiles + splits - 1) / splits; // (a run that is left empty sums to zero)
    const dim3 grid(Np / 64, splits, nb), block(256);
    int32_t   *pt = splits > 1 ? partial : nullptr;
    if (skinny)
        pack_b_kernel<true><<<grid, block, 0, s>>>((const uint8_t *)B, ldb, b_bs, K, N, Kp, Np, flip ? 0x80808080u : 0u, kf, per, out, pt, f);
    else
        pack_b_kernel<false><<<grid, block, 0, s>>>((const uint8_t *)B, ldb, b_bs, K, N, Kp, Np, flip ? 0x80808080u : 0u, kf, per, out, pt, f);
    if (splits > 1)
        colsum_finish_kernel<<<dim3((Np + 255) / 256, nb), dim3(256), 0, s>>>(partial, splits, Np, f);
    return launch_status();
}

// B already K-contiguous: Bt[N][ldk] (convolution weights [OFM][KH*KW*C], the layout CpuWeightsReshapeKernel
// produces transposed: src/cpu/kernels/CpuWeightsReshapeKernel.cpp:150-166). One wave per packed row, so a row's sum needs
// no other wave.
template <bool SKINNY>
__global__ __launch_bounds__(256) void pack_bt_kernel(const uint8_t *__restrict__ Bt, int64_t ldk, int64_t b_bs, int K, int N, int Kp,
                                                      int Np, uint32_t flip4, int kf, int8_t *__restrict__ out, ColumnFinish f,
                                                      int8_t *__restrict__ operands)
{
    const int b = blockIdx.y, n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    out += (int64_t)b * Np * Kp;
    const uint8_t *row = Bt + (int64_t)b * b_bs + (int64_t)n * ldk;
    int32_t        s   = 0;
    for (int kc = lane * 16; kc < Kp; kc += 64 * 16)
    {
        uint32_t w[4] = {0, 0, 0, 0};
        if (n < N && kc + 16 <= K && kf <= 1)
        {
            __builtin_memcpy(w, row + kc, 16);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                w[t] ^= flip4;
        }
        else if (n < N)
        {
#pragma unroll
            for (int t = 0; t < 16; ++t)
                if (kc + t < K)
                    w[t >> 2] |= (uint32_t)(uint8_t)(row[k_source(kc + t, K, kf)] ^ (uint8_t)flip4) << (8 * (t & 3));
        }
        s += sum4_i8((int)w[0]) + sum4_i8((int)w[1]) + sum4_i8((int)w[2]) + sum4_i8((int)w[3]);
        *(v4i *)(out + packed_offset<SKINNY>(n, kc, Kp)) = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        if (!SKINNY && operands)
            *(v4i *)(operands + packed_offset<true>(n, kc, Kp)) = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        s += __shfl_xor(s, o);
    if (lane == 0)
        finish_column(f, Np, b, n, s);
}

int pack_bt_launch(const void *Bt, int64_t ldk, int64_t b_bs, int nb, int K, int N, int Kp, int Np, bool flip, int kf, bool skinny,
                   int8_t *out, const ColumnFinish &f, hipStream_t s, int8_t *operands)
{
    if (Np % 4 || Kp % 64 || (operands && (nb != 1 || skinny)) || Np < N || Kp < K || nb < 1 || nb > 65535 || (kf > 1 && K % kf != 0))
        return (int)hipErrorInvalidValue;
    const dim3 grid(Np / 4, nb), block(256);
    if (skinny)
        pack_bt_kernel<true><<<grid, block, 0, s>>>((const uint8_t *)Bt, ldk, b_bs, K, N, Kp, Np, flip ? 0x80808080u : 0u, kf, out, f, nullptr);
    else
        pack_bt_kernel<false><<<grid, block, 0, s>>>((const uint8_t *)Bt, ldk, b_bs, K, N, Kp, Np, flip ? 0x80808080u : 0u, kf, out, f, operands);
    return launch_status();
}

// Row sums of the patch matrix without the patch matrix: rowvec[m] = b_off * sum over the taps and channels of output
// pixel m of the (sign-normalised) source byte, the padding value where a tap lies outside the image - what
// CpuGemmLowpMatrixAReductionKernel computes from the im2col buffer
// (src/cpu/kernels/CpuGemmLowpMatrixReductionKernel.cpp:133-204). One thread per output pixel.
__global__ __launch_bounds__(256) void conv_rowsum_kernel(const uint8_t *__restrict__ src, ConvGeom g, int M, uint8_t flip,
                                                          uint32_t b_off, int32_t *__restrict__ rowvec)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M)
        return;
    const int     ox = m % g.OW, t = m / g.OW, oy = t % g.OH, n = t / g.OH;
    const int     pad = (int8_t)((g.pad_word & 0xFFu) ^ flip);
    const int64_t img = (int64_t)n * g.H * g.W * g.C;
    int32_t       sum = 0;
    for (int ky = 0; ky < g.KH; ++ky)
        for (int kx = 0; kx < g.KW; ++kx)
        {
            const int iy = oy * g.stride_y - g.pad_top + ky * g.dil_y, ix = ox * g.stride_x - g.pad_left + kx * g.dil_x;
            if (iy < 0 || iy >= g.H || ix < 0 || ix >= g.W)
            {
                sum += pad * g.C;
                continue;
            }
            const uint8_t *p = src + img + ((int64_t)iy * g.W + ix) * g.C;
            int            c = 0;
            if ((((uintptr_t)p) & 3) == 0)
                for (; c + 4 <= g.C; c += 4)
                {
                    const uint32_t w = *(const uint32_t *)(p + c) ^ (flip * 0x01010101u);
                    sum += (int8_t)(w & 0xFF) + (int8_t)((w >> 8) & 0xFF) + (int8_t)((w >> 16) & 0xFF) + (int8_t)(w >> 24);
                }
            for (; c < g.C; ++c)
                sum += (int8_t)(p[c] ^ flip);
        }
    rowvec[m] = (int32_t)(b_off * (uint32_t)sum);
}

// g.pad_word: the raw padding byte replicated
int conv_rowsum_launch(const void *src, const ConvGeom &g, int M, bool flip, int32_t b_off, int32_t *rowvec, hipStream_t s)
{
    conv_rowsum_kernel<<<dim3((M + 255) / 256), dim3(256), 0, s>>>((const uint8_t *)src, g, M, flip ? 0x80 : 0, (uint32_t)b_off,
                                                                  rowvec);
    return launch_status();
}

// The first `rows` (a multiple of 64) rows of Bp as the narrow kernel keeps them in LDS: rows of `chunks` 16-byte pieces of data plus
// NARROW_PAD_PIECES of padding, zero beyond Kp - the workgroups copy this image into LDS with plain linear transfers. The
// padding of a panel's 64 rows holds one more row of the patch, piece p in padding piece p % 2 of row p / 2: a one for
// every byte that counts in the row sums of A, zeros for channels from c_true of C on and for k from K on.
__global__ __launch_bounds__(256) void pack_b_narrow_kernel(const int8_t *__restrict__ Bp, int Kp, int chunks, int rows, int K, int C,
                                                            int c_true, int8_t *__restrict__ Bn)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    constexpr int PAD = NARROW_PAD_PIECES;
    if (idx >= rows * (chunks + PAD))
        return;
    const int r = idx / (chunks + PAD), c = idx - r * (chunks + PAD);
    v4i       v = {0, 0, 0, 0};
    if (c < chunks && c * 16 < Kp)
        v = *(const v4i *)(Bp + (int64_t)r * Kp + c * 16);
    else if (c >= chunks)
    {
        const int k0 = ((r & 63) * PAD + c - chunks) * 16;
#pragma unroll
        for (int t = 0; t < 16; ++t)
            if (k0 + t < K && (k0 + t) % C < c_true)
                v[t >> 2] |= 1 << (8 * (t & 3));
    }
    *(v4i *)(Bn + (int64_t)idx * 16) = v;
}

int pack_b_narrow_launch(const int8_t *Bp, int Kp, int Np, int chunks, int rows, int K, int C, int c_true, int8_t *Bn, hipStream_t s)
{
    if (Kp % 16 || rows < 64 || rows % 64 != 0 || Np < rows || chunks < 1 || C < 1)
        return (int)hipErrorInvalidValue;
    pack_b_narrow_kernel<<<dim3((rows * (chunks + NARROW_PAD_PIECES) + 255) / 256), dim3(256), 0, s>>>(Bp, Kp, chunks, rows, K, C, c_true, Bn);
    return launch_status();
}

// the per-column term again from the column sums that are there (new offsets), all batch entries in one launch
__global__ __launch_bounds__(256) void colvec_kernel(int Np, ColumnFinish f)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (j < f.N)
        finish_column(f, Np, b, j, f.colsum[(int64_t)b * Np + j]);
}

int colvec_launch(int Np, int nb, const ColumnFinish &f, hipStream_t s)
{
    if (nb < 1 || nb > 65535)
        return (int)hipErrorInvalidValue;
    colvec_kernel<<<dim3((f.N + 255) / 256, nb), dim3(256), 0, s>>>(Np, f);
    return launch_status();
}

// Digest (multiplier, shift) per column into the QP_* vectors of epilogue.hpp; *neg is set when a multiplier is negative
// (then the branch-free form does not apply). mult / shift may be nullptr: per-tensor values mult_s / shift_s.
__global__ void qparams_kernel(const int32_t *__restrict__ mult, const int32_t *__restrict__ shift, int32_t mult_s,
                               int32_t shift_s, int N, int Np, int32_t *__restrict__ qp, int32_t *__restrict__ neg)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= Np)
        return;
    int32_t m = 0, s = 0;
    if (j < N)
    {
        m = mult ? mult[j] : mult_s;
        s = shift ? shift[j] : shift_s;
    }
    if (m < 0)
        atomicOr(neg, 1);
    if (j < N && !(m >= 0x40000000 && s >= 2 && s <= STD_MAX_SHIFT))
        atomicOr(neg, 2); // not the common case (see std_requant)
    if (s >= 32 || s <= -32)
        m = 0, s = 0; // the reference arithmetic yields 0 for these
    qp[QP_M * (int64_t)Np + j]   = m;
    qp[QP_SM1 * (int64_t)Np + j] = s - 1;
}

int qparams_launch(const int32_t *mult, const int32_t *shift, int32_t mult_s, int32_t shift_s, int N, int Np,
                   int32_t *qp, int32_t *neg, hipStream_t s)
{
    int e = fill_i32_launch(neg, 0, 1, s);
    if (e)
        return e;
    qparams_kernel<<<dim3((Np + 255) / 256), dim3(256), 0, s>>>(mult, shift, mult_s, shift_s, N, Np, qp, neg);
    return launch_status();
}

// ---- A pre-pass -----------------------------------------------------------------------------------------------------
// One block per row. Optionally writes the row sign-flipped and zero-padded to Kp (for A whose rows are not 16-byte
// aligned), optionally reduces it: rowvec[i] = b_off * sum_k flip(A[i][k])
// (CpuGemmLowpMatrixAReductionKernel, src/cpu/kernels/CpuGemmLowpMatrixReductionKernel.cpp:133-204).
template <int VEC>
__global__ __launch_bounds__(256) void a_prepass_kernel(const uint8_t *__restrict__ A, int64_t lda, int64_t a_bs, int K, uint8_t flip,
                                                        int8_t *__restrict__ Ap, int Kp, int32_t *__restrict__ rowvec,
                                                        uint32_t b_off)
{
    // (grid: rows x batch entries; the copies and the sums of the entries lie one after the other)
    const int      row  = blockIdx.y * gridDim.x + blockIdx.x;
    const uint8_t *src  = A + (int64_t)blockIdx.y * a_bs + (int64_t)blockIdx.x * lda;
    const int      kmax = Ap ? Kp : K;
    int32_t        s    = 0;
    for (int k = threadIdx.x * VEC; k < kmax; k += 256 * VEC)
    {
        union
        {
            uint8_t  b[VEC];
            uint32_t w[VEC >= 4 ? VEC / 4 : 1];
        } u;
        if (k < K)
        {
            if (VEC == 1)
                u.b[0] = src[k] ^ flip;
            else
            {
#pragma unroll
                for (int t = 0; t < VEC / 4; ++t)
                    u.w[t] = *(const uint32_t *)(src + k + 4 * t) ^ (flip * 0x01010101u);
            }
        }
        else
        {
#pragma unroll
            for (int t = 0; t < (VEC >= 4 ? VEC / 4 : 1); ++t)
                u.w[t] = 0;
            if (VEC == 1)
                u.b[0] = 0;
        }
        if (VEC == 1)
            s += (int8_t)u.b[0];
        else
        {
#pragma unroll
            for (int t = 0; t < VEC / 4; ++t)
                s += sum4_i8((int32_t)u.w[t]);
        }
        if (Ap)
        {
            if (VEC == 1)
                Ap[(int64_t)row * Kp + k] = (int8_t)u.b[0];
            else
            {
#pragma unroll
                for (int t = 0; t < VEC / 4; ++t)
                    *(uint32_t *)(Ap + (int64_t)row * Kp + k + 4 * t) = u.w[t];
            }
        }
    }
    if (rowvec)
    {
        __shared__ int32_t part[4];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            s += __shfl_xor(s, o);
        if ((threadIdx.x & 63) == 0)
            part[threadIdx.x >> 6] = s;
        __syncthreads();
        if (threadIdx.x == 0)
            rowvec[row] = (int32_t)(b_off * (uint32_t)(part[0] + part[1] + part[2] + part[3]));
    }
}

int a_prepass_launch(const void *A, int64_t lda, int64_t a_bs, int batch, int M, int K, bool flip, int8_t *Ap, int Kp,
                     int32_t *rowvec, int32_t b_off, hipStream_t s)
{
    if (M <= 0 || batch <= 0)
        return 0;
    if (batch > 65535)
        return (int)hipErrorInvalidValue;
    const uintptr_t mix  = (uintptr_t)A | (uintptr_t)lda | (uintptr_t)K | (batch > 1 ? (uintptr_t)a_bs : 0);
    const uint8_t   f    = flip ? 0x80 : 0;
    const dim3      grid(M, batch), block(256);
    if ((mix & 15) == 0)
        a_prepass_kernel<16><<<grid, block, 0, s>>>((const uint8_t *)A, lda, a_bs, K, f, Ap, Kp, rowvec, (uint32_t)b_off);
    else if ((mix & 7) == 0)
        a_prepass_kernel<8><<<grid, block, 0, s>>>((const uint8_t *)A, lda, a_bs, K, f, Ap, Kp, rowvec, (uint32_t)b_off);
    else if ((mix & 3) == 0)
        a_prepass_kernel<4><<<grid, block, 0, s>>>((const uint8_t *)A, lda, a_bs, K, f, Ap, Kp, rowvec, (uint32_t)b_off);
    else
        a_prepass_kernel<1><<<grid, block, 0, s>>>((const uint8_t *)A, lda, a_bs, K, f, Ap, Kp, rowvec, (uint32_t)b_off);
    return launch_status();
}

// ---- K2: stand-alone output stage --------------------------------------------------------------------------------------
// CpuGemmLowpQuantizeDownInt32To{Int8,Uint8}ScaleByFixedPointKernel
// (src/cpu/kernels/CpuGemmLowpQuantizeDownInt32ToInt8ScaleByFixedPointKernel.cpp:79-181): 4 B read + 1 B written per element
template <bool VEC4>
__global__ __launch_bounds__(256) void output_stage_kernel(const int32_t *__restrict__ src, int64_t ld_src,
                                                           const int32_t *__restrict__ bias, int8_t *__restrict__ dst,
                                                           int64_t ld_dst, int M, int N, EpiParams p)
{
    const int     per_row = VEC4 ? N / 4 : N;
    const int64_t idx     = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)M * per_row)
        return;
    const int i = (int)(idx / per_row), q = (int)(idx % per_row);
    if (VEC4)
    {
        const int j = q * 4;
        v4i       v = *(const v4i *)(src + (int64_t)i * ld_src + j);
        v4i       b = {0, 0, 0, 0};
        if (bias)
            b = *(const v4i *)(bias + j);
        uint32_t out = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
        {
            const int32_t mu = p.mult ? p.mult[j + t] : p.mult_s;
            const int32_t sh = p.shift ? p.shift[j + t] : p.shift_s;
            out |= ((uint32_t)epi_fixedpoint(v[t], b[t], 0, mu, sh, p) & 0xFFu) << (8 * t);
        }
        *(uint32_t *)(dst + (int64_t)i * ld_dst + j) = out;
    }
    else
    {
        const int32_t mu = p.mult ? p.mult[q] : p.mult_s;
        const int32_t sh = p.shift ? p.shift[q] : p.shift_s;
        dst[(int64_t)i * ld_dst + q] =
            (int8_t)epi_fixedpoint(src[(int64_t)i * ld_src + q], bias ? bias[q] : 0, 0, mu, sh, p);
    }
}

// CpuGemmLowpQuantizeDownInt32ToInt16ScaleByFixedPointKernel
// (src/cpu/kernels/CpuGemmLowpQuantizeDownInt32ToInt16ScaleByFixedPointKernel.cpp:76-200): 4 B read + 2 B written per element
template <bool VEC4>
__global__ __launch_bounds__(256) void output_stage_s16_kernel(const int32_t *__restrict__ src, int64_t ld_src,
                                                               const int32_t *__restrict__ bias, int16_t *__restrict__ dst,
                                                               int64_t ld_dst, int M, int N, EpiParams p)
{
    const int     per_row = VEC4 ? N / 4 : N;
    const int64_t idx     = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)M * per_row)
        return;
    const int i = (int)(idx / per_row), q = (int)(idx % per_row);
    if (VEC4)
    {
        typedef short v4s __attribute__((ext_vector_type(4)));
        const int j = q * 4;
        v4i       v = *(const v4i *)(src + (int64_t)i * ld_src + j);
        v4i       b = {0, 0, 0, 0};
        if (bias)
            b = *(const v4i *)(bias + j);
        v4s o;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            o[t] = (short)requant_fixedpoint_s16((int32_t)((uint32_t)v[t] + (uint32_t)b[t]), p.mult_s, p.shift_s, p.lo, p.hi);
        *(v4s *)(dst + (int64_t)i * ld_dst + j) = o;
    }
    else
        dst[(int64_t)i * ld_dst + q] = (int16_t)requant_fixedpoint_s16(
            (int32_t)((uint32_t)src[(int64_t)i * ld_src + q] + (uint32_t)(bias ? bias[q] : 0)), p.mult_s, p.shift_s, p.lo, p.hi);
}

int output_stage_s16_launch(const int32_t *src, int64_t ld_src, const int32_t *bias, void *dst, int64_t ld_dst, int M,
                            int N, const EpiParams &epi, hipStream_t s)
{
    if (M <= 0 || N <= 0)
        return 0;
    const bool vec = (N % 4 == 0) && (ld_src % 4 == 0) && (ld_dst % 4 == 0) && (((uintptr_t)src & 15) == 0) &&
                     (((uintptr_t)dst & 7) == 0) && (bias == nullptr || ((uintptr_t)bias & 15) == 0);
    const int64_t total = (int64_t)M * (vec ? N / 4 : N);
    const dim3    grid((unsigned)((total + 255) / 256)), block(256);
    if (vec)
        output_stage_s16_kernel<true><<<grid, block, 0, s>>>(src, ld_src, bias, (int16_t *)dst, ld_dst, M, N, epi);
    else
        output_stage_s16_kernel<false><<<grid, block, 0, s>>>(src, ld_src, bias, (int16_t *)dst, ld_dst, M, N, epi);
    return launch_status();
}

int output_stage_launch(const int32_t *src, int64_t ld_src, const int32_t *bias, void *dst, int64_t ld_dst, int M,
                        int N, const EpiParams &epi, hipStream_t s)
{
    if (M <= 0 || N <= 0)
        return 0;
    const bool vec = (N % 4 == 0) && (ld_src % 4 == 0) && (ld_dst % 4 == 0) && (((uintptr_t)src & 15) == 0) &&
                     (((uintptr_t)dst & 3) == 0) && (bias == nullptr || ((uintptr_t)bias & 15) == 0);
    const int64_t total = (int64_t)M * (vec ? N / 4 : N);
    const dim3    grid((unsigned)((total + 255) / 256)), block(256);
    if (vec)
        output_stage_kernel<true><<<grid, block, 0, s>>>(src, ld_src, bias, (int8_t *)dst, ld_dst, M, N, epi);
    else
        output_stage_kernel<false><<<grid, block, 0, s>>>(src, ld_src, bias, (int8_t *)dst, ld_dst, M, N, epi);
    return launch_status();
}

// ---- explicit im2col (NHWC) ----------------------------------------------------------------------------------------------
// CpuIm2ColKernel / linearize_volume_nhwc (src/cpu/kernels/directconv2d/impl.h:148-220,307-389). Used when the implicit
// loader does not apply (channel count not a multiple of 16, asymmetric weights) and exported on its own.
template <int VEC>
__global__ __launch_bounds__(256) void im2col_nhwc_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst,
                                                          int64_t rows, ConvGeom g, int64_t ld_dst)
{
    const int     K    = g.KH * g.KW * g.C;
    const int     upr  = K / VEC; // units per row
    const int64_t idx  = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * upr)
        return;
    const int64_t m = idx / upr;
    const int     k = (int)(idx % upr) * VEC;
    const int     tap = k / g.C, c0 = k - tap * g.C;
    const int     ky = tap / g.KW, kx = tap - ky * g.KW;
    const int     ox = (int)(m % g.OW);
    const int64_t t  = m / g.OW;
    const int     oy = (int)(t % g.OH);
    const int64_t n  = t / g.OH;
    const int     iy = oy * g.stride_y - g.pad_top + ky * g.dil_y;
    const int     ix = ox * g.stride_x - g.pad_left + kx * g.dil_x;
    const bool    in = iy >= 0 && iy < g.H && ix >= 0 && ix < g.W;
    const uint8_t *s = src + ((n * g.H + iy) * g.W + ix) * g.C + c0;
    uint8_t       *d = dst + m * ld_dst + k;
    if (VEC == 16)
    {
        const int pw = (int)g.pad_word;
        v4i       v  = {pw, pw, pw, pw};
        if (in)
            v = *(const v4i *)s;
        *(v4i *)d = v;
    }
    else
        *d = in ? *s : (uint8_t)(g.pad_word & 0xFF);
}

int im2col_nhwc_launch(const void *src, void *dst, int batch, const ConvGeom &g, int64_t ld_dst, hipStream_t s)
{
    const int64_t rows = (int64_t)batch * g.OH * g.OW;
    const int     K    = g.KH * g.KW * g.C;
    if (rows <= 0 || K <= 0)
        return 0;
    const bool vec = (g.C % 16 == 0) && (((uintptr_t)src & 15) == 0) && (((uintptr_t)dst & 15) == 0) &&
                     (ld_dst % 16 == 0);
    const int64_t total = rows * (vec ? K / 16 : K);
    const dim3    grid((unsigned)((total + 255) / 256)), block(256);
    if (vec)
        im2col_nhwc_kernel<16><<<grid, block, 0, s>>>((const uint8_t *)src, (uint8_t *)dst, rows, g, ld_dst);
    else
        im2col_nhwc_kernel<1><<<grid, block, 0, s>>>((const uint8_t *)src, (uint8_t *)dst, rows, g, ld_dst);
    return launch_status();
}

// ---- matrix transpose of bytes or 32-bit words: [batch][R][C] -> [batch][C][R] --------------------------------------
// The NCHW <-> NHWC conversions around the NHWC convolution kernel (one image is a C x HW matrix of bytes, or of floats
// for the dequantised destination) and of NCHW weights ([OFM][C][KH*KW] -> [OFM][KH*KW][C]). 64 x 64 tiles through LDS
// so that reads and writes both run along rows.
template <typename T>
__global__ __launch_bounds__(256) void transpose_kernel(const T *__restrict__ src, T *__restrict__ dst, int R, int C)
{
    __shared__ T tile[64][65];
    const int64_t      base = (int64_t)blockIdx.z * R * C;
    const int          r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
    const int          tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll 4
    for (int y = ty; y < 64; y += 4)
        if (r0 + y < R && c0 + tx < C)
            tile[y][tx] = src[base + (int64_t)(r0 + y) * C + c0 + tx];
    __syncthreads();
#pragma unroll 4
    for (int y = ty; y < 64; y += 4)
        if (c0 + y < C && r0 + tx < R)
            dst[base + (int64_t)(c0 + y) * R + r0 + tx] = tile[tx][y];
}

// The same for bytes, TR x TC per workgroup: 16-byte loads and stores (unaligned where the row length asks for it), and
// 4 x 4 blocks turned round in registers, so that nothing moves byte by byte. A thread owns 16 rows x 4 columns between
// LDS and the stores; TR / 16 threads of neighbouring row blocks write up to TR contiguous bytes. The 16-byte pieces of LDS rows
// are swizzled with the row's 16-block (a read takes several blocks at once). Bounded by latency at the sizes of one layer.
// 32 x (128 x 784): 2.4 to 4 us each way, byte by byte 7 to 10.
template <int TR, int TC>
__global__ __launch_bounds__(256) void transpose_bytes_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int R, int C)
{
    static_assert(TR * TC == 256 * 64, "64 bytes per thread");
    typedef int v4i __attribute__((ext_vector_type(4)));
    typedef v4i v4i_any __attribute__((aligned(1)));
    typedef int int_any __attribute__((aligned(1)));
    constexpr int PIECES = TC / 16, BLOCKS = TR / 16, ROWS = 256 / PIECES; // rows per pass of loads
    __shared__ __attribute__((aligned(16))) uint32_t tile[TR * TC / 4];
    const uint8_t *in  = src + (int64_t)blockIdx.z * R * C;
    uint8_t       *out = dst + (int64_t)blockIdx.z * R * C;
    const int      r0 = blockIdx.y * TR, c0 = blockIdx.x * TC, tid = threadIdx.x;
    const int      lp = tid % PIECES, lrow = tid / PIECES, c = c0 + lp * 16;
    v4i            v[4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
    {
        const int r = r0 + p * ROWS + lrow;
        v[p]        = (v4i){0, 0, 0, 0};
        if (r < R && c < C)
        {
            const uint8_t *at = in + (int64_t)r * C + c;
            if (c + 16 <= C)
                v[p] = *(const v4i_any *)at;
            else
            {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                {
                    if (c + t * 4 + 4 <= C)
                        v[p][t] = *(const int_any *)(at + t * 4);
                    else
                        for (int q = 0; q < 3; ++q)
                            if (c + t * 4 + q < C)
                                v[p][t] |= (int)((uint32_t)at[t * 4 + q] << (8 * q));
                }
            }
        }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
    {
        const int r = p * ROWS + lrow;
        *(v4i *)&tile[r * (TC / 4) + (lp ^ ((r >> 4) % PIECES)) * 4] = v[p];
    }
    __syncthreads();
    const int ii = tid % BLOCKS, j = tid / BLOCKS; // rows 16 * ii .. + 15, columns 4 * j .. + 3
    const int rr = r0 + ii * 16;
    if (rr >= R || c0 + j * 4 >= C)
        return;
    uint32_t o[4][4]; // [column][dword of rows]
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        uint32_t w[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            w[t] = tile[(ii * 16 + q * 4 + t) * (TC / 4) + (j ^ ((ii % PIECES) * 4))];
        const uint32_t lo01 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
        o[0][q] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u), o[1][q] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
        o[2][q] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), o[3][q] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
    {
        if (c0 + j * 4 + t >= C)
            break;
        uint8_t *at = out + (int64_t)(c0 + j * 4 + t) * R + rr;
        if (rr + 16 <= R)
            *(v4i_any *)at = (v4i){(int)o[t][0], (int)o[t][1], (int)o[t][2], (int)o[t][3]};
        else
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                if (rr + q * 4 + 4 <= R)
                    *(int_any *)(at + q * 4) = (int)o[t][q];
                else
                    for (int b = 0; b < 3; ++b)
                        if (rr + q * 4 + b < R)
                            at[q * 4 + b] = (uint8_t)(o[t][q] >> (8 * b));
            }
        }
    }
}

int transpose_bytes_launch(const void *src, void *dst, int batch, int R, int C, hipStream_t s)
{
    if (batch <= 0 || R <= 0 || C <= 0)
        return 0;
    if (batch > 65535 || (R + 63) / 64 > 65535)
        return (int)hipErrorInvalidValue;
    // The tile follows the short side; below 16 a thread's 16 bytes would mostly be edge (weights of few taps): byte by byte.
    // NCHW convolutions, us: 32 x 28x28x128 -> 128, 3x3 31.8 -> 19.8; 1x1 23.7 -> 14.0; 4 x 112x112x64 -> 64, s2 22.5 -> 13.4;
    // 16 x 57x57x24 -> 40 (no side aligned) 23.0 -> 22.8.
    if (R >= 16 && C >= 16)
    {
        auto go = [&](auto kernel, int tr, int tc)
        {
            kernel<<<dim3((unsigned)((C + tc - 1) / tc), (unsigned)((R + tr - 1) / tr), (unsigned)batch), dim3(256), 0, s>>>((const uint8_t *)src,
                                                                                                                    (uint8_t *)dst, R, C);
        };
        if (R <= 64)
            go(transpose_bytes_kernel<64, 256>, 64, 256);
        else if (C <= 64)
            go(transpose_bytes_kernel<256, 64>, 256, 64);
        else
            go(transpose_bytes_kernel<128, 128>, 128, 128);
        return launch_status();
    }
    const dim3 grid((unsigned)((C + 63) / 64), (unsigned)((R + 63) / 64), (unsigned)batch), block(256);
    transpose_kernel<uint8_t><<<grid, block, 0, s>>>((const uint8_t *)src, (uint8_t *)dst, R, C);
    return launch_status();
}

int transpose_words_launch(const void *src, void *dst, int batch, int R, int C, hipStream_t s)
{
    if (batch <= 0 || R <= 0 || C <= 0)
        return 0;
    if (batch > 65535 || (R + 63) / 64 > 65535)
        return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)((C + 63) / 64), (unsigned)((R + 63) / 64), (unsigned)batch), block(256);
    transpose_kernel<uint32_t><<<grid, block, 0, s>>>((const uint32_t *)src, (uint32_t *)dst, R, C);
    return launch_status();
}

// ---- segment gather / scatter between two stride sets ------------------------------------------------------------------
// Segment (i1, i2, i3) of seg bytes lives at i1*st[0] + i2*st[1] + i3*st[2] on either side: tensors that carry padding
// (along the channel dimension, between rows, between planes or images; ITensorInfo::strides_in_bytes()) to dense and back.
__global__ __launch_bounds__(256) void restride_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst,
                                                       int64_t total, int seg, int64_t n1, int64_t n2, RestrideSteps ss,
                                                       RestrideSteps ds)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total)
        return;
    const int64_t sgm = idx / seg;
    const int     c   = (int)(idx - sgm * seg);
    const int64_t q1  = sgm / n1, i1 = sgm - q1 * n1;
    const int64_t i3 = q1 / n2, i2 = q1 - i3 * n2;
    dst[i1 * ds.st[0] + i2 * ds.st[1] + i3 * ds.st[2] + c] = src[i1 * ss.st[0] + i2 * ss.st[1] + i3 * ss.st[2] + c];
}

int restride_nd_launch(const void *src, void *dst, int seg, int64_t n1, int64_t n2, int64_t n3, const RestrideSteps &ss,
                       const RestrideSteps &ds, hipStream_t s)
{
    if (seg <= 0 || n1 <= 0 || n2 <= 0 || n3 <= 0)
        return 0;
    const int64_t total = n1 * n2 * n3 * seg;
    if ((total + 255) / 256 > 0x7FFFFFFF)
        return (int)hipErrorInvalidValue;
    restride_kernel<<<dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s>>>((const uint8_t *)src, (uint8_t *)dst, total,
                                                                                 seg, n1, n2, ss, ds);
    return launch_status();
}

int restride_launch(const void *src, void *dst, int64_t segments, int seg, int64_t src_stride, int64_t dst_stride,
                    hipStream_t s)
{
    return restride_nd_launch(src, dst, seg, segments, 1, 1, RestrideSteps{{src_stride, 0, 0}}, RestrideSteps{{dst_stride, 0, 0}}, s);
}

// ---- F16 destinations: [batch][M][N] halfs with row / batch strides <- the dense F32 matrix the GEMM kernels write --------
// Conversion to half rounds to nearest even (the reference's host-side half type is configured the same way,
// support/Half.h:33-34). Accumulating: the rounded half is added to the previous half as the reference's test oracle
// adds halfs (both widened, one float addition, rounded again; tests/validation/fixtures/GEMMLowpFixture.h:912-918),
// and the activation clamp follows the addition.
// Bounded by HBM and L2 (4 bytes read, 2 written per element). A thread takes V elements of a row at any alignment (the
// hardware takes vector accesses on any element), a workgroup a block of rows (256 / tx) x V * tx columns, tx the power of two
// that the row fills. One element per thread with two 64-bit divisions to find it took 7.0 us at 512 x 4096; V = 8: 4.5 us.
template <int V>
__global__ __launch_bounds__(256) void f32_to_f16_kernel(const float *__restrict__ f, _Float16 *__restrict__ h,
                                                         int64_t rows, int M, int N, int64_t ldh, int64_t h_batch_stride,
                                                         int log_tx, int accumulate, float act_min, float act_max)
{
    typedef float    v4f __attribute__((ext_vector_type(4)));
    typedef v4f      v4f_any __attribute__((aligned(4)));
    typedef _Float16 v8h __attribute__((ext_vector_type(8)));
    typedef v8h      v8h_any __attribute__((aligned(2)));
    const int64_t row = ((int64_t)blockIdx.x << (8 - log_tx)) + (threadIdx.x >> log_tx);
    if (row >= rows)
        return;
    const int64_t bz   = rows == M ? 0 : row / M;
    const float  *in   = f + row * N;
    _Float16     *out  = h + bz * h_batch_stride + (row - bz * M) * ldh;
    const int64_t step = ((int64_t)gridDim.y << log_tx) * V;
    for (int64_t j = (((int64_t)blockIdx.y << log_tx) + (threadIdx.x & ((1 << log_tx) - 1))) * V; j < N; j += step)
    {
        if constexpr (V == 1)
        {
            _Float16 v = (_Float16)in[j];
            if (accumulate)
                v = (_Float16)fminf(fmaxf((float)out[j] + (float)v, act_min), act_max);
            out[j] = v;
            continue;
        }
        const bool whole = j + 8 <= N;
        const int  left  = whole ? 8 : (int)(N - j);
        v8h        v     = {0, 0, 0, 0, 0, 0, 0, 0}, was = v;
        if (whole)
        {
            const v4f lo = *(const v4f_any *)(in + j), hi = *(const v4f_any *)(in + j + 4);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                v[t] = (_Float16)lo[t], v[t + 4] = (_Float16)hi[t];
            if (accumulate)
                was = *(const v8h_any *)(out + j);
        }
        else
        {
#pragma unroll
            for (int t = 0; t < 7; ++t)
                if (t < left)
                {
                    v[t] = (_Float16)in[j + t];
                    if (accumulate)
                        was[t] = out[j + t];
                }
        }
        if (accumulate)
        {
#pragma unroll
            for (int t = 0; t < 8; ++t)
                v[t] = (_Float16)fminf(fmaxf((float)was[t] + (float)v[t], act_min), act_max);
        }
        if (whole)
            *(v8h_any *)(out + j) = v;
        else
        {
#pragma unroll
            for (int t = 0; t < 7; ++t)
                if (t < left)
                    out[j + t] = v[t];
        }
    }
}

int f32_to_f16_launch(const float *dense_f32, void *half_matrix, int batch, int M, int N, int64_t ldh,
                      int64_t h_batch_stride, bool accumulate, float act_min, float act_max, hipStream_t s)
{
    const int64_t rows = (int64_t)batch * M;
    if (rows <= 0 || N <= 0)
        return 0;
    // 8 elements per thread from two waves per compute unit on. GEMM and rounding, us, 1 element -> 8: 2048 x 8192 106.9 -> 82.2,
    // 512 x 4096 23.9 -> 20.7, 64 x 4096 13.3 -> 13.2; below, 2048 x 65: 8.7 -> 9.0.
    const int     per   = rows * N >= 262144 ? 8 : 1;
    const int64_t units = ((int64_t)N + per - 1) / per;
    int log_tx = 0;
    while (log_tx < 8 && ((int64_t)1 << log_tx) < units)
        ++log_tx;
    const int64_t row_blocks = (rows + (256 >> log_tx) - 1) >> (8 - log_tx), col_blocks = std::min<int64_t>((units + (1 << log_tx) - 1) >> log_tx, 65535);
    if (row_blocks > 0x7FFFFFFF)
        return (int)hipErrorInvalidValue;
    const auto kernel = per == 8 ? f32_to_f16_kernel<8> : f32_to_f16_kernel<1>;
    kernel<<<dim3((unsigned)row_blocks, (unsigned)col_blocks), dim3(256), 0, s>>>(
        dense_f32, (_Float16 *)half_matrix, rows, M, N, ldh, h_batch_stride, log_tx, accumulate ? 1 : 0, act_min, act_max);
    return launch_status();
}

// ---- one thread per output: the plainest possible statement of the path, for cross-checking only ----------------------
template <int EPI>
__global__ __launch_bounds__(256) void simple_gemm_kernel(GemmArgs g, uint8_t flip)
{
    const int j = blockIdx.x * 16 + (threadIdx.x & 15);
    const int i = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int bz = blockIdx.z;
    if (i >= g.M || j >= g.N)
        return;
    const uint8_t *a = (const uint8_t *)g.A + (int64_t)bz * g.a_batch_stride + (int64_t)i * g.lda;
    const int8_t  *b = g.Bp + (int64_t)bz * g.bp_batch_stride + (int64_t)j * g.Kp;
    int32_t        acc = 0;
    for (int k = 0; k < g.K; ++k)
        acc += (int32_t)(int8_t)(a[k] ^ flip) * (int32_t)b[k];
    const EpiParams &p   = g.epi;
    const int32_t    cv  = p.colvec[(int64_t)bz * p.colvec_batch_stride + j];
    const int32_t    rv  = p.rowvec ? p.rowvec[(int64_t)bz * p.rowvec_batch_stride + i] : 0;
    const int64_t    idx = (int64_t)bz * g.d_batch_stride + (int64_t)i * g.ldd + j;
    if (EPI == EPI_S32)
        ((int32_t *)g.D)[idx] = (int32_t)((uint32_t)acc + (uint32_t)cv + (uint32_t)rv +
                                          (p.accumulate ? (uint32_t)((int32_t *)g.D)[idx] : 0u));
    else if (EPI == EPI_FIXEDPOINT)
        ((int8_t *)g.D)[idx] =
            (int8_t)epi_fixedpoint(acc, cv, rv, p.mult ? p.mult[j] : p.mult_s, p.shift ? p.shift[j] : p.shift_s, p);
    else
        ((float *)g.D)[idx] = epi_f32(acc, (int32_t)((uint32_t)cv + (uint32_t)rv), p.bias_f32 ? p.bias_f32[j] : 0.f,
                                      p.bias_f32 != nullptr, p, p.accumulate ? ((float *)g.D)[idx] : 0.f);
}

int simple_gemm_launch(int epi, bool flip_a, const GemmArgs &args, int batch, hipStream_t s)
{
    const dim3    grid((args.N + 15) / 16, (args.M + 15) / 16, batch), block(256);
    const uint8_t f = flip_a ? 0x80 : 0;
    if (epi == EPI_S32)
        simple_gemm_kernel<EPI_S32><<<grid, block, 0, s>>>(args, f);
    else if (epi == EPI_FIXEDPOINT)
        simple_gemm_kernel<EPI_FIXEDPOINT><<<grid, block, 0, s>>>(args, f);
    else
        simple_gemm_kernel<EPI_F32><<<grid, block, 0, s>>>(args, f);
    return launch_status();
}
// ---- runs of C bytes -> runs of Cp >= C bytes (the first C copied, the rest set to `fill`): pixels of an NHWC image or
// taps of OHWI weights whose channel count the 16-byte loaders cannot take, padded to the next multiple of 16. The
// channels added meet weights that are zero in the kernels' signed form, so they change no sum. One thread per
// 16 bytes of output.
__global__ __launch_bounds__(256) void channel_pad_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int64_t runs, int C,
                                                          int Cp, uint32_t fill)
{
    typedef int v4i __attribute__((ext_vector_type(4)));
    const int     per = Cp / 16;
    const int64_t t   = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= runs * per)
        return;
    const int64_t  r  = t / per;
    const int      c0 = (int)(t - r * per) * 16;
    const uint8_t *in = src + r * C + c0;
    uint32_t       w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        w[q] = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
        {
            const int c = c0 + q * 4 + b;
            w[q] |= (uint32_t)(c < C ? in[q * 4 + b] : (uint8_t)fill) << (8 * b);
        }
    }
    *(v4i *)(dst + r * Cp + c0) = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}
int channel_pad_launch(const void *src, void *dst, int64_t runs, int C, int Cp, uint8_t fill, hipStream_t s)
{
    if (runs <= 0)
        return 0;
    if (C < 1 || Cp < C || Cp % 16 != 0 || ((uintptr_t)dst & 15) != 0)
        return (int)hipErrorInvalidValue;
    const int64_t n = runs * (Cp / 16);
    if ((n + 255) / 256 > 0x7fffffff)
        return (int)hipErrorInvalidValue;
    channel_pad_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>((const uint8_t *)src, (uint8_t *)dst, runs, C, Cp, fill);
    return launch_status();
}

// ---- an NHWC image as patch rows: for every image row and output column the KW taps of C channels that lie side by side
// under the kernel window, Cr >= KW * C bytes (a multiple of 16) apart. A KH x KW convolution of C channels becomes one of
// KH x 1 over OW columns of KW * C channels. Bounded by the image it writes. One thread per 16 bytes: inside a row they are
// one unaligned load; at its ends the load is moved into the row and its bytes shifted back, `fill` where the row has none.
// Bytes from KW * C on hold whatever follows in the row and meet zero weights.
// 32 x 224 x 224 x 3 under 7 x 7, stride 2 (25.7 MB written): 9 us, as long as the copy of single pixels took that it replaces; the
// convolution behind it 44 -> 28 us.
__global__ __launch_bounds__(256) void patch_rows_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int row_bytes, int step,
                                                         int left, int per, uint32_t magic_per, int units, uint32_t blocks_per_row, uint32_t fill)
{
    typedef int v4i __attribute__((ext_vector_type(4)));
    typedef v4i v4i_any __attribute__((aligned(1)));
    const uint32_t row = blockIdx.x / blocks_per_row;
    const int      u   = (int)((blockIdx.x - row * blocks_per_row) * 256 + threadIdx.x);
    if (u >= units)
        return;
    const int      ox = fast_div(u, magic_per);
    const int      b  = ox * step - left + (u - ox * per) * 16; // first byte in the row
    const uint8_t *in = src + (int64_t)row * row_bytes;
    v4i            v;
    if (b >= 0 && b + 16 <= row_bytes)
        v = *(const v4i_any *)(in + b);
    else if (row_bytes >= 16)
    {
        const int               at = min(max(b, 0), row_bytes - 16), sh = b - at;
        const unsigned __int128 x = __builtin_bit_cast(unsigned __int128, (v4i)(*(const v4i_any *)(in + at))), ones = ~(unsigned __int128)0;
        const unsigned __int128 f = __builtin_bit_cast(unsigned __int128, (v4i){(int)fill, (int)fill, (int)fill, (int)fill});
        unsigned __int128       y = f;
        if (sh > 0 && sh < 16)
            y = (x >> (8 * sh)) | (f & ~(ones >> (8 * sh)));
        else if (sh < 0 && sh > -16)
            y = (x << (-8 * sh)) | (f & ~(ones << (-8 * sh)));
        v = __builtin_bit_cast(v4i, y);
    }
    else
    {
        uint32_t w[4];
        for (int q = 0; q < 4; ++q)
        {
            w[q] = 0;
            for (int t = 0; t < 4; ++t)
            {
                const int at = b + q * 4 + t;
                w[q] |= (at >= 0 && at < row_bytes ? (uint32_t)in[at] : (fill & 0xFFu)) << (8 * t);
            }
        }
        v = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
    *(v4i *)(dst + ((int64_t)row * units + u) * 16) = v;
}
// what the kernel's 32-bit arithmetic takes
bool patch_rows_fit(int64_t rows, int W, int C, int OW, int stride_x, int pad_left, int Cr)
{
    const int64_t units = (int64_t)OW * (Cr / 16), bpr = (units + 255) / 256;
    return rows >= 1 && W >= 1 && C >= 1 && OW >= 1 && Cr >= 16 && Cr % 16 == 0 && rows * bpr <= 0x7fffffff && units * 16 <= 0x7fffffff &&
           (int64_t)W * C <= 0x7fffffff && ((int64_t)OW * stride_x + pad_left) * C + Cr <= 0x7fffffff &&
           units * (Cr / 16) < ((int64_t)1 << 32);
}

int patch_rows_launch(const void *src, void *dst, int64_t rows, int W, int C, int OW, int stride_x, int pad_left, int Cr, uint8_t fill, hipStream_t s)
{
    if (!patch_rows_fit(rows, W, C, OW, stride_x, pad_left, Cr) || ((uintptr_t)dst & 15) != 0)
        return (int)hipErrorInvalidValue;
    const int64_t  units = (int64_t)OW * (Cr / 16), bpr = (units + 255) / 256;
    const int      per   = Cr / 16;
    const uint32_t magic = per == 1 ? 0u : (uint32_t)(((uint64_t)1 << 32) / (uint64_t)per) + 1u; // exact while units * per < 2^32
    patch_rows_kernel<<<dim3((unsigned)(rows * bpr)), dim3(256), 0, s>>>((const uint8_t *)src, (uint8_t *)dst, W * C, stride_x * C, pad_left * C, per,
                                                                         magic, (int)units, (uint32_t)bpr, 0x01010101u * fill);
    return launch_status();
}

} // namespace mi355
