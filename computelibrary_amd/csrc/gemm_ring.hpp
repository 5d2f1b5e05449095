// K1 / K4, tiles of one workgroup whose waves all load and all multiply (the pipelined kernel's small and middle tiles and the
// implicit convolution; gemm_dma.hip holds the division into loading and multiplying waves that 256 x 128 tiles run).
//
// A stage of the ring is one K step of the tile, (BM + BN) x BK bytes, brought in by direct-to-LDS loads: 1 KiB units, dealt out to
// the waves in turn. Operand blocks go from LDS into one of two register sets, one sub-step (64 of K) ahead of the matrix
// instructions that use them. There is ONE barrier per K step, in front of the reads of the next stage's first sub-step: by
// then every wave has the last operands of this stage in registers, so behind the barrier the slot takes the loads of stage
// kt + NS - the whole ring is in flight. Loads and operand reads go out one at a time between the matrix instructions.
//
// KG = 1: 4 waves, 2 x 2. KG = 2: 8 waves in two such groups, each of which multiplies half of every K step's depth; their
// accumulators are added up behind the loop. That halves what a wave issues per step, which pays where the addresses of the
// loads are what a wave's time goes into: in convolutions (14x14x256 -> 256, 3x3, batch 32: 64 x 64 tiles of a 256-deep step
// 12.1 us with two groups).
//
// What bounds it: the loads. A compute unit takes a KiB to LDS every 16 to 18 clocks, so the 16, 24 and 32 KiB of a 64 x 64, 128 x 64
// and 128 x 128 step are 270, 410 and 540 of the 380, 660 and 850 clocks that one takes with one workgroup per compute unit. Operand reads
// keep the LDS busy 0.17 to 0.20 of the time and the matrix cores are 0.16 to 0.31 (counters: 128 x 4096 x 4096, 512 x 4096 x 4096,
// 2048 x 2048 x 2048); the rest is the barrier's wait for the last wave. With
// loading waves apart, two barriers a step and a wave of loads behind each, a step was 800 to 1000 clocks whatever the tile
// (128 x 4096 x 4096: 17.7 us in 128 x 64 tiles, now 8.8 in 64 x 64; 2048 x 2048 x 2048: 15.9 to 11.3; 14x14x256 -> 256: 15.2 to 12.1).
#pragma once
#include "direct_lds.hpp"

namespace mi355
{
enum : int
{
    RING_DENSE = 0, // dword-aligned rows of A
    RING_CONV  = 1, // implicit convolution
    RING_BYTES = 2  // rows of A on any byte
};

// One wave's loads of a stage: AU / 4 units of A behind BU / 4 units of B
template <int BM, int BN, int BK, int NS, int KG, int MODE>
struct RingLoader
{
    static constexpr int NW    = 4 * KG;
    static constexpr int CPR   = BK / 16;   // 16-byte columns per tile row
    static constexpr int RPU   = 1024 / BK; // tile rows per unit
    static constexpr int AU = BM / RPU, BU = BN / RPU;
    static constexpr int LA = AU / NW, LB = BU / NW; // this wave's units
    static constexpr int STAGE = (BM + BN) * BK, LDS = NS * STAGE + (MODE == RING_CONV ? 1024 : 0);
    static_assert(AU % NW == 0 && BU % NW == 0, "units are dealt out evenly");
    // (the swizzle of a unit's rows depends on u * RPU mod CPR only, and u = wave + 4 i keeps that)
    static_assert((CPR == 8 || CPR == 16) && (NW * RPU) % CPR == 0, "one column per lane for all units of a wave");

    const int8_t *a_base, *b_base, *fill16, *a_end;
    uint32_t      a_off[LA]; // dense: byte offset of the lane's row and column; convolution: of its pixel's top-left tap
    int           iy0[MODE == RING_CONV ? LA : 1], ix0[MODE == RING_CONV ? LA : 1];
    uint32_t      b_off;
    uint32_t      spare; // convolution: LDS address of 1 KiB that nothing reads
    uint32_t      lds0, b_unit; // b_unit: bytes of the packed B between two units of this wave
    int           c16, K, k_base, lane_id;
    int           row_c;     // convolution: bytes of an image row
    bool          never_out; // convolution: no tap of any pixel lies outside the image
    bool          tail_whole; // a last step that K ends in may be fetched whole
    ConvGeom      conv;
    v4i           pad; // convolution: the 16 bytes a tap outside the image reads

    __device__ __forceinline__ void init(const GemmArgs &g, int m0, int n0, int bz, int wave, int lane, uint32_t lds_base)
    {
        lds0 = lds_base + (uint32_t)wave * 1024u, lane_id = lane, spare = lds_base + NS * STAGE;
        K = g.K, fill16 = g.fill16, a_end = g.a_end;
        const int ur = lane / CPR;
        c16          = ((lane % CPR) ^ swz<CPR>(wave * RPU + ur)) * 16;
        b_base       = g.Bp + (int64_t)bz * g.bp_batch_stride + (int64_t)n0 * g.Kp + (int64_t)wave * RPU * g.Kp;
        b_off        = (uint32_t)ur * (uint32_t)g.Kp + (uint32_t)c16;
        b_unit       = (uint32_t)(NW * RPU) * (uint32_t)g.Kp;
        tail_whole   = g.lean_tail_bz >= 0 && !(bz == g.lean_tail_bz && m0 + BM >= g.M);
        if (MODE == RING_CONV)
        {
            conv   = g.conv;
            row_c  = conv.W * conv.C;
            pad    = (v4i){(int)conv.pad_word, (int)conv.pad_word, (int)conv.pad_word, (int)conv.pad_word};
            asm volatile("" : "+v"(pad)); // (stays in its registers)
            never_out = conv.pad_top == 0 && conv.pad_left == 0 && (conv.OH - 1) * conv.stride_y + (conv.KH - 1) * conv.dil_y < conv.H &&
                        (conv.OW - 1) * conv.stride_x + (conv.KW - 1) * conv.dil_x < conv.W;
            a_base = g.A + (int64_t)bz * g.a_batch_stride;
            k_base = bz * g.k_slice;
        }
        else
        {
            a_base = g.A + (int64_t)bz * g.a_batch_stride + (int64_t)m0 * g.lda;
            k_base = 0;
        }
#pragma unroll
        for (int i = 0; i < LA; ++i)
        {
            const int r = (wave + i * NW) * RPU + ur;
            if (MODE == RING_CONV)
            {
                const int gr = min(m0 + r, g.M - 1);
                const int t  = fast_div(gr, conv.magic_OW);
                const int ox = gr - t * conv.OW;
                const int n  = fast_div(t, conv.magic_OH);
                const int oy = t - n * conv.OH;
                iy0[i]       = oy * conv.stride_y - conv.pad_top;
                ix0[i]       = ox * conv.stride_x - conv.pad_left;
                a_off[i]     = (uint32_t)n * (uint32_t)(conv.H * conv.W * conv.C) + (uint32_t)((iy0[i] * conv.W + ix0[i]) * conv.C);
            }
            else // (rows beyond M re-read the last one: their results are never stored)
                a_off[i] = (uint32_t)min(r, g.M - 1 - m0) * (uint32_t)g.lda + (uint32_t)c16;
        }
    }

    // Where stage kt's loads come from and go to. `whole`: no column of the stage lies beyond K (or may be read anyway)
    struct Step
    {
        const int8_t *a_k, *b_k;
        uint32_t      dst, off, slot; // slot: LDS address of this lane's 16 bytes of the wave's first unit
        int           dy, dx, k0;
        bool          inside; // convolution: no lane's tap lies outside the image, whatever the tile
    };
    __device__ __forceinline__ bool whole(int kt) const { return MODE == RING_CONV || (kt + 1) * BK <= K || tail_whole; }
    __device__ __forceinline__ Step step(int kt, int slot) const
    {
        Step t;
        t.k0  = kt * BK;
        t.dst = lds0 + (uint32_t)slot * STAGE;
        t.a_k = MODE == RING_CONV ? a_base : a_base + t.k0;
        t.b_k = b_base + t.k0; // inside the zero-padded packed panel
        if (MODE == RING_CONV)
        {
            // one tap per lane and step: the lane's column is the same in every unit (24-bit factors: see conv_taps_ok)
            const int k   = k_base + t.k0 + c16;
            const int tap = (int)__umulhi((uint32_t)k, conv.magic_C) + (conv.magic_C ? 0 : k);
            const int c0  = k - (int)__umul24(tap, conv.C);
            const int ky  = (int)__umulhi((uint32_t)tap, conv.magic_KW) + (conv.magic_KW ? 0 : tap);
            const int kx  = tap - (int)__umul24(ky, conv.KW);
            t.dy = (int)__umul24(ky, conv.dil_y), t.dx = (int)__umul24(kx, conv.dil_x);
            t.off  = __umul24(t.dy, row_c) + __umul24(t.dx, conv.C) + c0;
            t.dy   = t.k0 + c16 < K ? t.dy : (1 << 30); // nothing beyond K
            t.slot = t.dst + (uint32_t)lane_id * 16u;
            t.inside = never_out && t.k0 + BK <= K;
        }
        return t;
    }
    // load i of this wave's LA + LB of a whole stage
    __device__ __forceinline__ void issue_one(const Step &t, int i) const
    {
        if (i >= LA)
            dma16s(t.b_k + (uint32_t)(i - LA) * (uint64_t)b_unit, b_off, t.dst, (AU + (i - LA) * NW) * 1024);
        else if (MODE == RING_CONV)
        {
            const uint32_t d = t.dst + (uint32_t)i * (NW * 1024u);
            // Where every lane's tap lies in the image the load goes out as it is. Else the other lanes write the padding to their
            // LDS slots themselves and the load goes out for the rest; where that is no lane at all it goes to the spare KiB
            // behind the ring: every wave's loads of a stage have to be the same number.
            uint64_t in = ~0ull;
            if (!t.inside)
                in = __builtin_amdgcn_ballot_w64((unsigned)(iy0[i] + t.dy) < (unsigned)conv.H) &
                     __builtin_amdgcn_ballot_w64((unsigned)(ix0[i] + t.dx) < (unsigned)conv.W);
            if (in == ~0ull)
                dma16s(t.a_k, a_off[i] + t.off, t.dst, i * (NW * 1024));
            else
                dma16s_or_pad(t.a_k, in ? a_off[i] + t.off : 0u, in ? d : spare, in ? in : ~0ull, ~in, t.slot, i * (NW * 1024), pad);
        }
        else
            dma16s(t.a_k, a_off[i], t.dst, i * (NW * 1024));
    }
    // all of a stage's
    __device__ __forceinline__ void issue(int kt, int slot) const
    {
        const Step t = step(kt, slot);
        if (whole(kt))
        {
#pragma unroll
            for (int i = 0; i < LA + LB; ++i)
                issue_one(t, i);
            return;
        }
        // Last K step. Columns at or beyond K read the fill bytes. A column that straddles K reads on into the next row
        // (those bytes meet the zero rows of the packed B) - except at the very end of A, where the lane fetches
        // just the valid bytes and writes its LDS slot itself.
        const int k = t.k0 + c16;
#pragma unroll
        for (int i = 0; i < LA; ++i)
        {
            const int8_t  *ptr = t.a_k + a_off[i];
            const uint32_t d   = t.dst + (uint32_t)i * (NW * 1024u);
            if (k >= K || ptr + 16 <= a_end)
                dma16(k < K ? ptr : fill16, d);
            else
            {
                const v4i v = load16_partial(ptr, K - k);
                *(__attribute__((address_space(3))) v4i *)(size_t)(d + (uint32_t)lane_id * 16u) = v;
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        }
#pragma unroll
        for (int i = LA; i < LA + LB; ++i)
            issue_one(t, i);
    }
};

// Rows of A that start on any byte, or whose sums have to stop inside a 16-byte column: direct-to-LDS loads cannot shift bytes,
// so A and B come into registers (compiler-visible loads) two stages ahead of their write to LDS and four ahead of their use. A
// lane loads the dwords that hold its 16 bytes - loads off a dword boundary are four times slower - and shifts them into
// place; bytes beyond K are zero. The copy that a pass in front would make (a_prepass_kernel: 3.3 us and more) is not needed.
template <int BM, int BN, int BK, int NS, int KG>
struct RingLoader<BM, BN, BK, NS, KG, RING_BYTES>
{
    static constexpr int NW = 4, CPR = BK / 16, RPU = 1024 / BK;
    static constexpr int AU = BM / RPU, BU = BN / RPU, LA = AU / NW, LB = BU / NW;
    static constexpr int STAGE = (BM + BN) * BK;
    static_assert(KG == 1 && BK == 128 && NS == 3, "built for this form");
    struct Step
    {
    };
    struct Set
    {
        v4i a[LA], b[LB];
        int x[LA]; // the dword behind the four of a[]
    };
    const int8_t *a_base, *b_base; // a_base: dword aligned
    uint32_t      a_off[LA], b_off, b_unit;
    int           shift[LA]; // bytes from a lane's first dword to its first byte
    uint32_t      flip;
    int           c16, K;
    char         *lds;

    __device__ __forceinline__ void init(const GemmArgs &g, int m0, int n0, int bz, int wave, int lane, char *smem, bool flip_a)
    {
        K = g.K, flip = flip_a ? 0x80808080u : 0u;
        const int ur = lane / CPR;
        c16          = ((lane % CPR) ^ swz<CPR>(wave * RPU + ur)) * 16;
        lds          = smem + wave * 1024 + lane * 16;
        b_base       = g.Bp + (int64_t)bz * g.bp_batch_stride + (int64_t)n0 * g.Kp + (int64_t)wave * RPU * g.Kp;
        b_off        = (uint32_t)ur * (uint32_t)g.Kp + (uint32_t)c16;
        b_unit       = (uint32_t)(NW * RPU) * (uint32_t)g.Kp;
        const int8_t  *a = g.A + (int64_t)bz * g.a_batch_stride + (int64_t)m0 * g.lda;
        const uint32_t e = (uint32_t)(uintptr_t)a & 3u;
        a_base           = a - e;
#pragma unroll
        for (int i = 0; i < LA; ++i)
        {
            // (rows beyond M re-read the last one: their results are never stored)
            const uint32_t at = e + (uint32_t)min((wave + i * NW) * RPU + ur, g.M - 1 - m0) * (uint32_t)g.lda;
            a_off[i]          = (at & ~3u) + (uint32_t)c16;
            shift[i]          = (int)(at & 3u);
        }
    }
    __device__ __forceinline__ void load(Set &s, int kt) const
    {
        const int8_t *a_k = a_base + kt * BK, *b_k = b_base + kt * BK;
        if ((kt + 1) * BK <= K)
        {
#pragma unroll
            for (int i = 0; i < LA; ++i)
            {
                // (aligned rows need no fifth dword: it may lie beyond A)
                s.a[i] = *(const v4i *)__builtin_assume_aligned(a_k + a_off[i], 4);
                s.x[i] = *(const int *)(a_k + a_off[i] + (shift[i] ? 16u : 0u));
            }
        }
        else
        {
            const int rem = min(max(K - kt * BK - c16, 0), 16); // of this lane's 16 bytes; every dword is read that holds one of them
#pragma unroll
            for (int i = 0; i < LA; ++i)
            {
                const int end = rem ? shift[i] + rem : 0;
#pragma unroll
                for (int t = 0; t < 5; ++t)
                {
                    int w = 0;
                    if (4 * t < end)
                        w = *(const int *)(a_k + a_off[i] + 4 * t);
                    if (t < 4)
                        s.a[i][t] = w;
                    else
                        s.x[i] = w;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < LB; ++i)
            s.b[i] = *(const v4i *)(b_k + (uint32_t)i * (uint64_t)b_unit + b_off);
    }
    // stage kt, loaded into s, to its ring slot
    __device__ __forceinline__ void store(const Set &s, int kt, int slot) const
    {
        char *dst = lds + slot * STAGE;
#pragma unroll
        for (int i = 0; i < LA; ++i)
        {
            v4i v;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                v[t] = (int)(__builtin_amdgcn_alignbyte((uint32_t)(t < 3 ? s.a[i][t < 3 ? t + 1 : 0] : s.x[i]), (uint32_t)s.a[i][t], (uint32_t)shift[i]) ^ flip);
            if ((kt + 1) * BK > K)
            {
                const int rem = K - kt * BK - c16;
#pragma unroll
                for (int t = 0; t < 4; ++t)
                {
                    const int n = min(max(rem - 4 * t, 0), 4);
                    v[t] &= n == 4 ? -1 : (1 << (8 * n)) - 1;
                }
            }
            *(v4i *)(dst + i * (NW * 1024)) = v;
        }
#pragma unroll
        for (int i = 0; i < LB; ++i)
            *(v4i *)(dst + (AU + i * NW) * 1024) = s.b[i];
    }
    // (no loads go out between the matrix instructions)
    __device__ __forceinline__ Step step(int, int) const { return {}; }
    __device__ __forceinline__ void issue_one(const Step &, int) const {}
    __device__ __forceinline__ void issue(int, int) const {}
};

template <typename Loader, int MODE>
struct ByteSet
{
    struct type
    {
    };
};
template <typename Loader>
struct ByteSet<Loader, RING_BYTES>
{
    using type = typename Loader::Set;
};

// K slices (GemmArgs::slices): the workgroups of a tile leave their sums in memory and count themselves in; the last one takes the counter
// back to zero, fetches the tile's sums and goes on to the epilogue. False for the others. Nobody waits for anybody. Up to JOIN_PLANES
// slices each has a place of its own, whose sums the last workgroup has in flight together; more of them add theirs up in one place,
// which the last one leaves zero (64 x 64 x 16384 as 8 slices 9.0 and 7.8 us, as 16 10.0 and 6.8; 256 x 256 x 8192 as 8 9.1 and 8.7; but 592 x 182 x 3856
// as 4 7.4 and 8.0, 500 x 500 x 5000 9.0 and 10.3: every addition is one to memory).
// All of it is of device scope, past the caches that dies do not share: when a wave's count of stores in flight is zero all can see
// them, so the barrier and the counter need no fence (a release fence writes back the whole L2).
// What it took the place of, a second launch over planes of sums, and this, us: 592 x 182 x 3856 9.3, 7.4 as 4 slices; 130 x 2048 x 4096 10.8, 8.9
// as 2; 48 x 548 x 3583 10.4, 7.6 as 6; 60 x 4096 x 11008 17.1, 16.1 as 4.
template <int RE, int QS, int NT>
__device__ __forceinline__ bool join_slices(v4i (&fin)[RE][QS], int32_t (&rfin)[RE], bool rowsum, const GemmArgs &g, int tile, int slice, int tid, int *flag)
{
    typedef unsigned long long                     u64;
    typedef __attribute__((address_space(1))) u64 *g64;
    typedef __attribute__((address_space(1))) int *g32;
    constexpr int SUMS = RE * QS * 2, ALL = SUMS + (RE + 1) / 2; // pairs of words of a thread: sums, then row terms
    constexpr int AT_ONCE = SUMS >= 32 ? 1 : 32 / SUMS;           // slices whose sums are in flight together
    const int     tiles = g.tiles_m * g.tiles_n;
    const bool    added = g.slices > JOIN_PLANES;
    auto          place = [&](int z) { return (g64)(uintptr_t)g.parts + ((int64_t)z * tiles + tile) * (ALL * NT) + tid; };
    auto          pair  = [](int lo, int hi) { return (u64)(uint32_t)lo | ((u64)(uint32_t)hi << 32); };
    // (one place: the words of a thread as single words, NT apart)
    const g32 sum_at = (g32)(uintptr_t)g.parts + (int64_t)tile * (ALL * 2 * NT) + tid;
    if (added)
    {
#pragma unroll
        for (int u = 0; u < SUMS * 2; ++u)
            __hip_atomic_fetch_add(sum_at + u * NT, fin[u / 4 / QS][u / 4 % QS][u % 4], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (rowsum)
#pragma unroll
            for (int i = 0; i < RE; ++i)
                __hip_atomic_fetch_add(sum_at + (SUMS * 2 + i) * NT, rfin[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    else
    {
        const g64 own = place(slice);
#pragma unroll
        for (int u = 0; u < SUMS; ++u)
            __hip_atomic_store(own + u * NT, pair(fin[u / 2 / QS][u / 2 % QS][u % 2 * 2], fin[u / 2 / QS][u / 2 % QS][u % 2 * 2 + 1]),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (rowsum)
#pragma unroll
            for (int i = 0; i < RE; i += 2)
                __hip_atomic_store(own + (SUMS + i / 2) * NT, pair(rfin[i], rfin[i + 1 < RE ? i + 1 : i]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const g32 count = (g32)(uintptr_t)g.arrived + tile;
    if (tid == 0)
        *flag = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g.slices - 1;
    __syncthreads();
    if (*flag == 0)
        return false;
    if (tid == 0)
        __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::: "memory");
    if (added)
    {
#pragma unroll
        for (int u = 0; u < SUMS * 2; ++u)
            fin[u / 4 / QS][u / 4 % QS][u % 4] = __hip_atomic_load(sum_at + u * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (rowsum)
#pragma unroll
            for (int i = 0; i < RE; ++i)
                rfin[i] = __hip_atomic_load(sum_at + (SUMS * 2 + i) * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int u = 0; u < SUMS * 2; ++u)
            __hip_atomic_store(sum_at + u * NT, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (rowsum)
#pragma unroll
            for (int i = 0; i < RE; ++i)
                __hip_atomic_store(sum_at + (SUMS * 2 + i) * NT, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads(); // the flag's place is the epilogue's
        return true;
    }
    for (int z0 = 1; z0 < g.slices; z0 += AT_ONCE)
    {
        u64 sums[AT_ONCE][SUMS], rows[AT_ONCE][(RE + 1) / 2];
#pragma unroll
        for (int y = 0; y < AT_ONCE; ++y)
        {
            const int z   = slice + z0 + y;
            const g64 its = place(z >= g.slices ? z - g.slices : z);
            if (z0 + y < g.slices)
            {
#pragma unroll
                for (int u = 0; u < SUMS; ++u)
                    sums[y][u] = __hip_atomic_load(its + u * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (rowsum)
#pragma unroll
                    for (int i = 0; i < (RE + 1) / 2; ++i)
                        rows[y][i] = __hip_atomic_load(its + (SUMS + i) * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
#pragma unroll
        for (int y = 0; y < AT_ONCE; ++y)
        {
            if (z0 + y < g.slices)
            {
#pragma unroll
                for (int u = 0; u < SUMS; ++u)
                {
                    fin[u / 2 / QS][u / 2 % QS][u % 2 * 2] += (int)(uint32_t)sums[y][u];
                    fin[u / 2 / QS][u / 2 % QS][u % 2 * 2 + 1] += (int)(uint32_t)(sums[y][u] >> 32);
                }
                if (rowsum)
#pragma unroll
                    for (int i = 0; i < RE; ++i)
                        rfin[i] += (int)(uint32_t)(rows[y][i / 2] >> (i % 2 * 32));
            }
        }
    }
    __syncthreads(); // the flag's place is the epilogue's
    return true;
}

template <int BM, int BN, int BK, int NS, int KG, int EPI, bool FLIP_A, int MODE>
__global__ __launch_bounds__(256 * KG) __attribute__((amdgpu_waves_per_eu(KG == 1 ? 2 : BM * BN <= 64 * 64 ? 4 : 2))) void gemm_ring_kernel(GemmArgs g_in)
{
    // What a workgroup needs before its first loads go out is read here, in one batch of scalar loads, and pinned in
    // registers (see gemm_dma_kernel)
    GemmArgs g = g_in;
    asm volatile(""
                 : "+s"(g.tiles_m), "+s"(g.tiles_n), "+s"(g.magic_tiles), "+s"(g.magic_group), "+s"(g.tile_magic_ok), "+s"(g.lda),
                   "+s"(g.a_batch_stride), "+s"(g.Kp), "+s"(g.bp_batch_stride), "+s"(g.M), "+s"(g.N), "+s"(g.K),
                   "+s"(g.epi.qp_stride), "+s"(g.epi.colvec_batch_stride), "+s"(g.nblocks), "+s"(g.k_slice));
    typedef const __attribute__((address_space(1))) int32_t *global_i32;
    uintptr_t u_cv = (uintptr_t)g.epi.colvec, u_qp = (uintptr_t)g.epi.qp, u_fl = (uintptr_t)g.epi.qp_flag;
    asm volatile("" : "+s"(u_cv), "+s"(u_qp), "+s"(u_fl));
    if (MODE == RING_CONV)
        asm volatile(""
                     : "+s"(g.conv.H), "+s"(g.conv.W), "+s"(g.conv.C), "+s"(g.conv.KW), "+s"(g.conv.OW), "+s"(g.conv.OH),
                       "+s"(g.conv.stride_x), "+s"(g.conv.stride_y), "+s"(g.conv.pad_left), "+s"(g.conv.pad_top), "+s"(g.conv.dil_x),
                       "+s"(g.conv.dil_y), "+s"(g.conv.magic_C), "+s"(g.conv.magic_KW), "+s"(g.conv.magic_OW), "+s"(g.conv.magic_OH));

    using Loader       = RingLoader<BM, BN, BK, NS, KG, MODE>;
    constexpr int NW = 4 * KG, CPR = BK / 16;
    constexpr int SUB = BK / 64 / KG; // sub-steps of a K step per wave: wave group kg takes the sub-steps kg, kg + 2 ...
    constexpr int LPW   = Loader::LA + Loader::LB;      // loads per wave and stage
    constexpr int STAGE = Loader::STAGE;
    constexpr int TM = BM / 2, TN = BN / 2;
    constexpr int RS = TM / 16, QS = TN / 16;
    constexpr int NM = RS * QS, NR = RS + QS; // matrix instructions / operand reads per sub-step
    static_assert(SUB == 1 || SUB == 2, "sub-steps per wave");
    static_assert((NS - 1) * LPW < 64 && NS >= 2, "vmcnt range");
    static_assert(NM >= NR, "an operand read behind each of the first matrix instructions");
    constexpr int RE = RS / KG; // row blocks a wave finishes: the two groups add their accumulators up crosswise
    static_assert(RS % KG == 0, "half of the row blocks each");
    static_assert(NW * 16 * (QS * 64 + 16) <= NS * STAGE, "the 32-bit epilogue stages through the ring's memory");
    static_assert(KG == 1 || NW * RE * QS * 1024 + NW * RE * 256 <= NS * STAGE, "the exchange of accumulators fits the ring's memory");

    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
    const int      tid  = threadIdx.x;
    const int      lane = tid & 63;
    const int      wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    int tm, tn, bz;
    if (g.tile_magic_ok)
        tile_coords_batched_fast(blockIdx.x, g.nblocks, g.tiles_m, g.tiles_n, g.magic_tiles, g.magic_group, bz, tm, tn);
    else
        tile_coords_batched(blockIdx.x, g.nblocks, g.tiles_m, g.tiles_n, bz, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    if (g.k_slice != 0) // K slices: this entry's part of K (the last one ends where K does)
        g.K = min(g.k_slice, g.K - bz * g.k_slice);
    const int nk = (g.K + BK - 1) / BK;
    int       qflag = 1;
    if (EPI == EPI_FIXEDPOINT && u_fl != 0)
        qflag = *(const __attribute__((address_space(4))) int32_t *)u_fl;

    Loader ld;
    if constexpr (MODE == RING_BYTES)
        ld.init(g, m0, n0, bz, wave, lane, smem, FLIP_A);
    else
    {
        ld.init(g, m0, n0, bz, wave, lane, lds0);
        ld.issue(0, 0);
    }
    // per-column epilogue constants: fetched behind the first stage, parked in registers, staged in LDS after the loop
    constexpr int NPAR = (EPI == EPI_FIXEDPOINT) ? PAR_LOADS : 0;
    constexpr int PPT  = (NPAR * BN + NW * 64 - 1) / (NW * 64);
    int32_t       par_reg[PPT > 0 ? PPT : 1];
    if (EPI == EPI_FIXEDPOINT && u_fl != 0)
    {
#pragma unroll
        for (int t = 0; t < PPT; ++t)
        {
            // (every lane loads: the count of loads in flight must not depend on the lane)
            const int idx = min(tid + t * NW * 64, NPAR * BN - 1);
            const int par = idx / BN, col = idx % BN;
            par_reg[t]    = par == 0 ? ((global_i32)u_cv)[(int64_t)bz * g.epi.colvec_batch_stride + n0 + col]
                                     : ((global_i32)u_qp)[(int64_t)(par - 1) * g.epi.qp_stride + n0 + col];
        }
    }
    typename ByteSet<Loader, MODE>::type set_a, set_b; // RING_BYTES: the stages on their way, even and odd ones
    if constexpr (MODE == RING_BYTES)
    {
        ld.load(set_a, 0);
        if (nk > 1)
            ld.load(set_b, 1);
    }
    else
    {
#pragma unroll
        for (int s = 1; s < NS; ++s)
            if (s < nk)
                ld.issue(s, s);
    }
    const bool fast = EPI == EPI_FIXEDPOINT && (qflag & 1) == 0;

    const int kg    = wave >> 2; // which half of a K step's depth this wave multiplies
    const int row_w = ((wave >> 1) & 1) * TM, col_w = (wave & 1) * TN;
    v4i       acc[RS][QS];
#pragma unroll
    for (int i = 0; i < RS; ++i)
#pragma unroll
        for (int j = 0; j < QS; ++j)
            acc[i][j] = (v4i){0, 0, 0, 0};
    // operand reads: lane -> (row lane % 16, 16-byte column lane / 16) of a block of 16 rows x 64 bytes. The swizzle of a row
    // repeats every 16 rows (for 8 and 16 columns per row alike), so one offset per sub-step serves all blocks
    const int lr = lane & 15, lh = lane >> 4;
    int       rd[SUB];
#pragma unroll
    for (int h = 0; h < SUB; ++h)
        rd[h] = lr * BK + ((((h * KG + kg) * 4 + lh) ^ swz<CPR>(lr)) << 4);
    const int a_rd = row_w * BK, b_rd = BM * BK + col_w * BK;

    const bool rowsum = g.epi.rowsum_mul != 0;
    int32_t    rsum[RS];
#pragma unroll
    for (int f = 0; f < RS; ++f)
        rsum[f] = 0;

    // this wave's loads of stage 0: behind them NS - 1 stages may still be in flight
    if constexpr (MODE == RING_BYTES)
    {
        ld.store(set_a, 0, 0);
        if (nk > 2)
            ld.load(set_a, 2);
        if (nk > 1)
            ld.store(set_b, 1, 1);
        if (nk > 3)
            ld.load(set_b, 3);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    else if (nk < NS)
        wait_vmcnt<0>();
    else
        wait_vmcnt<(NS - 1) * LPW>();
    if constexpr (MODE == RING_CONV) // ... and the padding it wrote there itself: the other waves read that too
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    block_barrier(); // stage 0 is in LDS

    v4i  fa[2][RS], fb[2][QS];
    auto read_one = [&](int set, int h, const char *s, int f)
    {
        if (f < RS)
            fa[set][f] = *(const v4i *)(s + a_rd + f * 16 * BK + rd[h]);
        else
            fb[set][f - RS] = *(const v4i *)(s + b_rd + (f - RS) * 16 * BK + rd[h]);
    };
    // One sub-step: the matrix instructions of the operands in set CUR, between them the reads of the next sub-step's into the
    // other set and NI loads from I0 on of the stage that t describes. The loads go out one by one: a wave's next one is taken
    // about 70 clocks after the one before and the wave stands still until then if it has nothing else to issue: in a row in
    // front of the matrix instructions they doubled the step.
    auto sub_step = [&](int kt, auto h_c, auto cur_c, const char *s_next, int h_next, const typename Loader::Step &t, auto first_c, auto count_c)
    {
        constexpr int H = decltype(h_c)::value, CUR = decltype(cur_c)::value;
        constexpr int I0 = decltype(first_c)::value, NI = decltype(count_c)::value;
        if (FLIP_A && MODE != RING_BYTES)
        {
#pragma unroll
            for (int f = 0; f < RS; ++f)
                fa[CUR][f] ^= (int)0x80808080;
        }
#pragma unroll
        for (int m = 0; m < NM; ++m)
        {
            const int i = m / QS, j = m % QS;
            acc[i][j]   = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[CUR][j], fa[CUR][i], acc[i][j], 0, 0, 0);
            if (m < NR)
                read_one(CUR ^ 1, h_next, s_next, m);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int l = m * NI / NM; l < (m + 1) * NI / NM; ++l)
                ld.issue_one(t, I0 + l);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (rowsum)
        {
            v4i ones = {ONES4, ONES4, ONES4, ONES4};
            if (MODE == RING_CONV && (g.conv.c_true != g.conv.C || (kt + 1) * BK > g.K))
            {
                const int k = kt * BK + (H * KG + kg) * 64 + lh * 16;
                ones        = patch_bytes(g.conv, k + bz * g.k_slice, k < g.K ? INT32_MAX : 0);
            }
#pragma unroll
            for (int f = 0; f < RS; ++f)
                rsum[f] = sum_bytes(fa[CUR][f], rsum[f], ones);
        }
    };
    using std::integral_constant;
    using set0 = integral_constant<int, 0>;
    using set1 = integral_constant<int, 1>;
    typename Loader::Step t{};
    int slot = 0;
    // One K step; par: the register set of its first sub-step. BEFORE / AFTER: loads go out in front of the barrier (the rest of
    // the stage whose first ones went out behind the last barrier) / behind it.
    constexpr int PER = (LPW + SUB - 1) / SUB; // loads behind the barrier
    auto k_step = [&](int kt, auto par_c, auto before_c, auto after_c)
    {
        constexpr bool BEFORE = decltype(before_c)::value, AFTER = decltype(after_c)::value;
        constexpr int  PAR = decltype(par_c)::value;
        if constexpr (SUB == 2)
            sub_step(kt, set0{}, par_c, smem + slot * STAGE, 1, t, integral_constant<int, PER>{}, integral_constant<int, BEFORE ? LPW - PER : 0>{});
        const int freed = slot;
        slot            = slot + 1 == NS ? 0 : slot + 1;
        if (AFTER)
            t = ld.step(kt + NS, freed); // (worked out while the matrix instructions run)
        // This wave's operands of the stage are in registers, and its loads of stage kt + 1 have to have landed, NS - 2 younger
        // stages may be in flight; behind the barrier the next stage may be read and this one's slot written.
        if (BEFORE || kt + NS <= nk)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * LPW) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        block_barrier();
        if (!AFTER && kt + NS < nk)
            ld.issue(kt + NS, freed);
        // (reads beyond the last step: whatever the slot holds, never used)
        sub_step(kt, integral_constant<int, SUB - 1>{}, integral_constant<int, (PAR + SUB - 1) & 1>{}, smem + slot * STAGE, 0, t, set0{},
                 integral_constant<int, AFTER ? PER : 0>{});
    };
#pragma unroll
    for (int f = 0; f < NR; ++f)
        read_one(0, 0, smem, f);
    using yes = std::true_type;
    using no  = std::false_type;
    if constexpr (MODE == RING_BYTES)
    {
        // Stage kt + 2 goes to LDS behind the barrier of step kt, stage kt + 4 takes over its registers
        auto byte_step = [&](int kt, typename Loader::Set &set)
        {
            sub_step(kt, set0{}, set0{}, smem + slot * STAGE, 1, t, set0{}, set0{});
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            block_barrier();
            slot = slot + 1 == NS ? 0 : slot + 1;
            if (kt + 2 < nk)
                ld.store(set, kt + 2, slot + 1 == NS ? 0 : slot + 1);
            if (kt + 4 < nk)
                ld.load(set, kt + 4);
            sub_step(kt, set1{}, set1{}, smem + slot * STAGE, 0, t, set0{}, set0{});
        };
        for (int kt = 0; kt < nk; kt += 2)
        {
            byte_step(kt, set_a);
            if (kt + 1 < nk)
                byte_step(kt + 1, set_b);
        }
    }
    else
    {
        // steps whose stage kt + NS is whole: [0, lean)
        const int lean = (ld.whole(nk - 1) ? nk : nk - 1) - NS;
        int       kt   = 0;
        if constexpr (SUB == 2)
        {
            if (lean > 0)
            {
                k_step(kt++, set0{}, no{}, yes{});
                for (; kt < lean; ++kt)
                    k_step(kt, set0{}, yes{}, yes{});
                k_step(kt++, set0{}, yes{}, no{}); // (nk > NS: there is such a step)
            }
            for (; kt < nk; ++kt)
                k_step(kt, set0{}, no{}, no{});
        }
        else
        {
            for (; kt + 1 < lean; kt += 2)
            {
                k_step(kt, set0{}, no{}, yes{});
                k_step(kt + 1, set1{}, no{}, yes{});
            }
            for (; kt < nk; kt += 2)
            {
                k_step(kt, set0{}, no{}, no{});
                if (kt + 1 < nk)
                    k_step(kt + 1, set1{}, no{}, no{});
            }
        }
    }
    // the reads issued last are never used, but must have left the LDS before the epilogue writes there
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    block_barrier();
    // The two groups' accumulators are added up: a wave hands the row blocks that its partner (wave ^ 4) finishes over through
    // LDS and takes its own, RE of RS each, so the epilogue is spread over all 8 waves
    v4i     fin[RE][QS];
    int32_t rfin[RE];
    if constexpr (KG == 1)
    {
#pragma unroll
        for (int i = 0; i < RE; ++i)
        {
#pragma unroll
            for (int j = 0; j < QS; ++j)
                fin[i][j] = acc[i][j];
            rfin[i] = rsum[i];
        }
    }
    else
    {
        v4i           *box = (v4i *)smem + (size_t)wave * RE * QS * 64 + lane, *obox = (v4i *)smem + (size_t)(wave ^ 4) * RE * QS * 64 + lane;
        int32_t       *rbox = (int32_t *)(smem + NW * RE * QS * 1024) + lane;
        auto give = [&](auto from_c)
        {
            constexpr int F = decltype(from_c)::value;
#pragma unroll
            for (int i = 0; i < RE; ++i)
            {
#pragma unroll
                for (int j = 0; j < QS; ++j)
                    box[(i * QS + j) * 64] = acc[F + i][j];
                rbox[(wave * RE + i) * 64] = rsum[F + i];
            }
        };
        auto take = [&](auto own_c)
        {
            constexpr int O = decltype(own_c)::value;
#pragma unroll
            for (int i = 0; i < RE; ++i)
            {
#pragma unroll
                for (int j = 0; j < QS; ++j)
                    fin[i][j] = acc[O + i][j] + obox[(i * QS + j) * 64];
                rfin[i] = rsum[O + i] + rbox[((wave ^ 4) * RE + i) * 64];
            }
        };
        using low  = integral_constant<int, 0>;
        using high = integral_constant<int, RE>;
        if (kg)
            give(low{});
        else
            give(high{});
        __syncthreads();
        if (kg)
            take(high{});
        else
            take(low{});
        __syncthreads();
    }
    const int row_e = row_w + kg * RE * 16;
    if (rowsum)
        finish_row_sums<RE>(rfin, g.epi.rowsum_mul, FLIP_A && MODE == RING_DENSE ? nk * BK - g.K : 0);
    // (rows on any byte: slices as planes and a second launch. With this behind their loop they were 3 to 5 % slower whole and 12 to 17 % in slices)
    if constexpr (MODE != RING_BYTES)
        if (g.slices > 1)
        {
            if (!join_slices<RE, QS, NW * 64>(fin, rfin, rowsum, g, tm * g.tiles_n + tn, bz, tid, (int *)smem))
                return;
            bz = 0;
        }

    if (fast)
    {
        int32_t *par = (int32_t *)smem;
#pragma unroll
        for (int t = 0; t < PPT; ++t)
        {
            const int idx = tid + t * NW * 64;
            if (idx < NPAR * BN)
                park_constant(par, idx, BN, par_reg[t], g.epi.result_offset);
        }
        __syncthreads();
        if (EPI == EPI_FIXEDPOINT)
        {
            char      *stage = smem + PAR_ROWS * BN * 4;
            const bool rowv  = g.epi.rowvec != nullptr || rowsum;
            auto       store = [&](auto planes_c)
            {
                constexpr bool PL = decltype(planes_c)::value;
                if (g.epi.qp_std && qflag == 0 && !rowv)
                    epilogue_store_staged<true, false, RE, QS, BM, BN, NW, PL>(fin, g, par, stage, m0, n0, row_e, col_w, wave, lane, bz,
                                                                               [] { __syncthreads(); });
                else if (g.epi.qp_std && qflag == 0)
                    epilogue_store_staged<true, true, RE, QS, BM, BN, NW, PL>(fin, g, par, stage, m0, n0, row_e, col_w, wave, lane, bz,
                                                                              [] { __syncthreads(); }, rfin, rowsum);
                else
                    epilogue_store_staged<false, true, RE, QS, BM, BN, NW, PL>(fin, g, par, stage, m0, n0, row_e, col_w, wave, lane, bz,
                                                                               [] { __syncthreads(); }, rfin, rowsum);
            };
            if (MODE == RING_CONV && g.epi.planes != 0)
                store(integral_constant<bool, MODE == RING_CONV>{});
            else
                store(no{});
        }
    }
    else if ((EPI == EPI_S32 || EPI == EPI_F32) && !g.epi.accumulate)
    {
        if constexpr (EPI != EPI_FIXEDPOINT)
            epilogue_store_wave32<EPI, RE, QS>(fin, g, smem + wave * 16 * (QS * 64 + 16), m0 + row_e, n0 + col_w, lane, bz, rfin, rowsum);
    }
    else if (MODE == RING_CONV && EPI == EPI_FIXEDPOINT && g.epi.planes != 0)
        epilogue_store_t<EPI, RE, QS, MODE == RING_CONV>(fin, g, m0 + row_e, n0 + col_w, lane, bz, rfin, rowsum);
    else
        epilogue_store_t<EPI, RE, QS>(fin, g, m0 + row_e, n0 + col_w, lane, bz, rfin, rowsum);
}
} // namespace mi355
