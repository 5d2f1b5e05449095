// Implementation of the C ABI declared in include/mi355_gemmlowp.h: descriptor checks, kernel selection, device
// workspace ownership, host <-> device staging, and the launches. No arithmetic lives here.
#include "../../include/mi355_gemmlowp.h"
#include "conv_rows_plan.hpp"
#include "conv_window_plan.hpp"
#include "internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <string>

using namespace mi355;

// Workspace of mi355_gemmlowp_run_noalloc: row sums of A, then (rows that are not dword aligned) the padded copy of A.
// One array per GPU for the life of the process; every call on a GPU shares it.
#define MI355_NOALLOC_SCRATCH_BYTES (8u << 20)
static __device__ __align__(256) unsigned char scratch[MI355_NOALLOC_SCRATCH_BYTES];

namespace
{
thread_local std::string g_err;

int fail(const char *fmt, ...)
{
    char    buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_err = buf;
    return 1;
}

#define HIP_TRY(expr)                                                                                  \
    do                                                                                                 \
    {                                                                                                  \
        const hipError_t e_ = (hipError_t)(expr);                                                      \
        if (e_ != hipSuccess)                                                                          \
            return fail("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__);    \
    } while (0)
#define TRY(expr)            \
    do                       \
    {                        \
        if ((expr) != 0)     \
            return 1;        \
    } while (0)

bool is_device_ptr(const void *p, bool *managed = nullptr)
{
    if (managed)
        *managed = false;
    if (p == nullptr)
        return false;
    hipPointerAttribute_t attr;
    const hipError_t      e = hipPointerGetAttributes(&attr, p);
    if (e != hipSuccess)
    {
        (void)hipGetLastError(); // plain host memory: clear the sticky error
        return false;
    }
    if (managed)
        *managed = attr.type == hipMemoryTypeManaged || (attr.type == hipMemoryTypeDevice && attr.isManaged);
    return attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged;
}

// What kind of memory an argument slot of a handle was last given: asked once per value and slot, so that a
// steady-state run() asks nothing. The answer lives and dies with the handle. It is stale only if the address is freed
// and handed out again by an allocation of the other kind between two runs of the same handle (the header says so).
struct PtrKind
{
    const void *p   = nullptr;
    bool        dev = false;
    bool        is_device(const void *q)
    {
        if (q == nullptr)
            return false;
        if (q != p)
            dev = is_device_ptr(q), p = q;
        return dev;
    }
};

struct DevBuf
{
    void  *p   = nullptr;
    size_t cap = 0;
    int    ensure(size_t bytes)
    {
        if (bytes <= cap && p != nullptr)
            return 0;
        if (p)
        {
            HIP_TRY(hipFree(p));
            p = nullptr, cap = 0;
        }
        if (bytes == 0)
            bytes = 16;
        HIP_TRY(hipMalloc(&p, bytes));
        cap = bytes;
        return 0;
    }
    void release()
    {
        if (p)
            (void)hipFree(p);
        p = nullptr, cap = 0;
    }
    template <typename T>
    T *as() const
    {
        return (T *)p;
    }
};

// brings `bytes` at `src` to the device if it is host memory; returns the device pointer to use. *host_may_write (when
// given) is set, never cleared, if the host may write the memory that is read: the staging buffer or managed memory.
int to_device(const void *src, size_t bytes, DevBuf &stage, hipStream_t s, const void **out, PtrKind *kind = nullptr,
              bool *host_may_write = nullptr)
{
    if (src == nullptr)
    {
        *out = nullptr;
        return 0;
    }
    bool managed = false;
    if (kind ? kind->is_device(src) : is_device_ptr(src, &managed))
    {
        if (host_may_write && managed)
            *host_may_write = true;
        *out = src;
        return 0;
    }
    if (host_may_write)
        *host_may_write = true;
    TRY(stage.ensure(bytes));
    HIP_TRY(hipMemcpyAsync(stage.p, src, bytes, hipMemcpyHostToDevice, s));
    *out = stage.p;
    return 0;
}

int num_cus()
{
    static int cus = -1;
    if (cus < 0)
    {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess)
            return 256;
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess)
            return 256;
        cus = prop.multiProcessorCount;
    }
    return cus;
}

bool is_8bit(int dt)
{
    return dt == MI355_U8 || dt == MI355_S8;
}

// The part of a GEMM that both the dense handle and the convolution handle need
struct GemmCore
{
    int     M = 0, N = 0, K = 0, batch = 1;
    int     epi       = EPI_S32;
    int     dst_dtype = MI355_S32;
    bool    flip_a = false, flip_b = false;
    int32_t a_offset = 0, b_offset = 0; // as given (added convention)
    mi355_requant rq{};
    float   scale = 1.f, act_min = -INFINITY, act_max = INFINITY;
    bool    accumulate = false, act_twice = false;
    bool    half_out = false; // this run's kernels round to half themselves (set around run_dense)
    int     path = MI355_PATH_AUTO, cfg_idx = 0, dma_idx = -1;
    int     force_tile = -1; // >= 0: the pipelined kernel's tile configuration the caller asked for (MI355_PATH_TILE + n)
    int     Kp = 0, Np = 0;
    bool    b_shared = true; // one B for all batches
    bool    has_bias = false, has_pc = false, prepared = false;
    bool    has_narrow = false; // Bn holds the narrow kernel's image of B
    bool    pt_vectors = false; // streaming path, per-tensor requantisation: mult / shift hold the scalars, replicated
    std::string kname;
    DevBuf  Bp, Bs, Bn, colsum, colvec, colpart, rowvec, mult, shift, bias, Ap, fill, qp, zeros, parts, zerocol, arrived;
    // A prepare that only enqueues (on the legacy default stream, every operand in device memory, nothing left to set up): an
    // event behind it, which runs on other streams wait for
    hipEvent_t  prep_done    = nullptr;
    bool        prep_pending = false;
    bool        recorded = false; // a run was recorded into a graph, which may be launched at any time
    // What is known of buffers that are written once and then kept (see keep_flags)
    int         fill_set = -1; // the byte the 16 filler bytes hold (-1: not known)
    bool        zeros_set = false, zerocol_set = false, arrived_set = false;
    ptrdiff_t    sums_at = -1; // where the sums of many slices lie in `arrived`, behind the counters (-1: in `parts`)
    SkinnySlices sk_plan; // the streaming kernel's K slices and their memory (prepare() fills it in)
    bool        qp_scalar_set = false; // the per-tensor requantisation vectors hold qp_rq
    bool        writes_recorded = false;
    mi355_requant qp_rq{};
    int     splitk = 1;      // K slices of the pipelined kernel
    int     byte_idx = -1; // the configuration that takes rows of A on any byte without a copy, and what the model prices it and the other at
    double  us_bytes = 0, us_dma = 0, us_copied = 0;
    bool    byte_lda = false;   // rows or batch entries of A that do not start on dwords, as far as the strides say
    bool    one_launch = false; // few rows, one launch of the pipelined kernel instead of two of the streaming one's
    int     splitk_plan = 1; // what the cost model chose with the tile shape (create()); prepare() checks it and allocates
    int         patch_c = 0, patch_c_true = 0; // a convolution's channels in the kernels' K, and how many of them count (0: dense)
    int         panels_from = 0; // rows of the output from which the narrow kernel takes several panels of columns
    const void *rs_src = nullptr; // conv_row_terms
    ConvGeom    rs_geom{};
    int     k_const = 0;       // > 0: the K of the constant term a_offset * b_offset * K, where the kernels' K counts padded channels
    bool    qp_on = false; // the digested requantisation vectors (and the flag word behind them) exist
    std::string kname_mfma, kname_dma, kprefix;
    // The names a run can report, composed when the choice is made (create, prepare, update): a run only points at one
    // of them - it must not touch the host heap
    std::string        kname_window, kname_narrow, kname_band, kname_dma_full, kname_bytes, kname_rows, kname_splitk, kname_mfma_full;
    const char        *kname_static = nullptr; // the streaming kernel names its forms itself
    const std::string *kname_run = nullptr; // what the last run took (nullptr: no run yet, kname is what create announced)
    uint8_t fill_byte = 0; // value of the 16 filler bytes (0, or the im2col pad value)
    void   *ext_ws = nullptr; // set around a run that must not allocate: see run_dense
    size_t  ext_ws_bytes = 0;
    bool    ext_ws_busy = false; // the caller's workspace may still be read by kernels of another stream
    bool    ext_ws_used = false; // set by run_dense: this run put something into the caller's workspace

    void refresh_names()
    {
        kname_window    = kprefix + "pp_window_64";
        kname_narrow    = kprefix + "narrow_32x64";
        kname_band      = kprefix + "band_32x64";
        kname_dma_full  = kprefix + kname_dma;
        kname_rows      = kprefix + "rows_32x64";
        kname_bytes     = byte_idx >= 0 ? kprefix + dma_config(byte_idx).name + "_bytes" : std::string();
        kname_splitk    = kname_dma_full + "_splitk" + std::to_string(splitk);
        kname_mfma_full = kprefix + kname_mfma;
    }
    const char *name() const { return kname_static ? kname_static : (kname_run ? kname_run->c_str() : kname.c_str()); }

    int32_t a_off_eff() const { return (int32_t)((uint32_t)a_offset + (flip_a ? 128u : 0u)); }
    int32_t b_off_eff() const { return (int32_t)((uint32_t)b_offset + (flip_b ? 128u : 0u)); }
    int     nb() const { return b_shared ? 1 : batch; }

    void release()
    {
        if (prep_done)
            (void)hipEventDestroy(prep_done);
        prep_done = nullptr, prep_pending = false;
        Bp.release(), Bs.release(), Bn.release(), colsum.release(), colvec.release(), colpart.release(), rowvec.release(), mult.release();
        shift.release(), bias.release(), Ap.release(), fill.release(), qp.release(), zeros.release(), parts.release(), zerocol.release(), arrived.release();
    }

    static constexpr int MOST_SLICES = 32;

    int choose_kernel()
    {
        Kp = round_up(K, PACK_K_ALIGN);
        Np = round_up(N, PACK_N_ALIGN);
        if (path >= MI355_PATH_TILE)
        {
            if (path - MI355_PATH_TILE >= dma_num_configs())
                return fail("path %d names tile configuration %d; there are %d", path, path - MI355_PATH_TILE, dma_num_configs());
            force_tile = path - MI355_PATH_TILE, path = MI355_PATH_MFMA;
        }
        else if (path < 0 || path > MI355_PATH_SKINNY)
            return fail("unknown path %d", path);
        const bool automatic = path == MI355_PATH_AUTO;
        if (automatic)
            // measured: up to 32 rows the streaming kernel always wins, up to 64 rows sometimes (below)
            // (a batch of small products runs the streaming kernel once per entry: the tiled kernels would spend a 64-row
            // tile, mostly padding, on each)
            path = (M <= 32 || (batch == 1 && M <= SKINNY_MAX_M)) ? MI355_PATH_SKINNY : MI355_PATH_MFMA;
        const int cus = num_cus();
        // The pipelined kernel's tile is chosen with a small cost model in microseconds (the prices and what they were fitted to
        // stand at g_dma_cost): a tile costs MfmaConfig::us_tile for its start-up and epilogue, of which the workgroups that
        // fit a compute unit together share all but us_more, plus us_step for every K step, which a full chip slows down
        // by a share us_load of it (L2, HBM and the power limit are shared by all compute units); the tiles that share a compute unit
        // take at least us_lone for a K step together.
        // A single GEMM may also run its K range as slices (see finish_prepare()): the tiles of all slices share the
        // chip, every slice has its share of the K steps, and the last workgroup of a tile adds up the others' sums: 0.7 us, 0.3 us per
        // slice and 0.6 us per million sums written and read again, beyond JOIN_PLANES slices 0.9 us and 4 us
        // per million additions, fitted to 14 products of 64 to 1162 rows with 2 to 16 slices, off by 0.4 on average (convolutions, fitted with
        // their tiles and a second launch for the sums, which took 1 us more: 3.2, 0.18 and 0.88; rows on any byte, which keep that launch: 2.4,
        // 0.1 and 2, and 0.88 of it all). The 1.06 of dense products: where both are priced alike whole tiles are the faster ones more often
        // (100 x 1000 x 2000: 6.3 us whole, 6.7 as 2 slices; 256 x 1024 x 2048: 6.0 and 7.0).
        auto finish_us = [&](int loader, int sl) -> double
        {
            const double sums = (double)sl * M * N;
            return sl <= 1           ? 0.0
                   : loader == 1     ? 3.2 + 0.18 * sl + 0.88e-6 * sums
                   : loader == 2     ? 2.4 + 0.1 * sl + 2e-6 * sums
                   : sl <= JOIN_PLANES ? 0.7 + 0.3 * sl + 0.6e-6 * sums
                                     : 0.9 + 4e-6 * sums;
        };
        auto pick_dma = [&](int loader, int &plan, double &best_cost, int fixed_slices = 0) -> int
        {
            int best = -1;
            for (int i = 0; i < dma_num_configs(); ++i)
            {
                const MfmaConfig c = dma_config(i, loader);
                if (c.us_tile <= 0 || (N <= 64 && c.BN > 64) || Kp % c.BK != 0)
                    continue;
                const double tiles   = (double)((M + c.BM - 1) / c.BM) * ((N + c.BN - 1) / c.BN) * batch;
                const int    occ_lds = (160 * 1024) / c.lds_bytes, occ_wav = 32 / c.waves;
                const double occ     = std::max(1, std::min(occ_lds, occ_wav));
                const int    nk      = (K + c.BK - 1) / c.BK;
                for (int want = fixed_slices ? fixed_slices : 1; want <= (fixed_slices ? fixed_slices : MOST_SLICES); ++want)
                {
                    // (slices of equal whole K steps but the last, none of them empty)
                    const int per = (nk + want - 1) / want, sl = (nk + per - 1) / per;
                    if (want > 1 && (batch != 1 || per * c.BK < 512 || (i == 0 && fixed_slices == 0)))
                        break;
                    if (sl != want)
                        continue;
                    const double per_cu = std::ceil(tiles * sl / cus), load = std::min(1.0, tiles * sl / cus);
                    const double finish = finish_us(loader, sl);
                    const double rounds = std::ceil(per_cu / occ), full = std::floor(per_cu / occ), rest = per_cu - full * occ, step = c.us_step * (1.0 + c.us_load * load);
                    const double steps  = per * (full * std::max(c.us_lone, occ * step) + (rest > 0 ? std::max(c.us_lone, rest * step) : 0.0));
                    const double cost   = (rounds * c.us_tile + (per_cu - rounds) * c.us_more + steps + finish) * (sl <= 1 || loader == 1 ? 1.0 : loader == 2 ? 0.88 : 1.06);
                    if (best < 0 || cost < best_cost)
                        best = i, best_cost = cost, plan = sl;
                }
            }
            return best;
        };
        if (automatic && path == MI355_PATH_SKINNY && M > 32 && K >= 16)
        {
            // 33 to 64 rows: the tiles, or up to a K of 4096 the streaming kernel, whose operand blocks of A then stay in registers (its
            // forms beyond are slower than the tiles everywhere: 60 rows, 3072 x 12128 23.8 us, tiles 17.6; 2880 x 7936 17.9 and 11.1), whichever
            // is priced lower. The tiles' prices come from a B that stays in the caches; weights that come from memory add what B is over
            // 20 MB at 3.3 TB/s (15 products of 0.8 to 78 MB: 0.9 to 17.4 us, off by 1). 60 rows, tiles and stream: 8640 x 2880 9.1 and
            // 13.0, 9792 x 3264 12.7 and 13.6; 3264 x 3264 9.8 and 8.7, 11008 x 4096 17.8 and 16.6, 768 x 2064 8.3 and 6.1.
            // (Whole 64-byte blocks with an offset on B, whose row sums take the streaming kernel a pass, were not measured and stay there.)
            int          plan = 1;
            double       tiles = 0;
            const double pass = byte_lda || b_off_eff() != 0 ? 2.5 : 0.0, cold = std::max(1.0, 0.3 * ((double)N * K * 1e-6 - 20.0));
            if (pick_dma(byte_lda || (b_off_eff() != 0 && K % 16 != 0) ? 2 : 0, plan, tiles) >= 0 &&
                (K > 4096 || ((b_off_eff() == 0 || K % 64 != 0) && tiles + cold < skinny_64rows_us(M, N, K, cus) + pass)))
                path = MI355_PATH_MFMA;
        }
        if (automatic && batch == 1 && path == MI355_PATH_SKINNY && (byte_lda || (b_off_eff() != 0 && K % 64 != 0)) && K >= 16 &&
            (double)N * K <= 4e6)
        {
            // The streaming kernel needs a pass in front here, for a copy of the rows or for their sums; the pipelined one does both
            // itself and is one launch. Launched one by one from the host two launches take 6.2 us at least and one 4.3, so it may gain there what
            // it loses in a graph: taken where it gains more than it loses (in a graph and one by one: 1 x 94 x 489: 3.7 -> 4.7 and 6.2 -> 5.2;
            // not 3 x 384 x 745: 4.2 -> 5.7 and 6.2 -> 6.1; 1 x 27 x 1327: 4.3 -> 8.1, 7.8 -> 8.2). The two launches in a graph: fitted
            // to 159 products (8 %); over these the choice is 5 % faster than two launches in a graph and 17 % one by one. From 4 MB of B on the stream
            // counts (50 x 6000 x 6001: 22.9 and 37.6), and rows of whole 64-byte blocks have the streaming kernel's best forms.
            int          plan = 1;
            double       us   = 0;
            const bool   bytes = byte_lda || K % 16 != 0;
            const int    idx  = pick_dma(bytes ? 2 : 0, plan, us, 1);
            if (bytes)
                us *= 0.82; // (a single row of tiles takes 0.90 of the price, over 222 products of up to 64 rows. The factor weighs the gain one by
                            // one against the loss in a graph: with 1 49 of them lose over 5 % one by one and 4 over 10 % in a graph, with 0.8 7 and 23)
            const double two  = M > 32 ? 4.2 + 2.0e-3 * K + 0.36e-6 * N * K : 3.9 + 0.64e-3 * K + 0.25e-6 * N * K;
            if (idx >= 0 && std::max(4.3, us) < (std::max(6.2, two) + two) / 2)
                path = MI355_PATH_MFMA, one_launch = true;
        }
        if (path == MI355_PATH_SKINNY && M > SKINNY_MAX_M)
            return fail("skinny path needs M <= %d", SKINNY_MAX_M);
        if (path == MI355_PATH_SIMPLE)
            kname = "simple";
        else if (path == MI355_PATH_SKINNY)
            kname = "skinny";
        else
        {
            auto pick = [&](int count, MfmaConfig (*get)(int), const char *env) -> int
            {
                int  best = -1;
                long most = -1;
                for (int i = 0; i < count; ++i)
                {
                    const MfmaConfig c     = get(i);
                    const long       tiles = (long)((M + c.BM - 1) / c.BM) * ((N + c.BN - 1) / c.BN) * batch;
                    if (N <= 64 && c.BN > 64)
                        continue;
                    if (tiles >= cus)
                        return i;
                    if (tiles > most)
                        most = tiles, best = i;
                }
                (void)env;
                return best;
            };
            cfg_idx = pick(mfma_num_configs(), mfma_config, nullptr);
            dma_idx = pick_dma(patch_c > 0 ? 1 : 0, splitk_plan, us_dma, one_launch ? 1 : 0);
            int byte_plan = 1;
            if (patch_c == 0 && force_tile < 0 && dma_idx >= 0) // (the planes are those of the other's slices)
            {
                byte_idx = pick_dma(2, byte_plan, us_bytes, splitk_plan);
                // (against rows on any byte, whose slices take the second launch: fitted with that launch and its prices on both sides)
                us_copied = splitk_plan > 1 ? 0.83 * us_dma + 0.88 * (finish_us(2, splitk_plan) - finish_us(0, splitk_plan)) : us_dma;
            }
            if (force_tile >= 0 && Kp % dma_config(force_tile).BK == 0 && dma_idx != force_tile)
            {
                // a tile shape named by the caller: as many slices as fill the chip once, at least 1024 deep
                dma_idx = force_tile, splitk_plan = 1;
                const MfmaConfig c     = dma_config(dma_idx);
                const int64_t    tiles = (int64_t)((M + c.BM - 1) / c.BM) * ((N + c.BN - 1) / c.BN);
                if (batch == 1 && tiles * 2 <= cus && K >= 2048)
                {
                    const int nk = (K + c.BK - 1) / c.BK, want = (int)std::min<int64_t>(std::min<int64_t>(cus / tiles, K / 1024), 8);
                    const int per = (nk + want - 1) / want;
                    splitk_plan   = (nk + per - 1) / per;
                }
            }
            if (K < 16)
                dma_idx = byte_idx = -1;
            kname_mfma = mfma_config(cfg_idx).name;
            kname_dma  = dma_idx >= 0 ? dma_config(dma_idx).name : "";
            kname      = dma_idx >= 0 ? kname_dma : kname_mfma;
        }
        refresh_names();
        return 0;
    }

    ColumnFinish column_finish(const int32_t *bias_in) const
    {
        return {colsum.as<int32_t>(), colvec.as<int32_t>(), bias_in, bias.as<int32_t>(), (uint32_t)a_off_eff(), (uint32_t)b_off_eff(),
                (uint32_t)(k_const > 0 ? k_const : K), N};
    }

    // B (device memory; N rows of K elements when transposed) -> the packed image the chosen kernel reads, the columns' sums
    // and the per-column terms of the epilogue. bias_in: device memory, or null
    // (both: one transposed B once more in operand order, behind the other image)
    int pack(const void *B, int64_t ldb, int64_t b_bs, bool transposed, int kf, const int32_t *bias_in, hipStream_t s, bool both = false)
    {
        const bool   skinny = path == MI355_PATH_SKINNY;
        DevBuf      &dst    = skinny ? Bs : Bp;
        const size_t image  = (size_t)Np * Kp;
        has_bias            = bias_in != nullptr;
        TRY(dst.ensure(image * (both ? 2 : nb())));
        TRY(colsum.ensure(sizeof(int32_t) * (size_t)Np * nb()));
        TRY(colvec.ensure(sizeof(int32_t) * (size_t)Np * nb()));
        if (has_bias)
            TRY(bias.ensure(sizeof(int32_t) * (size_t)N));
        constexpr int MOST = 32768; // batch entries along a grid dimension
        // (one count for all parts, the last of which may be small: the workspace is sized by it)
        const int     splits = transposed ? 1 : pack_b_splits(Kp, Np, std::min(nb(), MOST));
        if (splits > 1)
            TRY(colpart.ensure(sizeof(int32_t) * (size_t)Np * nb() * splits));
        for (int b = 0; b < nb(); b += MOST)
        {
            const int      n   = std::min(MOST, nb() - b);
            const uint8_t *src = (const uint8_t *)B + (int64_t)b * b_bs;
            int8_t        *out = dst.as<int8_t>() + (size_t)b * image;
            ColumnFinish   f   = column_finish(epi == EPI_FIXEDPOINT ? bias_in : nullptr);
            f.colsum += (int64_t)b * Np, f.colvec += (int64_t)b * Np;
            if (transposed)
                HIP_TRY(pack_bt_launch(src, ldb, b_bs, n, K, N, Kp, Np, flip_b, kf, skinny, out, f, s, both ? out + image : nullptr));
            else
                HIP_TRY(pack_b_launch(src, ldb, b_bs, n, K, N, Kp, Np, flip_b, kf, skinny, splits, out, colpart.as<int32_t>(), f, s));
        }
        return 0;
    }

    // Whether `s` is recording a graph (an error of the query counts as recording)
    static bool capturing(hipStream_t s)
    {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cap) == hipSuccess)
            return cap != hipStreamCaptureStatusNone;
        (void)hipGetLastError();
        return true;
    }

    // Behind a prepare (or an update behind one) whose work is left running on the legacy default stream. Only there: a stream
    // that can be captured may be recording the run that follows, and then neither the host nor another stream is allowed to
    // wait for an event that was recorded in it.
    int prepare_enqueued()
    {
        prep_pending = false;
        if (capturing(nullptr))
        {
            HIP_TRY(hipStreamSynchronize(nullptr));
            return 0;
        }
        // (nothing on the host reads what the kernels wrote: without the system fence the event costs 0.9 us between the two
        // kernels instead of 2.7)
        if (prep_done == nullptr)
            HIP_TRY(hipEventCreateWithFlags(&prep_done, hipEventDisableTiming | hipEventDisableSystemFence));
        HIP_TRY(hipEventRecord(prep_done, nullptr));
        prep_pending = true;
        return 0;
    }

    // in front of whatever reads or writes on s what a prepare writes
    int wait_for_prepare(hipStream_t s)
    {
        if (s == nullptr)
            return 0;
        if (recorded ? prep_pending && capturing(s) : capturing(s))
        {
            // a graph under construction cannot wait for work outside it, and may be launched on any stream
            recorded = true;
            return prepare_over();
        }
        if (!prep_pending)
            return 0;
        // (once it is over no later run waits again: 0.1 us of host time each)
        const hipError_t e = event_call(hipEventQuery);
        if (e == hipSuccess)
            prep_pending = false;
        else if (e == hipErrorNotReady)
            HIP_TRY(hipStreamWaitEvent(s, prep_done, 0));
        else
            HIP_TRY(e);
        return 0;
    }

    // the host waits
    int prepare_over()
    {
        if (!prep_pending)
            return 0;
        HIP_TRY(event_call(hipEventSynchronize));
        prep_pending = false;
        return 0;
    }

    // `call` on the prepare's event, whatever the thread is recording
    hipError_t event_call(hipError_t (*call)(hipEvent_t))
    {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        hipError_t           e    = hipThreadExchangeStreamCaptureMode(&mode);
        if (e != hipSuccess)
            return e;
        const hipError_t got = call(prep_done);
        if (got == hipErrorNotReady)
            (void)hipGetLastError(); // not an error: the launches behind it ask for the last one
        e = hipThreadExchangeStreamCaptureMode(&mode);
        return e != hipSuccess ? e : got;
    }

    // whether the narrow kernel's image of B is made
    bool narrow_form() const
    {
        return path == MI355_PATH_MFMA && patch_c > 0 && nb() == 1 && (N <= 64 || (N <= 256 && K <= 192 && M >= panels_from)) && narrow_panel_chunks(K) > 0;
    }

    // after pack(): everything else a run reads
    int finish_prepare(const int32_t *mult_in, const int32_t *shift_in, hipStream_t s)
    {
        keep_flags(s);
        has_pc = epi == EPI_FIXEDPOINT && rq.per_channel != 0;
        if (has_pc)
        {
            if (mult_in == nullptr || shift_in == nullptr)
                return fail("per-channel requantisation needs multiplier and shift arrays");
            // padded like the packed B panel: the epilogue reads these as 16-byte vectors
            TRY(mult.ensure(sizeof(int32_t) * (size_t)Np));
            TRY(shift.ensure(sizeof(int32_t) * (size_t)Np));
            HIP_TRY(fill_i32_launch(mult.as<int32_t>(), 0, Np, s));
            HIP_TRY(fill_i32_launch(shift.as<int32_t>(), 0, Np, s));
            HIP_TRY(hipMemcpyAsync(mult.p, mult_in, sizeof(int32_t) * (size_t)N, hipMemcpyDefault, s));
            HIP_TRY(hipMemcpyAsync(shift.p, shift_in, sizeof(int32_t) * (size_t)N, hipMemcpyDefault, s));
        }
        // few output columns and a short K: the image of the B panel the narrow kernel copies into LDS
        has_narrow = narrow_form();
        if (has_narrow)
        {
            const int chunks = narrow_panel_chunks(K);
            const int rows = round_up(N, 64); // panels of 64 columns (Np, a multiple of 256, covers them)
            TRY(Bn.ensure((size_t)rows * (chunks + NARROW_PAD_PIECES) * 16));
            HIP_TRY(pack_b_narrow_launch(Bp.as<int8_t>(), Kp, Np, chunks, rows, K, patch_c, patch_c_true, Bn.as<int8_t>(), s));
        }
        TRY(set_fill(s));
        if (path == MI355_PATH_SKINNY && !zeros_set)
        {
            // the streaming kernel fetches its per-row vector without asking whether there is one
            TRY(zeros.ensure(sizeof(int32_t) * SKINNY_MAX_M));
            HIP_TRY(fill_i32_launch(zeros.as<int32_t>(), 0, SKINNY_MAX_M, s));
            zeros_set = true;
        }
        if (path == MI355_PATH_SKINNY && batch == 1)
        {
            sk_plan = skinny_slices(M, N, K, num_cus());
            if (sk_plan.slices > 1)
            {
                TRY(parts.ensure(sizeof(int32_t) * sk_plan.words));
                TRY(clear_arrived(sk_plan.grid, s));
                sk_plan.parts = parts.as<int32_t>(), sk_plan.arrived = arrived.as<int32_t>();
            }
        }
        // A deep K under few output tiles: the pipelined kernel would leave most compute units idle, each of the others
        // walking the whole K. The K range is cut into slices that run as the batch entries of one launch (the slice
        // offset is the batch stride of A and of the packed B alike); a tile's last workgroup sums its slices and applies the
        // epilogue. Slices are whole K steps of the tile shape, the last one as many as are left.
        splitk = 1;
        if (path == MI355_PATH_MFMA && dma_idx >= 0 && batch == 1)
            splitk = splitk_plan;
        if (splitk > 1)
        {
            size_t words = 0, tiles = 0;
            if (dma_idx > 0)
            {
                const MfmaConfig c = dma_config(dma_idx);
                tiles = (size_t)((M + c.BM - 1) / c.BM) * ((N + c.BN - 1) / c.BN);
                words = tiles * (size_t)ring_slice_words(c.BM, c.BN);
            }
            const size_t ldp = ((size_t)N + 3) & ~(size_t)3;
            // (many slices: one place for the sums of a tile, behind the counters. 256 x 128 tiles, rows on any byte: planes of sums)
            const bool added = splitk > JOIN_PLANES;
            tiles            = (tiles + 1) & ~(size_t)1;
            sums_at          = added ? (ptrdiff_t)tiles : -1;
            TRY(clear_arrived(tiles + (added ? words : 0), s));
            TRY(parts.ensure(sizeof(int32_t) * (size_t)splitk * std::max(added ? (size_t)0 : words, dma_idx == 0 || byte_idx >= 0 ? (size_t)M * ldp : (size_t)0)));
            if (own_row_terms())
                TRY(rowvec.ensure(sizeof(int32_t) * (size_t)M));
            if (!zerocol_set)
            {
                TRY(zerocol.ensure(sizeof(int32_t) * (size_t)Np));
                HIP_TRY(fill_i32_launch(zerocol.as<int32_t>(), 0, Np, s));
                zerocol_set = true;
            }
        }
        TRY(refresh_qparams(s));
        refresh_names();
        keep_flags(s); // (what was set on the way here may only have been recorded)
        return 0;
    }

    // In front of what the flags decide and behind what sets them. Under capture a write only goes into a graph: it has not
    // happened, and launching the graph repeats it whatever came after. From the first one on nothing is taken as known, and
    // every prepare and update writes all of it.
    void keep_flags(hipStream_t s)
    {
        if (!writes_recorded && s != nullptr && capturing(s))
            writes_recorded = true;
        if (writes_recorded)
            fill_set = -1, zeros_set = zerocol_set = arrived_set = qp_scalar_set = false;
    }

    // the counters of workgroups that finish a slice of K (each run leaves them zero)
    int clear_arrived(size_t n, hipStream_t s)
    {
        if (n == 0 || (arrived_set && arrived.cap >= sizeof(int32_t) * n))
            return 0;
        arrived_set = false;
        TRY(arrived.ensure(sizeof(int32_t) * n));
        HIP_TRY(fill_i32_launch(arrived.as<int32_t>(), 0, (int64_t)n, s));
        arrived_set = true;
        return 0;
    }

    int set_fill(hipStream_t s)
    {
        TRY(fill.ensure(16));
        if (fill_set == fill_byte)
            return 0;
        fill_set = -1;
        HIP_TRY(fill_i32_launch(fill.as<int32_t>(), (int32_t)(0x01010101u * fill_byte), 4, s));
        fill_set = fill_byte;
        return 0;
    }

    int refresh_colvec(hipStream_t s)
    {
        constexpr int MOST = 32768;
        for (int b = 0; b < nb(); b += MOST)
        {
            ColumnFinish f = column_finish((has_bias && epi == EPI_FIXEDPOINT) ? bias.as<int32_t>() : nullptr);
            f.colsum += (int64_t)b * Np, f.colvec += (int64_t)b * Np;
            HIP_TRY(colvec_launch(Np, std::min(MOST, nb() - b), f, s));
        }
        return 0;
    }

    // Digest multipliers / shifts for the pipelined kernel's epilogue. Whether the branch-free forms apply (no negative
    // multiplier; every column normalised) is left in a flag word behind the vectors, which the kernel reads itself:
    // nothing here waits for the device.
    int refresh_qparams(hipStream_t s)
    {
        // per-tensor: what is there still holds unless the requantisation has changed
        if (!has_pc && qp_scalar_set && memcmp(&qp_rq, &rq, sizeof(rq)) == 0)
            return 0;
        qp_scalar_set = false;
        TRY(write_qparams(s));
        qp_scalar_set = !has_pc, qp_rq = rq;
        return 0;
    }

    int write_qparams(hipStream_t s)
    {
        qp_on = false;
        if (path == MI355_PATH_SKINNY && epi == EPI_FIXEDPOINT && !has_pc)
        {
            // the streaming kernel always reads per-column vectors (a fetch behind a condition would cost it the exact
            // count of its loads in flight): per-tensor constants are replicated
            TRY(mult.ensure(sizeof(int32_t) * (size_t)Np));
            TRY(shift.ensure(sizeof(int32_t) * (size_t)Np));
            HIP_TRY(fill_i32_launch(mult.as<int32_t>(), rq.multiplier, Np, s));
            HIP_TRY(fill_i32_launch(shift.as<int32_t>(), rq.shift, Np, s));
            pt_vectors = true;
        }
        if (epi != EPI_FIXEDPOINT || rq.stage != MI355_STAGE_FIXEDPOINT)
            return 0;
        TRY(qp.ensure(sizeof(int32_t) * ((size_t)QP_COUNT * Np + 4)));
        int32_t *flag = qp.as<int32_t>() + (size_t)QP_COUNT * Np;
        HIP_TRY(qparams_launch(has_pc ? mult.as<int32_t>() : nullptr, has_pc ? shift.as<int32_t>() : nullptr,
                               rq.multiplier, rq.shift, N, Np, qp.as<int32_t>(), flag, s));
        qp_on = true;
        return 0;
    }

    void fill_epi(EpiParams &p, const float *bias_f32) const
    {
        p.qp                  = qp_on ? qp.as<int32_t>() : nullptr;
        p.qp_flag             = qp_on ? qp.as<int32_t>() + (size_t)QP_COUNT * Np : nullptr;
        p.qp_std              = (qp_on && rq.result_offset >= -STD_MAX_OFFSET && rq.result_offset <= STD_MAX_OFFSET) ? 1 : 0;
        p.qp_stride           = Np;
        p.colvec              = colvec.as<int32_t>();
        p.rowvec              = nullptr;
        p.mult                = (has_pc || pt_vectors) ? mult.as<int32_t>() : nullptr;
        p.shift               = (has_pc || pt_vectors) ? shift.as<int32_t>() : nullptr;
        p.bias_f32            = bias_f32;
        p.colvec_batch_stride = b_shared ? 0 : Np;
        p.rowvec_batch_stride = M;
        p.mult_s              = rq.multiplier;
        p.shift_s             = rq.shift;
        p.result_offset       = rq.result_offset;
        p.stage               = rq.stage;
        const int32_t tlo = dst_dtype == MI355_S8 ? -128 : 0, thi = dst_dtype == MI355_S8 ? 127 : 255;
        p.lo                  = rq.min_bound > tlo ? rq.min_bound : tlo;
        p.hi                  = rq.max_bound < thi ? rq.max_bound : thi;
        p.scale               = scale;
        p.act_min             = act_min;
        p.act_max             = act_max;
        p.has_offsets         = (a_offset != 0 || b_offset != 0) ? 1 : 0;
        p.dst_signed          = dst_dtype == MI355_S8;
        p.accumulate          = accumulate ? 1 : 0;
        p.act_twice           = act_twice ? 1 : 0;
        p.half_out            = half_out ? 1 : 0;
    }

    // K slices to a float destination take the row terms from a pass (see run_dense) that the same product whole would not
    // need: the vector is there from prepare on, so that a first run can be recorded and a run_noalloc needs no workspace
    bool own_row_terms() const { return splitk > 1 && epi == EPI_F32; }

    // Whether the kernel that a run takes can round to half itself: the streaming and the pipelined one, not the fallbacks
    bool rounds_to_half(int64_t lda) const
    {
        return !accumulate && (path == MI355_PATH_SKINNY || (path == MI355_PATH_MFMA && dma_idx >= 0 && K >= 16 && (int64_t)std::max(lda, (int64_t)Kp) * 256 + Kp < ((int64_t)1 << 32)));
    }

    // (behind choose_kernel) the register-staged kernel runs what is not the narrow one's
    void no_pipelined_kernel()
    {
        dma_idx = byte_idx = -1, splitk_plan = 1;
        kname_dma.clear();
        kname = kname_mfma;
    }

    // A, D and bias_f32 are device pointers here
    int run_dense(const int8_t *A, int64_t lda, int64_t a_bs, void *D, int64_t ldd, int64_t d_bs,
                  const float *bias_f32, hipStream_t s)
    {
        if (!prepared)
            return fail("run before prepare");
        GemmArgs g{};
        fill_epi(g.epi, bias_f32);
        bool flip_in_loader = flip_a;
        int  k_valid        = K;
        const bool direct =
            path == MI355_PATH_SIMPLE || ((((uintptr_t)A | (uintptr_t)lda | (uintptr_t)a_bs) & 3) == 0);
        // the per-row term b_offset * rowsum(A): the pipelined kernels sum the rows of A themselves while its tiles pass
        // through them (dword-aligned rows, K a whole number of 16-byte columns; under K slices every slice its part, which
        // the float epilogue could not take apart again); otherwise one pass over A
        // in front of the GEMM leaves the sums in a vector
        // (rows on any byte, or sums that stop inside a 16-byte column, without a pass in front: where the model prices the tile's
        // own shifting lower than the copy. run_noalloc keeps to the copy and with it to its limits)
        // (the pass: what 370 products took more than their tiles' price, mean error of both together 8 %. A workgroup walks along one row,
        // hence the term in K)
        // (sums alone, which copy nothing: the older fit of both sides, whose price of the tiles is about 0.82 of the present one)
        const double copy_us = direct ? std::max(2.5, 1.05 + (double)M * batch * K * 4.5e-7 + K * 0.49e-3)
                                      : 2.15 + (double)M * batch * (K + Kp) * 5.17e-7 + K * 0.46e-3;
        const bool   byte_rows = (!direct || (b_off_eff() != 0 && K % 16 != 0)) && ext_ws == nullptr && path == MI355_PATH_MFMA && byte_idx >= 0 &&
                               !(own_row_terms() && b_off_eff() != 0) && (int64_t)lda * 256 + K < ((int64_t)1 << 32) &&
                               (one_launch || us_bytes * (direct ? 0.82 : 1.0) < us_copied + copy_us);
        const bool rowsum_in_kernel = byte_rows ? b_off_eff() != 0 : b_off_eff() != 0 && direct && path == MI355_PATH_MFMA && dma_idx >= 0 && K % 16 == 0 && K >= 16 &&
                                      (splitk == 1 || epi != EPI_F32) && (int64_t)lda * 256 + K < ((int64_t)1 << 32);
        const bool need_rowvec = b_off_eff() != 0 && !rowsum_in_kernel;
        // the two workspaces of a run: owned by the handle and grown on demand, or carved out of a buffer the caller of
        // this function brings (ext_ws != nullptr: nothing is allocated, sizes beyond ext_ws_bytes are an error)
        const size_t rv_size  = (sizeof(int32_t) * (size_t)M * batch + 255) & ~(size_t)255;
        const size_t rv_bytes = need_rowvec && !own_row_terms() ? rv_size : 0;
        const size_t ap_bytes = direct || byte_rows ? 0 : (size_t)batch * M * Kp;
        int32_t     *rv       = nullptr;
        int8_t      *ap       = nullptr;
        if (ext_ws != nullptr)
        {
            if (rv_bytes + ap_bytes > 0 && ext_ws_busy)
                return fail("mi355_gemmlowp_run_noalloc: this GPU's workspace is still in use by a call on another stream");
            ext_ws_used = rv_bytes + ap_bytes > 0;
            if (rv_bytes + ap_bytes > ext_ws_bytes)
                return fail("this run needs %zu bytes of workspace (row sums %zu + padded copy of A %zu); the fixed "
                            "workspace holds %zu",
                            rv_bytes + ap_bytes, rv_bytes, ap_bytes, ext_ws_bytes);
            rv = (int32_t *)ext_ws, ap = (int8_t *)ext_ws + rv_bytes;
        }
        else
        {
            if (rv_bytes > 0)
                TRY(rowvec.ensure(rv_bytes));
            if (ap_bytes > 0)
                TRY(Ap.ensure(ap_bytes));
            // (sums inside the kernel now, by a pass where another A's rows start on dwords: a run that is recorded later finds the vector)
            if (byte_rows && b_off_eff() != 0 && rowvec.cap < rv_size && !capturing(s))
                TRY(rowvec.ensure(rv_size));
            rv = rowvec.as<int32_t>(), ap = Ap.as<int8_t>();
        }
        if (own_row_terms())
            rv = rowvec.as<int32_t>();
        g.byte_rows = byte_rows ? 1 : 0;
        if (!direct && !byte_rows)
        {
            // rows not dword aligned: padded, sign-normalised copy (and the row sums in the same pass)
            HIP_TRY(a_prepass_launch(A, lda, a_bs, batch, M, K, flip_a, ap, Kp, need_rowvec ? rv : nullptr, b_off_eff(), s));
            A = ap, lda = Kp, a_bs = (int64_t)M * Kp, k_valid = Kp, flip_in_loader = false;
        }
        else if (need_rowvec)
        {
            HIP_TRY(a_prepass_launch(A, lda, a_bs, batch, M, K, flip_a, nullptr, Kp, rv, b_off_eff(), s));
        }
        if (rowsum_in_kernel)
            g.epi.rowsum_mul = b_off_eff();
        if (need_rowvec)
            g.epi.rowvec = rv;
        else if (path == MI355_PATH_SKINNY)
            g.epi.rowvec = zeros.as<int32_t>();
        g.A = A, g.lda = lda, g.a_batch_stride = a_bs;
        g.Bp = Bp.as<int8_t>(), g.Kp = Kp, g.bp_batch_stride = b_shared ? 0 : (int64_t)Np * Kp;
        g.D = D, g.ldd = ldd, g.d_batch_stride = d_bs;
        g.M = M, g.N = N, g.K = k_valid;
        set_vec_store(g);
        return launch(g, flip_in_loader, false, s);
    }

    // 4 consecutive outputs of a row may leave as one store when every row start is aligned to 4 elements
    void set_vec_store(GemmArgs &g) const
    {
        const size_t esz = (epi == EPI_FIXEDPOINT) ? 1 : half_out ? 2 : 4;
        g.epi.vec_store  = (((uintptr_t)g.D % (4 * esz)) == 0 && g.ldd % 4 == 0 && g.d_batch_stride % 4 == 0) ? 1 : 0;
        g.epi.vec_store16 = (esz == 1 && ((uintptr_t)g.D % 16) == 0 && g.ldd % 16 == 0 && g.d_batch_stride % 16 == 0) ? 1 : 0;
    }

    // The row terms of a convolution by a pass over the source (rs_src, rs_geom: the caller's channel count), for the kernels
    // that do not sum the patches themselves
    int conv_row_terms(GemmArgs &g, hipStream_t s)
    {
        TRY(rowvec.ensure(sizeof(int32_t) * (size_t)M));
        HIP_TRY(conv_rowsum_launch(rs_src, rs_geom, M, flip_a, g.epi.rowsum_mul, rowvec.as<int32_t>(), s));
        g.epi.rowvec = rowvec.as<int32_t>(), g.epi.rowsum_mul = 0;
        return 0;
    }

    // Whether the kernel that launch() gives this convolution writes its 8-bit results as planes (EpiParams::planes) on request: the
    // pipelined one's tiles, whole K
    bool stores_planes(const GemmArgs &g) const
    {
        const int64_t span = (int64_t)((g.M + g.conv.OH * g.conv.OW - 1) / (g.conv.OH * g.conv.OW)) * g.conv.H * g.conv.W * g.conv.C;
        const bool    narrow = has_narrow && span < ((int64_t)1 << 31) && narrow_applies(g);
        return epi == EPI_FIXEDPOINT && path == MI355_PATH_MFMA && splitk == 1 && dma_idx > 0 && !narrow && g.conv.C % 16 == 0 &&
               ((uintptr_t)g.A & 15) == 0 && g.K % 16 == 0 && g.K >= 16 && span < ((int64_t)1 << 32);
    }

    int launch(GemmArgs &g, bool flip_in_loader, bool conv, hipStream_t s)
    {
        if (path == MI355_PATH_SIMPLE)
            HIP_TRY(simple_gemm_launch(epi, flip_in_loader, g, batch, s));
        else if (path == MI355_PATH_SKINNY)
        {
            GemmArgs gb        = g;
            gb.Bp              = Bs.as<int8_t>();
            gb.bp_batch_stride = b_shared ? 0 : (int64_t)Np * Kp;
            if (g.epi.rowvec == zeros.as<int32_t>() || g.epi.rowvec == nullptr)
                gb.epi.rowvec_batch_stride = 0;
            // A batch of small products (under 4 MiB of B each, where the launches themselves are what costs) goes out
            // as one launch with the entries along the grid; larger ones one launch per entry, each free to take the
            // form that stages its A once
            if (batch > 1 && (int64_t)Np * Kp <= ((int64_t)4 << 20) && batch <= 65535)
                HIP_TRY(skinny_launch(epi, flip_in_loader, gb, batch, s, &kname_static));
            else
                for (int b = 0; b < batch; ++b)
                {
                    GemmArgs ge = gb;
                    ge.A        = gb.A + (int64_t)b * gb.a_batch_stride;
                    ge.Bp       = gb.Bp + (int64_t)b * gb.bp_batch_stride;
                    ge.D        = (char *)gb.D + (int64_t)b * gb.d_batch_stride * (epi == EPI_FIXEDPOINT ? 1 : half_out ? 2 : 4);
                    ge.epi.colvec += (int64_t)b * gb.epi.colvec_batch_stride;
                    if (ge.epi.rowvec != nullptr)
                        ge.epi.rowvec += (int64_t)b * gb.epi.rowvec_batch_stride;
                    HIP_TRY(skinny_launch(epi, flip_in_loader, ge, 1, s, &kname_static, batch == 1 ? &sk_plan : nullptr));
                }
        }
        else
        {
            g.fill16 = fill.as<int8_t>();
            // the pipelined kernel moves 16-byte columns of dword-aligned rows straight into LDS
            const bool aligned = g.byte_rows != 0 ||
                (conv ? (g.conv.C % 16 == 0 && ((uintptr_t)g.A & 15) == 0 && g.K % 16 == 0)
                     : ((((uintptr_t)g.A | (uintptr_t)g.lda | (uintptr_t)g.a_batch_stride) & 3) == 0));
            g.a_end = conv ? nullptr : g.A + (int64_t)(batch - 1) * g.a_batch_stride + (int64_t)(g.M - 1) * g.lda + g.K;
            // its producers address a block's A rows (dense) or the whole image batch (convolution) with 32-bit offsets
            const int64_t span = conv ? (int64_t)((g.M + g.conv.OH * g.conv.OW - 1) / (g.conv.OH * g.conv.OW)) *
                                            g.conv.H * g.conv.W * g.conv.C
                                      : (int64_t)g.lda * 256 + g.K;
            // few output columns and a short K: every wave for itself, weights resident in LDS (gemm_narrow.hip)
            if (has_narrow && batch == 1 && conv && !g.epi.accumulate && span < ((int64_t)1 << 31) &&
                narrow_applies(g))
            {
                g.Bp            = Bn.as<int8_t>();
                g.conv.pad_word = 0x01010101u * fill_byte; // as in the image: the kernel flips what it loads
                bool band       = false;
                HIP_TRY(narrow_launch(epi, flip_in_loader, g, s, &band));
                kname_run = band ? &kname_band : &kname_narrow;
            }
            else if (dma_idx >= 0 && aligned && g.K >= 16 && span < ((int64_t)1 << 32))
            {
                const int        idx = g.byte_rows ? byte_idx : dma_idx;
                const MfmaConfig c   = dma_config(idx);
                g.tiles_m          = (g.M + c.BM - 1) / c.BM;
                g.tiles_n          = (g.N + c.BN - 1) / c.BN;
                kname_run          = g.byte_rows ? &kname_bytes : &kname_dma_full;
                if (conv)
                    g.conv.pad_word = 0x01010101u * fill_byte; // as in the image: the kernel flips what it loads
                if (splitk > 1 && batch == 1)
                {
                    // the float epilogue rounds the product and the offset terms apart: they must not meet in the planes
                    if (conv && epi == EPI_F32 && g.epi.rowsum_mul != 0)
                        TRY(conv_row_terms(g, s));
                    const int64_t kc = (int64_t)(((K + c.BK - 1) / c.BK + splitk - 1) / splitk) * c.BK;
                    GemmArgs      gp = g;
                    // (dense: a slice starts kc bytes into every row of A; convolution: kc values into every patch,
                    // which the loader adds to the k it decodes)
                    // (g.K: K, or K padded to whole steps where the rows of A were copied)
                    gp.a_batch_stride = conv ? 0 : kc, gp.bp_batch_stride = kc, gp.k_slice = (int32_t)kc;
                    gp.epi.colvec_batch_stride = gp.epi.rowvec_batch_stride = 0, gp.d_batch_stride = 0;
                    kname_run = &kname_splitk;
                    if (idx > 0 && !g.byte_rows)
                    {
                        gp.slices = splitk, gp.arrived = arrived.as<int32_t>(), gp.parts = sums_at >= 0 ? gp.arrived + sums_at : parts.as<int32_t>();
                        HIP_TRY(dma_launch(idx, epi, flip_in_loader, conv, gp, splitk, s));
                        return 0;
                    }
                    // 256 x 128 tiles, where the caller names them, and rows on any byte: a second launch sums the slices' planes
                    const int ldp              = (N + 3) & ~3;
                    gp.epi                     = EpiParams{};
                    gp.epi.colvec              = zerocol.as<int32_t>();
                    gp.epi.vec_store           = 1;
                    gp.epi.rowsum_mul          = g.epi.rowsum_mul; // every slice adds its own part of the row terms
                    gp.D = parts.as<int32_t>(), gp.ldd = ldp, gp.d_batch_stride = (int64_t)M * ldp;
                    HIP_TRY(dma_launch(idx, EPI_S32, flip_in_loader, conv, gp, splitk, s));
                    HIP_TRY(splitk_finish_launch(epi, g, parts.as<int32_t>(), (int64_t)M * ldp, ldp, splitk, s));
                    return 0;
                }
                HIP_TRY(dma_launch(idx, epi, flip_in_loader, conv, g, batch, s));
            }
            else
            {
                const MfmaConfig c = mfma_config(cfg_idx);
                g.tiles_m          = (g.M + c.BM - 1) / c.BM;
                g.tiles_n          = (g.N + c.BN - 1) / c.BN;
                kname_run          = &kname_mfma_full;
                if (conv && g.epi.rowsum_mul != 0)
                    TRY(conv_row_terms(g, s));
                if (conv)
                    g.conv.pad_word = (0x01010101u * fill_byte) ^ (flip_in_loader ? 0x80808080u : 0u);
                HIP_TRY(mfma_launch(cfg_idx, epi, flip_in_loader, conv, g, batch, s));
            }
        }
        return 0;
    }
};

int check_requant(const mi355_requant &rq, int dst_dtype)
{
    if (rq.min_bound > rq.max_bound)
        return fail("min_bound > max_bound");
    if (rq.stage != MI355_STAGE_FIXEDPOINT && rq.stage != MI355_STAGE_SCALE)
        return fail("unknown output stage %d", rq.stage);
    if (rq.stage == MI355_STAGE_SCALE && !rq.per_channel && (rq.shift < 0 || rq.shift > 31))
        return fail("QUANTIZE_DOWN needs a shift in [0, 31] (got %d)", rq.shift);
    // Bounds inside the destination type's range clamp; bounds that cover it only saturate. Bounds with one end inside
    // and one outside are refused: the reference's three implementations disagree there (the stand-alone kernel narrows
    // the bound to 8 bits, src/cpu/kernels/CpuGemmLowpOffsetContributionOutputStageKernel.cpp:502-503; the assembly path
    // clamps in int32 and keeps the low byte, src/core/NEON/kernels/arm_gemm/quantized.cpp:36-46,254-261)
    const int32_t tlo = dst_dtype == MI355_S8 ? -128 : 0, thi = dst_dtype == MI355_S8 ? 127 : 255;
    const bool    covers = rq.min_bound <= tlo && rq.max_bound >= thi;
    const bool    inside = rq.min_bound >= tlo && rq.max_bound <= thi;
    if (!covers && !inside)
        return fail("clamp bounds [%d,%d] are partly outside the destination type's range [%d,%d]", rq.min_bound,
                    rq.max_bound, tlo, thi);
    return 0;
}
} // namespace

struct mi355_gemm_handle
{
    mi355_gemm_desc d;
    GemmCore        core;
    DevBuf          stageA, stageB, stageD, stageBiasF, stageBias, stageMult, stageShift;
    DevBuf          wsF32; // MI355_F16 destination: the dense F32 matrix the kernels write
    DevBuf          denseA, denseD; // matrices handed over as planes with gaps between them, without the gaps
    PtrKind         kindA, kindD, kindBiasF; // host or device memory, per argument of run()
    bool a_planes() const { return d.a_plane_rows > 0 && d.a_plane_stride != (int64_t)d.a_plane_rows * d.lda; }
    bool d_planes() const { return d.d_plane_rows > 0 && d.d_plane_stride != (int64_t)d.d_plane_rows * d.ldd; }
};

static int check_planes(const mi355_gemm_desc &d)
{
    if (d.a_plane_rows < 0 || d.d_plane_rows < 0 || (d.a_plane_rows > 0 && d.M % d.a_plane_rows != 0) ||
        (d.d_plane_rows > 0 && d.M % d.d_plane_rows != 0))
        return fail("plane_rows must divide M");
    if (d.a_plane_rows > 0 && d.a_plane_stride < (int64_t)(d.a_plane_rows - 1) * d.lda + d.K)
        return fail("A plane stride smaller than one plane");
    if (d.d_plane_rows > 0 && d.d_plane_stride < (int64_t)(d.d_plane_rows - 1) * d.ldd + d.N)
        return fail("D plane stride smaller than one plane");
    return 0;
}

// bytes (A) / elements (D) from the first element of a batch entry's matrix to one past its last
static int64_t a_span(const mi355_gemm_desc &d)
{
    return d.a_plane_rows > 0 ? (int64_t)(d.M / d.a_plane_rows - 1) * d.a_plane_stride + (int64_t)(d.a_plane_rows - 1) * d.lda + d.K
                              : (int64_t)(d.M - 1) * d.lda + d.K;
}
static int64_t d_span(const mi355_gemm_desc &d)
{
    return d.d_plane_rows > 0 ? (int64_t)(d.M / d.d_plane_rows - 1) * d.d_plane_stride + (int64_t)(d.d_plane_rows - 1) * d.ldd + d.N
                              : (int64_t)(d.M - 1) * d.ldd + d.N;
}

struct mi355_conv_handle
{
    mi355_conv_desc d;
    GemmCore        core;
    ConvGeom        geom;
    bool            implicit = false;
    DevBuf          stageSrc, stageW, stageDst, stageBias, stageMult, stageShift, cols;
    DevBuf          nhwcSrc, nhwcW, nhwcDst; // MI355_NCHW: the tensors in the kernels' layout
    DevBuf          denseSrc, denseW, denseDst; // tensors that came with gaps, without them
    DevBuf          biasF;                   // F32 destination: the float bias
    bool            has_bias_f32 = false;
    int             c_pad = 0;               // > 0: the kernels see this many channels (source and weights padded, see create)
    ConvGeom        geom_true;               // ... and the geometry with the caller's channel count, for the patches' row sums
    bool            patch_rows = false;      // ... one pixel being the KW taps of a patch row
    bool            raw_rows = false;        // ... whose kernel takes them from the caller's image where there is no weights offset
    DevBuf          padSrc, padW;
    PtrKind         kindSrc, kindDst; // host or device memory, per argument of run()
    bool       window_made = false, window = false; // gemm_window.hip runs it: decided at create; with the present offsets
    WindowPlan window_plan;
    bool       from_window() const { return window && core.rq.stage == MI355_STAGE_FIXEDPOINT; }
    // how it is divided (which depends on whether there is a weights offset)
    bool divide_window()
    {
        return conv_window_plan(geom_true, d.batch, d.OFM, d.layout == MI355_NCHW, core.b_off_eff() != 0, num_cus(), window_plan);
    }
    bool choose_window()
    {
        const bool planes = d.layout == MI355_NCHW;
        if (d.path != MI355_CONV_AUTO || core.epi != EPI_FIXEDPOINT || raw_rows || !divide_window())
            return false;
        // (the narrow kernel needs no copy and starts half a microsecond earlier: 18 x 18 x 48 -> 24, 1 x 1: 3.6 us, 4.3 here. Several of its panels are up
        // to a fifth slower: 21 x 24 x 24 x 16 -> 88, 3 x 3 stride 2: 5.4, 4.6)
        if (!planes && (c_pad == 0 || patch_rows) && core.narrow_form())
            return false;
        // (register-staged tiles, which run what the pipelined kernel does not take, look every byte up)
        const double tiles_us = core.dma_idx >= 0 ? core.us_dma : 1e9;
        return conv_window_pays(window_plan.us, conv_other_us(geom_true, d.batch, d.OFM, core.K, planes, core.b_off_eff() != 0, c_pad > 0, core.narrow_form(), tiles_us, num_cus()),
                                !planes && c_pad == 0 && core.splitk_plan > 1);
    }
    bool   from_image() const { return raw_rows && core.b_off_eff() == 0 && core.rq.stage == MI355_STAGE_FIXEDPOINT; }
    size_t pad_bytes() const { return (size_t)d.batch * d.H * geom.W * c_pad; }
};

extern "C"
{
const char *mi355_last_error(void)
{
    return g_err.c_str();
}

int mi355_device_info(char *name, size_t name_len)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
    {
        (void)hipGetLastError();
        fail("no HIP device");
        return -1;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess)
    {
        fail("hipGetDeviceProperties failed");
        return -1;
    }
    if (name && name_len)
    {
        strncpy(name, prop.gcnArchName, name_len - 1);
        name[name_len - 1] = 0;
    }
    return prop.multiProcessorCount;
}

int mi355_gemmlowp_create(const mi355_gemm_desc *desc, mi355_gemm_handle **out)
{
    if (!desc || !out)
        return fail("null argument");
    const mi355_gemm_desc &d = *desc;
    if (d.M < 1 || d.N < 1 || d.K < 1 || d.batch < 1)
        return fail("M, N, K, batch must be positive (got %d %d %d %d)", d.M, d.N, d.K, d.batch);
    if (!is_8bit(d.a_dtype) || !is_8bit(d.b_dtype))
        return fail("A and B must be 8-bit");
    if (d.lda < d.K || d.ldb < (d.b_transposed ? d.K : d.N) || d.ldd < d.N)
        return fail("row stride smaller than the row");
    if (d.b_k_interleave < 0 || (d.b_k_interleave > 1 && d.K % d.b_k_interleave != 0))
        return fail("b_k_interleave must divide K");
    switch (d.epilogue)
    {
        case MI355_EPI_S32:
            if (d.dst_dtype != MI355_S32)
                return fail("S32 epilogue needs an S32 destination");
            break;
        case MI355_EPI_FIXEDPOINT:
            if (!is_8bit(d.dst_dtype))
                return fail("FIXEDPOINT epilogue needs an 8-bit destination");
            if (check_requant(d.requant, d.dst_dtype))
                return 1;
            break;
        case MI355_EPI_F32:
            if (d.dst_dtype != MI355_F32 && d.dst_dtype != MI355_F16)
                return fail("F32 epilogue needs an F32 or F16 destination");
            break;
        default:
            return fail("unknown epilogue %d", d.epilogue);
    }
    if ((d.flags & ~(MI355_GEMM_ACCUMULATE | MI355_GEMM_ACT_TWICE)) != 0)
        return fail("unknown flag bits 0x%x", d.flags);
    if ((d.flags & MI355_GEMM_ACCUMULATE) && d.epilogue == MI355_EPI_FIXEDPOINT)
        return fail("accumulation is only possible into an S32 or F32 destination");
    TRY(check_planes(d));
    if (d.batch > 1 && (d.a_batch_stride < a_span(d) || d.d_batch_stride < d_span(d)))
        return fail("batch stride smaller than one matrix");
    if (d.batch > 1 && d.b_batch_stride != 0 &&
        d.b_batch_stride < (d.b_transposed ? (int64_t)(d.N - 1) * d.ldb + d.K : (int64_t)(d.K - 1) * d.ldb + d.N))
        return fail("B batch stride smaller than one matrix");
    mi355_gemm_handle *h = new (std::nothrow) mi355_gemm_handle();
    if (!h)
        return fail("out of host memory");
    h->d        = d;
    GemmCore &c = h->core;
    c.M = d.M, c.N = d.N, c.K = d.K, c.batch = d.batch;
    c.epi = d.epilogue, c.dst_dtype = d.dst_dtype;
    c.flip_a = d.a_dtype == MI355_U8, c.flip_b = d.b_dtype == MI355_U8;
    c.a_offset = d.a_offset, c.b_offset = d.b_offset;
    c.rq = d.requant, c.scale = d.scale, c.act_min = d.act_min, c.act_max = d.act_max;
    c.path     = d.path;
    c.accumulate = (d.flags & MI355_GEMM_ACCUMULATE) != 0, c.act_twice = (d.flags & MI355_GEMM_ACT_TWICE) != 0;
    c.b_shared = d.batch == 1 || d.b_batch_stride == 0;
    c.byte_lda = ((d.lda | (d.batch > 1 ? d.a_batch_stride : 0)) & 3) != 0;
    if (c.choose_kernel())
    {
        delete h;
        return 1;
    }
    *out = h;
    return 0;
}

int mi355_gemmlowp_prepare(mi355_gemm_handle *h, const void *B, const int32_t *bias, const int32_t *mult,
                           const int32_t *shift, void *stream)
{
    if (!h || !B)
        return fail("null argument");
    hipStream_t            s = (hipStream_t)stream;
    GemmCore              &c = h->core;
    const mi355_gemm_desc &d = h->d;
    const int              nb = c.nb();
    const size_t           b_bytes = (size_t)(nb - 1) * d.b_batch_stride +
                           (d.b_transposed ? (size_t)(d.N - 1) * d.ldb + d.K : (size_t)(d.K - 1) * d.ldb + d.N);
    const void            *Bd, *biasd, *multd, *shiftd;
    // Staging buffers are reused by later calls and managed memory is written by the host, so what was read from them has to
    // be read before this returns; and a first prepare ends with the handle's own set-up done. After that, preparing a new B
    // on the legacy default stream only enqueues (see prepare_enqueued) - unless there may be a graph with a run in it:
    // nothing of this library is called when it is launched, so nothing could wait.
    bool wait = s != nullptr || !c.prepared || c.recorded;
    TRY(to_device(B, b_bytes, h->stageB, s, &Bd, nullptr, &wait));
    TRY(to_device(bias, sizeof(int32_t) * d.N, h->stageBias, s, &biasd, nullptr, &wait));
    TRY(to_device(c.rq.per_channel ? mult : nullptr, sizeof(int32_t) * d.N, h->stageMult, s, &multd, nullptr, &wait));
    TRY(to_device(c.rq.per_channel ? shift : nullptr, sizeof(int32_t) * d.N, h->stageShift, s, &shiftd, nullptr, &wait));
    TRY(c.wait_for_prepare(s));
    TRY(c.pack(Bd, d.ldb, nb > 1 ? d.b_batch_stride : 0, d.b_transposed != 0, d.b_k_interleave, (const int32_t *)biasd, s));
    TRY(c.finish_prepare((const int32_t *)multd, (const int32_t *)shiftd, s));
    if (!wait)
        return c.prepare_enqueued();
    HIP_TRY(hipStreamSynchronize(s));
    c.prep_pending = false, c.prepared = true;
    return 0;
}

int mi355_gemmlowp_update_quant(mi355_gemm_handle *h, int32_t a_offset, int32_t b_offset, const mi355_requant *requant,
                                float scale, void *stream)
{
    if (!h)
        return fail("null argument");
    GemmCore &c = h->core;
    if (requant)
    {
        if (c.epi == EPI_FIXEDPOINT && check_requant(*requant, c.dst_dtype))
            return 1;
        if (requant->per_channel != c.rq.per_channel)
            return fail("update cannot switch between per-tensor and per-channel requantisation");
        c.rq = *requant;
    }
    c.a_offset = a_offset, c.b_offset = b_offset, c.scale = scale;
    h->d.a_offset = a_offset, h->d.b_offset = b_offset, h->d.scale = scale;
    if (!c.prepared)
        return 0;
    // behind a prepare that is still running elsewhere: it writes the column sums that are read here, and terms of its own
    // (with the offsets from before) over the ones that are written here
    hipStream_t s = (hipStream_t)stream;
    if (s != nullptr)
        TRY(c.prepare_over());
    c.keep_flags(s);
    TRY(c.refresh_colvec(s));
    TRY(c.refresh_qparams(s));
    c.keep_flags(s);
    return c.prep_pending ? c.prepare_enqueued() : 0; // a run on another stream comes behind both
}

static int set_gemm_strides(mi355_gemm_handle *h, int64_t lda, int64_t ldb, int64_t ldd, int64_t a_batch_stride,
                            int64_t b_batch_stride, int64_t d_batch_stride, int64_t a_plane_stride, int64_t d_plane_stride)
{
    const mi355_gemm_desc &d = h->d;
    if (lda < d.K || ldb < (d.b_transposed ? d.K : d.N) || ldd < d.N)
        return fail("row stride smaller than the row");
    mi355_gemm_desc n = d;
    n.lda = lda, n.ldb = ldb, n.ldd = ldd;
    n.a_plane_stride = a_plane_stride, n.d_plane_stride = d_plane_stride;
    n.a_batch_stride = a_batch_stride, n.b_batch_stride = b_batch_stride, n.d_batch_stride = d_batch_stride;
    TRY(check_planes(n));
    if (d.batch > 1 && (a_batch_stride < a_span(n) || d_batch_stride < d_span(n)))
        return fail("batch stride smaller than one matrix");
    if (d.batch > 1 && (b_batch_stride == 0) != h->core.b_shared)
        return fail("set_strides cannot switch between one shared B and one B per batch entry");
    if (d.batch > 1 && b_batch_stride != 0 &&
        b_batch_stride < (d.b_transposed ? (int64_t)(d.N - 1) * ldb + d.K : (int64_t)(d.K - 1) * ldb + d.N))
        return fail("B batch stride smaller than one matrix");
    h->d = n;
    return 0;
}

int mi355_gemmlowp_set_strides(mi355_gemm_handle *h, int64_t lda, int64_t ldb, int64_t ldd, int64_t a_batch_stride,
                               int64_t b_batch_stride, int64_t d_batch_stride)
{
    if (!h)
        return fail("null argument");
    // planes keep following one another without a gap under the new row strides
    return set_gemm_strides(h, lda, ldb, ldd, a_batch_stride, b_batch_stride, d_batch_stride,
                            (int64_t)h->d.a_plane_rows * lda, (int64_t)h->d.d_plane_rows * ldd);
}

int mi355_gemmlowp_set_strides_3d(mi355_gemm_handle *h, int64_t lda, int64_t ldb, int64_t ldd, int64_t a_batch_stride,
                                  int64_t b_batch_stride, int64_t d_batch_stride, int64_t a_plane_stride,
                                  int64_t d_plane_stride)
{
    if (!h)
        return fail("null argument");
    return set_gemm_strides(h, lda, ldb, ldd, a_batch_stride, b_batch_stride, d_batch_stride, a_plane_stride, d_plane_stride);
}

int mi355_gemmlowp_run(mi355_gemm_handle *h, const void *A, const float *bias_f32, void *D, void *stream)
{
    if (!h || !A || !D)
        return fail("null argument");
    hipStream_t            s = (hipStream_t)stream;
    GemmCore              &c = h->core;
    const mi355_gemm_desc &d = h->d;
    if (bias_f32 && c.epi != EPI_F32)
        return fail("float bias is only valid with the F32 epilogue");
    const bool   f16     = d.dst_dtype == MI355_F16;
    const size_t esz     = d.dst_dtype == MI355_S32 || d.dst_dtype == MI355_F32 ? 4 : (f16 ? 2 : 1);
    const size_t a_bytes = (size_t)(d.batch - 1) * d.a_batch_stride + (size_t)a_span(d);
    const size_t d_elems = (size_t)(d.batch - 1) * d.d_batch_stride + (size_t)d_span(d);
    const void  *Ad, *bfd;
    TRY(c.wait_for_prepare(s));
    TRY(to_device(A, a_bytes, h->stageA, s, &Ad, &h->kindA));
    TRY(to_device(bias_f32, sizeof(float) * d.N, h->stageBiasF, s, &bfd, &h->kindBiasF));
    const bool d_host = !h->kindD.is_device(D);
    void      *Dd     = D;
    if (d_host)
    {
        TRY(h->stageD.ensure(d_elems * esz));
        Dd = h->stageD.p;
        if (c.accumulate || d.ldd != d.N || h->d_planes() || (d.batch > 1 && d.d_batch_stride != (int64_t)d.M * d.ldd))
            HIP_TRY(hipMemcpyAsync(Dd, D, d_elems * esz, hipMemcpyHostToDevice, s)); // previous values / padding
    }
    const bool staged_in = Ad != A || bfd != bias_f32;
    // planes with gaps between them: the kernels see dense copies
    int64_t lda = d.lda, a_bs = d.a_batch_stride, ldd = d.ldd, d_bs = d.d_batch_stride;
    void   *Dplanes = nullptr;
    if (h->a_planes())
    {
        const int64_t row = round_up(d.K, 16);
        TRY(h->denseA.ensure((size_t)d.batch * d.M * row));
        HIP_TRY(restride_nd_launch(Ad, h->denseA.p, d.K, d.a_plane_rows, d.M / d.a_plane_rows, d.batch,
                                   RestrideSteps{{d.lda, d.a_plane_stride, d.a_batch_stride}},
                                   RestrideSteps{{row, row * d.a_plane_rows, row * d.M}}, s));
        Ad = h->denseA.p, lda = row, a_bs = row * d.M;
    }
    const RestrideSteps d_given{{d.ldd * (int64_t)esz, d.d_plane_stride * (int64_t)esz, d.d_batch_stride * (int64_t)esz}};
    const RestrideSteps d_dense{{d.N * (int64_t)esz, d.N * (int64_t)esz * d.d_plane_rows, d.N * (int64_t)esz * d.M}};
    if (h->d_planes())
    {
        TRY(h->denseD.ensure((size_t)d.batch * d.M * d.N * esz));
        Dplanes = Dd, Dd = h->denseD.p, ldd = d.N, d_bs = (int64_t)d.M * d.N;
        if (c.accumulate) // the previous values
            HIP_TRY(restride_nd_launch(Dplanes, Dd, (int)(d.N * esz), d.d_plane_rows, d.M / d.d_plane_rows, d.batch, d_given, d_dense, s));
    }
    if (f16 && c.rounds_to_half(lda))
    {
        c.half_out   = true;
        const int rc = c.run_dense((const int8_t *)Ad, lda, a_bs, Dd, ldd, d_bs, (const float *)bfd, s);
        c.half_out   = false;
        if (rc)
            return rc;
    }
    else if (f16)
    {
        // Accumulating, and where a fallback kernel runs: a dense F32 matrix, rounded into the half destination afterwards. Accumulating:
        // the addition (and the activation, which has to follow it) happens in that second step, on halfs.
        TRY(h->wsF32.ensure(sizeof(float) * (size_t)d.batch * d.M * d.N));
        float      *ws  = h->wsF32.as<float>();
        const bool  acc = c.accumulate, twice = c.act_twice;
        const float lo = c.act_min, hi = c.act_max;
        if (acc)
            c.accumulate = false, c.act_twice = false, c.act_min = -INFINITY, c.act_max = INFINITY;
        const int rc = c.run_dense((const int8_t *)Ad, lda, a_bs, ws, d.N, (int64_t)d.M * d.N, (const float *)bfd, s);
        c.accumulate = acc, c.act_twice = twice, c.act_min = lo, c.act_max = hi;
        if (rc)
            return rc;
        HIP_TRY(f32_to_f16_launch(ws, Dd, d.batch, d.M, d.N, ldd, d_bs, acc, lo, hi, s));
    }
    else
        TRY(c.run_dense((const int8_t *)Ad, lda, a_bs, Dd, ldd, d_bs, (const float *)bfd, s));
    if (Dplanes)
    {
        HIP_TRY(restride_nd_launch(Dd, Dplanes, (int)(d.N * esz), d.d_plane_rows, d.M / d.d_plane_rows, d.batch, d_dense, d_given, s));
        Dd = Dplanes;
    }
    if (d_host)
    {
        HIP_TRY(hipMemcpyAsync(D, Dd, d_elems * esz, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    else if (staged_in)
        HIP_TRY(hipStreamSynchronize(s)); // staged inputs must be consumed before the caller may reuse them
    return 0;
}

// Per GPU: the address of its copy of the workspace array, asked once (with that device current), and an event behind
// the last call's kernels, created in the same set-up step. Calls on one stream are ordered by the stream; a call that
// arrives on another stream while the event is still pending would overwrite the workspace under running kernels and
// is refused.
struct NoallocState
{
    void       *ptr      = nullptr;
    hipEvent_t  done     = nullptr;
    hipStream_t last     = nullptr;
    bool        recorded = false;
};
static std::mutex g_noalloc_mutex;
static int noalloc_state(NoallocState **out)
{
    static NoallocState states[64];
    int                 dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64)
        return fail("device index %d out of range", dev);
    NoallocState &st = states[dev];
    if (st.ptr == nullptr)
    {
        void *p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr)
            return fail("hipGetSymbolAddress returned no address for the workspace");
        HIP_TRY(hipEventCreateWithFlags(&st.done, hipEventDisableTiming));
        st.ptr = p;
    }
    *out = &st;
    return 0;
}

size_t mi355_gemmlowp_noalloc_workspace_bytes(void)
{
    return MI355_NOALLOC_SCRATCH_BYTES;
}

int mi355_gemmlowp_run_noalloc(mi355_gemm_handle *h, const void *A, const float *bias_f32, void *D, void *stream)
{
    if (!h || !A || !D)
        return fail("null argument");
    hipStream_t            s = (hipStream_t)stream;
    GemmCore              &c = h->core;
    const mi355_gemm_desc &d = h->d;
    if (!c.prepared)
        return fail("run before prepare");
    if (bias_f32 && c.epi != EPI_F32)
        return fail("float bias is only valid with the F32 epilogue");
    if (d.dst_dtype == MI355_F16)
        return fail("mi355_gemmlowp_run_noalloc does not write F16 destinations (some need a float matrix as workspace)");
    if (h->a_planes() || h->d_planes())
        return fail("mi355_gemmlowp_run_noalloc does not take planes with gaps between them (they need dense copies)");
    if (!h->kindA.is_device(A) || !h->kindD.is_device(D) || (bias_f32 && !h->kindBiasF.is_device(bias_f32)))
        return fail("mi355_gemmlowp_run_noalloc takes device memory only");
    std::lock_guard<std::mutex> lock(g_noalloc_mutex);
    NoallocState               *st = nullptr;
    TRY(noalloc_state(&st));
    // (a stream under graph capture records no event and is not checked: the graph's own order is the caller's)
    const bool tracked = !GemmCore::capturing(s);
    if (tracked && st->recorded && st->last != s)
    {
        const hipError_t q = hipEventQuery(st->done);
        if (q == hipErrorNotReady)
        {
            (void)hipGetLastError();
            c.ext_ws_busy = true; // an error if this run needs the workspace at all
        }
        else
            HIP_TRY(q);
    }
    TRY(c.wait_for_prepare(s));
    c.ext_ws = st->ptr, c.ext_ws_bytes = MI355_NOALLOC_SCRATCH_BYTES, c.ext_ws_used = false;
    const int  rc   = c.run_dense((const int8_t *)A, d.lda, d.a_batch_stride, D, d.ldd, d.d_batch_stride, bias_f32, s);
    const bool used = c.ext_ws_used;
    c.ext_ws = nullptr, c.ext_ws_bytes = 0, c.ext_ws_busy = false;
    if (tracked && used && rc == 0)
    {
        HIP_TRY(hipEventRecord(st->done, s));
        st->last = s, st->recorded = true;
    }
    return rc;
}

void mi355_gemmlowp_destroy(mi355_gemm_handle *h)
{
    if (!h)
        return;
    h->core.release();
    h->stageA.release(), h->stageB.release(), h->stageD.release(), h->stageBiasF.release(), h->stageBias.release();
    h->stageMult.release(), h->stageShift.release(), h->wsF32.release(), h->denseA.release(), h->denseD.release();
    delete h;
}

const char *mi355_gemmlowp_kernel_name(const mi355_gemm_handle *h)
{
    return h ? h->core.name() : "";
}

int mi355_output_stage_run(const mi355_output_stage_desc *desc, const int32_t *src, const int32_t *bias, void *dst,
                           void *stream)
{
    if (!desc || !src || !dst)
        return fail("null argument");
    const mi355_output_stage_desc &d = *desc;
    if (d.M < 1 || d.N < 1 || d.ld_src < d.N || d.ld_dst < d.N)
        return fail("bad output-stage shape");
    const bool s16 = d.dst_dtype == MI355_S16;
    if (!is_8bit(d.dst_dtype) && !s16)
        return fail("output stage writes QASYMM8, QASYMM8_SIGNED or QSYMM16");
    if (d.requant.per_channel)
        return fail("the stand-alone output stage is per-tensor");
    if (s16)
    {
        if (d.requant.stage != MI355_STAGE_FIXEDPOINT || d.requant.result_offset != 0)
            return fail("the QSYMM16 output stage is QUANTIZE_DOWN_FIXEDPOINT without a result offset");
        if (d.requant.min_bound > d.requant.max_bound)
            return fail("min_bound > max_bound");
        // the reference narrows the bounds to int16 with a plain cast: only bounds that survive it are meaningful
        const bool whole = d.requant.min_bound <= -32768 && d.requant.max_bound >= 32767;
        if (!whole && (d.requant.min_bound < -32768 || d.requant.max_bound > 32767))
            return fail("QSYMM16 clamp bounds [%d,%d] are partly outside the int16 range", d.requant.min_bound,
                        d.requant.max_bound);
    }
    else if (check_requant(d.requant, d.dst_dtype))
        return 1;
    const size_t desz = s16 ? 2 : 1;
    hipStream_t s = (hipStream_t)stream;
    DevBuf      sSrc, sBias, sDst;
    const void *srcd, *biasd;
    const size_t s_elems = (size_t)(d.M - 1) * d.ld_src + d.N, d_elems = (size_t)(d.M - 1) * d.ld_dst + d.N;
    int          rc      = 0;
    void        *Dd      = dst;
    const bool   d_host  = !is_device_ptr(dst);
    EpiParams    p{};
    p.mult_s = d.requant.multiplier, p.shift_s = d.requant.shift, p.result_offset = d.requant.result_offset;
    p.stage  = d.requant.stage;
    const int32_t tlo = s16 ? -32768 : d.dst_dtype == MI355_S8 ? -128 : 0, thi = s16 ? 32767 : d.dst_dtype == MI355_S8 ? 127 : 255;
    p.lo = d.requant.min_bound > tlo ? d.requant.min_bound : tlo;
    p.hi = d.requant.max_bound < thi ? d.requant.max_bound : thi;
    auto body = [&]() -> int
    {
        TRY(to_device(src, s_elems * 4, sSrc, s, &srcd));
        TRY(to_device(bias, sizeof(int32_t) * d.N, sBias, s, &biasd));
        if (d_host)
        {
            TRY(sDst.ensure(d_elems * desz));
            Dd = sDst.p;
            if (d.ld_dst != d.N)
                HIP_TRY(hipMemcpyAsync(Dd, dst, d_elems * desz, hipMemcpyHostToDevice, s));
        }
        if (s16)
            HIP_TRY(output_stage_s16_launch((const int32_t *)srcd, d.ld_src, (const int32_t *)biasd, Dd, d.ld_dst, d.M, d.N, p, s));
        else
            HIP_TRY(output_stage_launch((const int32_t *)srcd, d.ld_src, (const int32_t *)biasd, Dd, d.ld_dst, d.M, d.N, p, s));
        if (d_host)
            HIP_TRY(hipMemcpyAsync(dst, Dd, d_elems * desz, hipMemcpyDeviceToHost, s));
        if (d_host || srcd != src || biasd != bias)
            HIP_TRY(hipStreamSynchronize(s));
        return 0;
    };
    rc = body();
    sSrc.release(), sBias.release(), sDst.release();
    return rc;
}

static void conv_geom(const mi355_conv_desc &d, ConvGeom &g)
{
    g.H = d.H, g.W = d.W, g.C = d.C, g.KH = d.KH, g.KW = d.KW;
    g.stride_x = d.stride_x, g.stride_y = d.stride_y, g.pad_left = d.pad_left, g.pad_top = d.pad_top;
    g.dil_x = d.dilation_x, g.dil_y = d.dilation_y;
    // FLOOR rounding of PadStrideInfo (src/core/Utils.cpp:288-332)
    int w = (int)std::floor((float)(d.W + d.pad_left + d.pad_right - (d.dilation_x * (d.KW - 1) + 1)) / (float)d.stride_x + 1.f);
    int h = (int)std::floor((float)(d.H + d.pad_top + d.pad_bottom - (d.dilation_y * (d.KH - 1) + 1)) / (float)d.stride_y + 1.f);
    g.OW = w < 1 ? 1 : w;
    g.OH = h < 1 ? 1 : h;
    auto magic = [](int32_t dv) -> uint32_t { return dv == 1 ? 0u : (uint32_t)(((uint64_t)1 << 32) / (uint64_t)dv) + 1u; };
    g.magic_C = magic(g.C), g.magic_KW = magic(g.KW), g.magic_OW = magic(g.OW), g.magic_OH = magic(g.OH);
}

// the implicit-GEMM loader divides by C, KW, OW and OH with 32-bit reciprocal multiplies: exact while x * d < 2^32
static bool conv_fast_div_ok(const mi355_conv_desc &d, const ConvGeom &g)
{
    const int64_t M = (int64_t)d.batch * g.OH * g.OW, K = (int64_t)d.KH * d.KW * d.C, lim = (int64_t)1 << 32;
    return M * g.OW < lim && (M / g.OW + 1) * g.OH < lim && (K + 256) * d.C < lim && ((int64_t)d.KH * d.KW + 256) * d.KW < lim;
}

// The ring kernel's loader works a tap's offset out with 24-bit factors (an image row's bytes and a dilated filter's extent among them)
// and puts what lies beyond K 2^30 rows down, outside any image.
static bool conv_taps_ok(const ConvGeom &g)
{
    const int64_t lim = (int64_t)1 << 24;
    return (int64_t)g.KH * g.KW < lim && g.C < lim && (int64_t)(g.KH - 1) * g.dil_y < lim && (int64_t)(g.KW - 1) * g.dil_x < lim &&
           (g.KH == 1 || (int64_t)g.W * g.C < lim) && g.H < (1 << 29) && g.pad_top < (1 << 29);
}

void mi355_conv_out_dims(const mi355_conv_desc *desc, int32_t *OH, int32_t *OW)
{
    ConvGeom g{};
    conv_geom(*desc, g);
    if (OH)
        *OH = g.OH;
    if (OW)
        *OW = g.OW;
}

// One tensor of a convolution as runs of contiguous bytes: seg bytes per run, n1 x n2 x n3 runs along dimensions 1..3 of
// the tensor, 'given' the caller's byte strides of those dimensions (0 resolved to "no gap"), 'dense' the gap-free ones
struct ConvTensorSteps
{
    int           seg = 0;
    int64_t       n1 = 0, n2 = 0, n3 = 0;
    RestrideSteps given{}, dense{};
    bool          padded = false;
    size_t        extent = 0, bytes = 0; // bytes spanned from the first element with and without the gaps
};

static int conv_tensor_steps(const char *name, int64_t seg, int64_t n1, int64_t n2, int64_t n3, int64_t s1, int64_t s2,
                             int64_t s3, ConvTensorSteps &t)
{
    const int64_t g1 = s1 ? s1 : seg, g2 = s2 ? s2 : g1 * n1, g3 = s3 ? s3 : g2 * n2;
    if (g1 < seg || g2 < g1 * n1 || g3 < g2 * n2)
        return fail("%s: a stride is smaller than what it steps over", name);
    t.seg = (int)seg, t.n1 = n1, t.n2 = n2, t.n3 = n3;
    t.given  = RestrideSteps{{g1, g2, g3}};
    t.dense  = RestrideSteps{{seg, seg * n1, seg * n1 * n2}};
    t.padded = g1 != t.dense.st[0] || g2 != t.dense.st[1] || g3 != t.dense.st[2];
    t.extent = (size_t)((n1 - 1) * g1 + (n2 - 1) * g2 + (n3 - 1) * g3 + seg);
    t.bytes  = (size_t)(seg * n1 * n2 * n3);
    return 0;
}

static int conv_src_steps(const mi355_conv_desc &d, ConvTensorSteps &t)
{
    return d.layout == MI355_NHWC
               ? conv_tensor_steps("src", d.C, d.W, d.H, d.batch, d.src_pixel_stride, d.src_stride2, d.src_stride3, t)
               : conv_tensor_steps("src", d.W, d.H, d.C, d.batch, d.src_pixel_stride, d.src_stride2, d.src_stride3, t);
}

static int conv_weights_steps(const mi355_conv_desc &d, ConvTensorSteps &t)
{
    return d.layout == MI355_NHWC ? conv_tensor_steps("weights", d.C, d.KW, d.KH, d.OFM, d.weights_pixel_stride,
                                                      d.weights_stride2, d.weights_stride3, t)
                                  : conv_tensor_steps("weights", d.KW, d.KH, d.C, d.OFM, d.weights_pixel_stride,
                                                      d.weights_stride2, d.weights_stride3, t);
}

static int conv_dst_steps(const mi355_conv_desc &d, ConvTensorSteps &t)
{
    ConvGeom g;
    conv_geom(d, g);
    const int64_t esz = d.dst_dtype == MI355_F32 ? 4 : 1;
    return d.layout == MI355_NHWC
               ? conv_tensor_steps("dst", d.OFM * esz, g.OW, g.OH, d.batch, d.dst_pixel_stride, d.dst_stride2, d.dst_stride3, t)
               : conv_tensor_steps("dst", g.OW * esz, g.OH, d.OFM, d.batch, d.dst_pixel_stride, d.dst_stride2, d.dst_stride3, t);
}

static int conv_check(const mi355_conv_desc &d)
{
    if (d.batch < 1 || d.H < 1 || d.W < 1 || d.C < 1 || d.OFM < 1 || d.KH < 1 || d.KW < 1)
        return fail("convolution dimensions must be positive");
    if (d.stride_x < 1 || d.stride_y < 1 || d.dilation_x < 1 || d.dilation_y < 1)
        return fail("stride and dilation must be >= 1");
    if (d.pad_left < 0 || d.pad_top < 0 || d.pad_right < 0 || d.pad_bottom < 0)
        return fail("negative padding");
    if (!is_8bit(d.src_dtype) || !is_8bit(d.weights_dtype) || (!is_8bit(d.dst_dtype) && d.dst_dtype != MI355_F32))
        return fail("convolution source and weights must be 8-bit, the destination 8-bit or F32");
    if (d.dst_dtype == MI355_F32)
    {
        if ((d.flags & ~MI355_GEMM_ACT_TWICE) != 0)
            return fail("unknown flag bits 0x%x", d.flags);
    }
    if (d.path < MI355_CONV_AUTO || d.path > MI355_CONV_IN_PLACE)
        return fail("unknown convolution path %d", d.path);
    if (d.layout != MI355_NHWC && d.layout != MI355_NCHW)
        return fail("unknown layout %d", d.layout);
    ConvGeom g;
    conv_geom(d, g);
    if (g.OH < 1 || g.OW < 1)
        return fail("the kernel does not fit into the padded image");
    ConvTensorSteps t;
    TRY(conv_src_steps(d, t));
    TRY(conv_weights_steps(d, t));
    TRY(conv_dst_steps(d, t));
    return 0;
}

int mi355_conv_create(const mi355_conv_desc *desc, mi355_conv_handle **out)
{
    if (!desc || !out)
        return fail("null argument");
    const mi355_conv_desc &d = *desc;
    TRY(conv_check(d));
    const bool f32 = d.dst_dtype == MI355_F32;
    if (!f32)
        TRY(check_requant(d.requant, d.dst_dtype));
    mi355_conv_handle *h = new (std::nothrow) mi355_conv_handle();
    if (!h)
        return fail("out of host memory");
    h->d = d;
    conv_geom(d, h->geom);
    GemmCore     &c  = h->core;
    // A channel count that is not a multiple of 16 (the RGB of a first layer, 24, 40 ...): the implicit loaders move
    // 16-byte pieces of one tap, and the fallback that looks up every byte runs at a few percent of what the bytes
    // allow. Channels can be added for nothing: source pixels and weight taps are copied into buffers with the channels
    // padded to the next multiple of 16, the added weights are zero in the kernels' signed form, so no dot product
    // changes and neither do the column sums of the weights. The two other offset terms are kept on the caller's
    // channel count: the row sums of the patches (needed under a weights offset) count only those,
    // and the constant a_offset * b_offset * K uses the unpadded K.
    h->geom_true = h->geom;
    h->geom.c_true = h->geom_true.c_true = d.C;
    int      taps_c = 0; // under patch rows: the padded channels of single taps, and their geometry
    ConvGeom taps_geom{};
    {
        if (d.path == MI355_CONV_AUTO && d.C % 16 != 0)
        {
            mi355_conv_desc dp = d;
            dp.C               = round_up(d.C, 16);
            ConvGeom gp;
            conv_geom(dp, gp);
            if (conv_fast_div_ok(dp, gp) && conv_fast_div_ok(d, h->geom) && (int64_t)d.batch * d.H * d.W * dp.C < ((int64_t)1 << 31))
                h->c_pad = dp.C, gp.c_true = d.C, h->geom = gp;
            // Few channels: rather than every tap, the whole row of KW taps is padded to 16 bytes. The source is copied as
            // patch rows (see patch_rows_kernel) and the convolution becomes KH x 1 over KW * C channels.
            // Taken where the copy does not grow by more than half, or where the padded K at least halves (us, channels padded
            // against rows padded, 32 images): 224 x 224 x 3 -> 64, 7 x 7: 54.9 -> 37.9 at stride 2, 168 -> 107 at stride 1;
            // 3 -> 32, 3 x 3: 29.8 -> 27.8, 75.7 -> 70.4; 8 images of 128 x 128 x 3 -> 96, 5 x 5: 24.4 -> 18.6; 16 of
            // 112 x 112 x 24 -> 32, 3 x 3, stride 2: 12.2 -> 11.1. Not: 112 x 112 x 8 -> 64, 3 x 3: 30.9 -> 31.8, 5 x 5: 32.7 ->
            // 34.3; 56 x 56 x 24, 3 x 3: 14.3 -> 15.0. Less than 8 bytes of a row save nothing where the padded K fits one batch of
            // the narrow kernel's k blocks (192) either way: 224 x 224 x 1 -> 64, 3 x 3: 91.4 -> 96.1.
            // Not either where the row's K just fits that one batch and the padded taps fit two, under few output rows: the form
            // for one batch, which knows several panels, starts half a microsecond later (6272 rows of 20 -> 32 channels, 3 x 3,
            // stride 2, channels padded 6.2, rows 6.5; 12544 rows: 7.1, 6.9). And up to 64 output channels, where the narrow kernel
            // runs either way, a K of 400 (5 x 5) or 576 saves less than a copy costs that is more than half again as large: 16 of 128 x
            // 128 x 4 -> 64, 5 x 5: 24.4 -> 28.3; -> 32: 21.9 -> 23.9 (7 x 7 saves more: see above).
            mi355_conv_desc dr = d;
            dr.C = round_up(d.KW * d.C, 16), dr.W = h->geom_true.OW, dr.KW = dr.stride_x = dr.dilation_x = 1, dr.pad_left = dr.pad_right = 0;
            const int64_t row_bytes = (int64_t)dr.W * dr.C, pad_bytes = (int64_t)d.W * dp.C, k_row = (int64_t)d.KH * dr.C, k_pad = (int64_t)d.KH * d.KW * dp.C;
            const bool    one_batch_late = d.OFM <= 64 && k_row <= 192 && k_pad > 192 && k_pad <= 384 && (int64_t)d.batch * gp.OH * gp.OW < 8192;
            const bool    large_copy = d.OFM <= 64 && 2 * row_bytes > 3 * pad_bytes && k_pad <= 576;
            const bool    pays = !one_batch_late && !large_copy && k_row < k_pad && (2 * row_bytes <= 3 * pad_bytes || 2 * k_row <= k_pad) &&
                              (d.KW * d.C >= 8 || k_pad > 192);
            // Without a weights offset nothing is copied at all: see gemm_rows.hip (more than two panels of output channels would
            // copy the window more often than the pipelined kernel fetches a patch)
            const bool raw = !f32 && d.requant.stage == MI355_STAGE_FIXEDPOINT && d.OFM <= 128 && d.weights_offset + (d.weights_dtype == MI355_U8 ? 128 : 0) == 0 &&
                             conv_rows_applies(h->geom_true);
            if (h->c_pad && (pays || raw) && d.KW > 1 && d.dilation_x == 1 && (int64_t)d.KW * d.C < 1024 &&
                (int64_t)d.batch * d.H * row_bytes < ((int64_t)1 << 31) &&
                patch_rows_fit((int64_t)d.batch * d.H, d.W, d.C, dr.W, d.stride_x, d.pad_left, dr.C))
            {
                taps_c = h->c_pad, taps_geom = h->geom;
                conv_geom(dr, gp);
                if (conv_fast_div_ok(dr, gp))
                    h->c_pad = dr.C, h->patch_rows = true, h->raw_rows = raw, gp.c_true = d.KW * d.C, h->geom = gp;
            }
        }
    }
    auto set_sizes = [&]() -> int
    {
        const int64_t M64 = (int64_t)d.batch * h->geom.OH * h->geom.OW;
        const int64_t K64 = (int64_t)d.KH * h->geom.KW * h->geom.C;
        if (M64 > INT32_MAX || K64 > INT32_MAX)
            return fail("convolution too large");
        c.M = (int)M64, c.N = d.OFM, c.K = (int)K64, c.batch = 1;
        c.k_const = h->c_pad ? d.KH * d.KW * d.C : 0;
        c.patch_c = h->geom.C, c.patch_c_true = h->geom.c_true;
        return 0;
    };
    if (set_sizes())
    {
        delete h;
        return 1;
    }
    // Patch rows bring a short K to convolutions of few channels whatever their size; one panel after the other pays from some
    // rows per compute unit on (us, panels against the pipelined kernel, 128 and 256 columns, 3 channels, 5 x 5, stride 2: 1568
    // rows 8.0 / 5.9 and 11.1 / 5.9; 12544: 8.3 / 6.9 and 11.7 / 8.4; 25088: 9.0 / 8.7 and 12.5 / 10.6; 18 channels, 3 x 3, 12544: 8.7 / 8.5
    // and 11.9 / 9.8; 25088: 9.9 / 9.9 and 13.3 / 13.6)
    c.panels_from = h->patch_rows ? 16384 : 0;
    c.epi = f32 ? EPI_F32 : EPI_FIXEDPOINT, c.dst_dtype = d.dst_dtype;
    c.flip_a = d.src_dtype == MI355_U8, c.flip_b = d.weights_dtype == MI355_U8;
    c.a_offset = d.src_offset, c.b_offset = d.weights_offset;
    c.rq = d.requant, c.path = MI355_PATH_MFMA, c.b_shared = true;
    if (f32)
    {
        c.rq    = mi355_requant{};
        c.scale = d.scale, c.act_min = d.act_min, c.act_max = d.act_max;
        c.act_twice = (d.flags & MI355_GEMM_ACT_TWICE) != 0;
    }
    if (c.choose_kernel())
    {
        delete h;
        return 1;
    }
    h->window_made = h->window = h->choose_window();
    if (h->window && h->patch_rows)
    {
        // its weights are those of single taps
        h->patch_rows = false, h->c_pad = taps_c, h->geom = taps_geom, c.panels_from = 0;
        if (set_sizes() || c.choose_kernel())
        {
            delete h;
            return 1;
        }
    }
    // The patch matrix is only materialised on request (path 1) or where the loaders' reciprocal divisions would not be
    // exact. Channel counts that are not a multiple of 16 and are not padded (see above: a request for the caller's tensor as
    // it is, or sizes beyond 31 bits) take the register-staged kernel, whose loader looks up every byte; there, and in K slices to
    // a float destination, a weights offset costs a pass over the source for the patches' row sums.
    h->implicit      = d.path != MI355_CONV_EXPLICIT && (h->c_pad > 0 || conv_fast_div_ok(d, h->geom));
    h->geom.pad_word = ((uint32_t)d.pad_value & 0xFFu) * 0x01010101u;
    if (h->implicit)
        c.fill_byte = (uint8_t)(d.pad_value & 0xFF);
    if (h->implicit && !conv_taps_ok(h->geom))
        c.no_pipelined_kernel();
    c.kprefix = h->implicit ? "implicit_" : "im2col+";
    c.kname   = c.kprefix + c.kname;
    c.refresh_names();
    *out                = h;
    return 0;
}

int mi355_conv_prepare(mi355_conv_handle *h, const void *weights, const void *bias, const int32_t *mult,
                       const int32_t *shift, void *stream)
{
    if (!h || !weights)
        return fail("null argument");
    hipStream_t s = (hipStream_t)stream;
    GemmCore   &c = h->core;
    const void *wd, *biasd, *multd, *shiftd;
    const bool  f32 = c.epi == EPI_F32;
    if (f32)
    {
        // the float bias is an argument of every launch: keep a device copy of the caller's values
        h->has_bias_f32 = bias != nullptr;
        if (bias)
        {
            TRY(h->biasF.ensure(sizeof(float) * (size_t)c.N));
            HIP_TRY(hipMemcpyAsync(h->biasF.p, bias, sizeof(float) * (size_t)c.N, hipMemcpyDefault, s));
        }
        bias = nullptr;
    }
    ConvTensorSteps wt;
    TRY(conv_weights_steps(h->d, wt));
    TRY(to_device(weights, wt.extent, h->stageW, s, &wd));
    if (wt.padded)
    {
        TRY(h->denseW.ensure(wt.bytes));
        HIP_TRY(restride_nd_launch(wd, h->denseW.p, wt.seg, wt.n1, wt.n2, wt.n3, wt.given, wt.dense, s));
        wd = h->denseW.p;
    }
    if (h->d.layout == MI355_NCHW)
    {
        // [OFM][C][KH*KW] -> [OFM][KH*KW][C]
        TRY(h->nhwcW.ensure((size_t)c.N * c.K));
        HIP_TRY(transpose_bytes_launch(wd, h->nhwcW.p, c.N, h->d.C, h->d.KH * h->d.KW, s));
        wd = h->nhwcW.p;
    }
    if (h->c_pad)
    {
        // taps (or rows of taps) of C weights -> c_pad weights; the added ones are zero once the packing has put them in signed form
        TRY(h->padW.ensure((size_t)c.N * c.K));
        HIP_TRY(channel_pad_launch(wd, h->padW.p, (int64_t)c.N * h->d.KH * h->geom.KW, h->geom.c_true, h->c_pad, c.flip_b ? 0x80 : 0x00, s));
        wd = h->padW.p;
    }
    TRY(to_device(bias, sizeof(int32_t) * c.N, h->stageBias, s, &biasd));
    TRY(to_device(c.rq.per_channel ? mult : nullptr, sizeof(int32_t) * c.N, h->stageMult, s, &multd));
    TRY(to_device(c.rq.per_channel ? shift : nullptr, sizeof(int32_t) * c.N, h->stageShift, s, &shiftd));
    // weights [OFM][KH][KW][C] are already the K-contiguous layout with k = c + kx*C + ky*C*KW
    // (src/cpu/kernels/CpuWeightsReshapeKernel.cpp:150-166)
    TRY(c.pack(wd, c.K, 0, true, 0, (const int32_t *)biasd, s, h->window_made));
    TRY(c.finish_prepare((const int32_t *)multd, (const int32_t *)shiftd, s));
    HIP_TRY(hipStreamSynchronize(s));
    c.prepared = true;
    return 0;
}

int mi355_conv_update_quant(mi355_conv_handle *h, int32_t src_offset, int32_t weights_offset, int32_t pad_value,
                            const mi355_requant *requant, const int32_t *mult, const int32_t *shift, void *stream)
{
    if (!h || !requant)
        return fail("null argument");
    hipStream_t s = (hipStream_t)stream;
    GemmCore   &c = h->core;
    if (c.epi == EPI_F32)
        return fail("the F32 destination has no requantisation to update: create a new handle for new scales");
    TRY(check_requant(*requant, c.dst_dtype));
    if ((requant->per_channel != 0) != (c.rq.per_channel != 0))
        return fail("update cannot switch between per-tensor and per-channel requantisation");
    h->d.src_offset = src_offset, h->d.weights_offset = weights_offset, h->d.pad_value = pad_value, h->d.requant = *requant;
    c.a_offset = src_offset, c.b_offset = weights_offset, c.rq = *requant;
    h->implicit      = h->d.path != MI355_CONV_EXPLICIT && (h->c_pad > 0 || conv_fast_div_ok(h->d, h->geom));
    h->geom.pad_word = ((uint32_t)pad_value & 0xFFu) * 0x01010101u;
    c.fill_byte      = (uint8_t)(pad_value & 0xFF);
    c.kprefix        = h->implicit ? "implicit_" : "im2col+";
    c.refresh_names();
    h->window = h->window_made && h->divide_window();
    if (!c.prepared)
        return 0;
    // a run that kept its window in LDS has neither padded channels nor turned a layout round: the next one may be recorded and could not make room
    if (h->window_made && !h->from_window())
    {
        if (h->c_pad)
            TRY(h->padSrc.ensure(h->pad_bytes()));
        if (h->d.layout == MI355_NCHW)
        {
            ConvTensorSteps st, dt;
            TRY(conv_src_steps(h->d, st));
            TRY(conv_dst_steps(h->d, dt));
            TRY(h->nhwcSrc.ensure(st.bytes));
            TRY(h->nhwcDst.ensure(dt.bytes));
        }
    }
    // a run that went straight from the image has made no patch rows: the next one may be recorded and could not make room for them
    if (h->raw_rows && !h->from_image())
        TRY(h->padSrc.ensure(h->pad_bytes()));
    if (c.rq.per_channel)
    {
        if (!mult || !shift)
            return fail("per-channel requantisation needs multiplier and shift arrays");
        const void *multd, *shiftd;
        TRY(to_device(mult, sizeof(int32_t) * c.N, h->stageMult, s, &multd));
        TRY(to_device(shift, sizeof(int32_t) * c.N, h->stageShift, s, &shiftd));
        HIP_TRY(hipMemcpyAsync(c.mult.p, multd, sizeof(int32_t) * (size_t)c.N, hipMemcpyDeviceToDevice, s));
        HIP_TRY(hipMemcpyAsync(c.shift.p, shiftd, sizeof(int32_t) * (size_t)c.N, hipMemcpyDeviceToDevice, s));
    }
    c.keep_flags(s);
    TRY(c.set_fill(s));
    TRY(c.refresh_colvec(s));
    TRY(c.refresh_qparams(s));
    c.keep_flags(s);
    HIP_TRY(hipStreamSynchronize(s));
    return 0;
}

int mi355_conv_set_strides(mi355_conv_handle *h, int64_t src_pixel_stride, int64_t weights_pixel_stride,
                           int64_t dst_pixel_stride)
{
    if (!h)
        return fail("null argument");
    const int64_t a[3] = {src_pixel_stride, 0, 0}, b[3] = {weights_pixel_stride, 0, 0}, c[3] = {dst_pixel_stride, 0, 0};
    return mi355_conv_set_strides_nd(h, a, b, c);
}

int mi355_conv_set_strides_nd(mi355_conv_handle *h, const int64_t src[3], const int64_t weights[3], const int64_t dst[3])
{
    if (!h || !src || !weights || !dst)
        return fail("null argument");
    mi355_conv_desc d = h->d;
    d.src_pixel_stride = src[0], d.src_stride2 = src[1], d.src_stride3 = src[2];
    d.weights_pixel_stride = weights[0], d.weights_stride2 = weights[1], d.weights_stride3 = weights[2];
    d.dst_pixel_stride = dst[0], d.dst_stride2 = dst[1], d.dst_stride3 = dst[2];
    TRY(conv_check(d));
    h->d = d;
    return 0;
}

int mi355_conv_run(mi355_conv_handle *h, const void *src, void *dst, void *stream)
{
    if (!h || !src || !dst)
        return fail("null argument");
    hipStream_t            s = (hipStream_t)stream;
    GemmCore              &c = h->core;
    const mi355_conv_desc &d = h->d;
    if (!c.prepared)
        return fail("run before prepare");
    ConvTensorSteps st, dt;
    TRY(conv_src_steps(d, st));
    TRY(conv_dst_steps(d, dt));
    const size_t src_bytes = st.bytes, dst_bytes = dt.bytes, dst_ext = dt.extent;
    const bool   s_pad = st.padded, d_pad = dt.padded;
    const void  *srcd;
    TRY(to_device(src, st.extent, h->stageSrc, s, &srcd, &h->kindSrc));
    if (s_pad)
    {
        TRY(h->denseSrc.ensure(src_bytes));
        HIP_TRY(restride_nd_launch(srcd, h->denseSrc.p, st.seg, st.n1, st.n2, st.n3, st.given, st.dense, s));
        srcd = h->denseSrc.p;
    }
    const bool d_host = !h->kindDst.is_device(dst);
    void      *Dd     = dst;
    if (d_host)
    {
        TRY(h->stageDst.ensure(dst_ext));
        Dd = h->stageDst.p;
        if (d_pad)
            HIP_TRY(hipMemcpyAsync(Dd, dst, dst_ext, hipMemcpyHostToDevice, s)); // keep the caller's padding bytes
    }
    void *Dpadded = Dd;
    if (d_pad)
    {
        TRY(h->denseDst.ensure(dst_bytes));
        Dd = h->denseDst.p;
    }
    const bool nchw   = d.layout == MI355_NCHW;
    void      *Dfinal = Dd;
    bool       planes = false; // the kernel writes NCHW itself
    // ... or [OH*OW][OFM] per image into a buffer of its own
    auto own_dst = [&]() -> int
    {
        TRY(h->nhwcDst.ensure(dst_bytes));
        Dd = h->nhwcDst.p;
        return 0;
    };
    if (h->from_window())
    {
        GemmArgs g{};
        c.fill_epi(g.epi, nullptr);
        g.epi.rowsum_mul = c.b_off_eff(), g.epi.planes = nchw ? h->geom.OH * h->geom.OW : 0;
        g.A = (const int8_t *)srcd, g.Bp = c.Bp.as<int8_t>() + (size_t)c.Np * c.Kp, g.Kp = c.Kp;
        g.D = Dd, g.ldd = c.N, g.M = c.M, g.N = c.N, g.K = c.K;
        g.conv          = h->geom_true;
        g.conv.pad_word = ((uint32_t)d.pad_value & 0xFFu) * 0x01010101u;
        HIP_TRY(conv_window_launch(h->window_plan, c.flip_a, g, d.batch, s));
        c.kname_run = &c.kname_window;
        planes      = nchw;
    }
    else if (nchw)
    {
        // every image [C][H*W] -> [H*W][C]
        TRY(h->nhwcSrc.ensure(src_bytes));
        HIP_TRY(transpose_bytes_launch(srcd, h->nhwcSrc.p, d.batch, d.C, d.H * d.W, s));
        srcd = h->nhwcSrc.p;
        // (an update moves a convolution of few channels between a kernel that writes planes and one that does not: made by either run)
        if (!h->implicit || h->raw_rows)
            TRY(own_dst());
    }
    const void *src_true = srcd; // the caller's channel count
    const bool  raw      = h->from_image();
    if (h->c_pad && !raw && !h->from_window())
    {
        // pixels of C channels -> pixels of c_pad channels (what the added ones hold meets zero weights; the padding value
        // keeps them in range of the source type)
        TRY(h->padSrc.ensure(h->pad_bytes()));
        if (h->patch_rows)
            HIP_TRY(patch_rows_launch(srcd, h->padSrc.p, (int64_t)d.batch * d.H, d.W, d.C, h->geom.W, d.stride_x, d.pad_left, h->c_pad, (uint8_t)(d.pad_value & 0xFF), s));
        else
            HIP_TRY(channel_pad_launch(srcd, h->padSrc.p, (int64_t)d.batch * d.H * d.W, d.C, h->c_pad, (uint8_t)(d.pad_value & 0xFF), s));
        srcd = h->padSrc.p;
    }
    if (h->from_window())
        ; // (done)
    else if (raw)
    {
        GemmArgs g{};
        c.fill_epi(g.epi, nullptr);
        g.A = (const int8_t *)src_true, g.Bp = c.Bp.as<int8_t>(), g.Kp = c.Kp;
        g.D = Dd, g.ldd = c.N, g.M = c.M, g.N = c.N, g.K = c.K;
        g.conv          = h->geom_true;
        g.conv.pad_word = ((uint32_t)d.pad_value & 0xFFu) * 0x01010101u;
        c.set_vec_store(g);
        HIP_TRY(conv_rows_launch(c.flip_a, g, d.batch, s));
        c.kname_run = &c.kname_rows;
    }
    else if (h->implicit)
    {
        GemmArgs g{};
        c.fill_epi(g.epi, h->has_bias_f32 ? h->biasF.as<float>() : nullptr);
        // a weights offset: the kernels sum the patches as they pass (see conv_row_terms for those that do not)
        g.epi.rowsum_mul   = c.b_off_eff();
        c.rs_src           = h->c_pad ? src_true : srcd;
        c.rs_geom          = h->c_pad ? h->geom_true : h->geom;
        c.rs_geom.pad_word = ((uint32_t)d.pad_value & 0xFFu) * 0x01010101u;
        g.A = (const int8_t *)srcd, g.lda = 0, g.a_batch_stride = 0;
        g.Bp = c.Bp.as<int8_t>(), g.Kp = c.Kp, g.bp_batch_stride = 0;
        g.ldd = c.N, g.d_batch_stride = 0;
        g.M = c.M, g.N = c.N, g.K = c.K;
        g.conv = h->geom;
        if (nchw && c.stores_planes(g))
            Dd = Dfinal, g.epi.planes = h->geom.OH * h->geom.OW, planes = true; // straight into the caller's planes
        else if (nchw)
            TRY(own_dst());
        g.D = Dd;
        c.set_vec_store(g);
        TRY(c.launch(g, c.flip_a, true, s));
    }
    else
    {
        // explicit lowering: patch matrix [M][Kp] in workspace, then the dense path
        ConvGeom g2   = h->geom;
        g2.pad_word   = ((uint32_t)d.pad_value & 0xFFu) * 0x01010101u;
        const int ldc = round_up(c.K, 16);
        TRY(h->cols.ensure((size_t)c.M * ldc));
        HIP_TRY(im2col_nhwc_launch(srcd, h->cols.p, d.batch, g2, ldc, s));
        TRY(c.run_dense(h->cols.as<int8_t>(), ldc, 0, Dd, c.N, 0, h->has_bias_f32 ? h->biasF.as<float>() : nullptr, s));
    }
    if (nchw && !planes)
    {
        HIP_TRY((c.epi == EPI_F32 ? transpose_words_launch : transpose_bytes_launch)(Dd, Dfinal, d.batch, h->geom.OH * h->geom.OW, c.N, s));
        Dd = Dfinal;
    }
    if (d_pad)
    {
        HIP_TRY(restride_nd_launch(Dd, Dpadded, dt.seg, dt.n1, dt.n2, dt.n3, dt.dense, dt.given, s));
        Dd = Dpadded;
    }
    if (d_host)
    {
        HIP_TRY(hipMemcpyAsync(dst, Dd, dst_ext, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    else if (!h->kindSrc.is_device(src))
        HIP_TRY(hipStreamSynchronize(s));
    return 0;
}

void mi355_conv_destroy(mi355_conv_handle *h)
{
    if (!h)
        return;
    h->core.release();
    h->stageSrc.release(), h->stageW.release(), h->stageDst.release(), h->stageBias.release();
    h->stageMult.release(), h->stageShift.release(), h->cols.release();
    h->nhwcSrc.release(), h->nhwcW.release(), h->nhwcDst.release(), h->biasF.release();
    h->denseSrc.release(), h->denseW.release(), h->denseDst.release(), h->padSrc.release(), h->padW.release();
    delete h;
}

const char *mi355_conv_kernel_name(const mi355_conv_handle *h)
{
    return h ? h->core.name() : "";
}

int mi355_im2col_nhwc_run(const mi355_conv_desc *desc, const void *src, void *dst, void *stream)
{
    if (!desc || !src || !dst)
        return fail("null argument");
    const mi355_conv_desc &d = *desc;
    TRY(conv_check(d));
    if (d.layout != MI355_NHWC)
        return fail("mi355_im2col_nhwc_run lowers NHWC tensors only");
    ConvGeom g{};
    conv_geom(d, g);
    g.pad_word      = ((uint32_t)d.pad_value & 0xFFu) * 0x01010101u;
    hipStream_t s   = (hipStream_t)stream;
    const size_t K  = (size_t)d.KH * d.KW * d.C, rows = (size_t)d.batch * g.OH * g.OW;
    DevBuf       sSrc, sDst;
    const void  *srcd;
    void        *Dd     = dst;
    const bool   d_host = !is_device_ptr(dst);
    auto         body   = [&]() -> int
    {
        TRY(to_device(src, (size_t)d.batch * d.H * d.W * d.C, sSrc, s, &srcd));
        if (d_host)
        {
            TRY(sDst.ensure(rows * K));
            Dd = sDst.p;
        }
        HIP_TRY(im2col_nhwc_launch(srcd, Dd, d.batch, g, (int64_t)K, s));
        if (d_host)
            HIP_TRY(hipMemcpyAsync(dst, Dd, rows * K, hipMemcpyDeviceToHost, s));
        if (d_host || srcd != src)
            HIP_TRY(hipStreamSynchronize(s));
        return 0;
    };
    const int rc = body();
    sSrc.release(), sDst.release();
    return rc;
}
} // extern "C"
