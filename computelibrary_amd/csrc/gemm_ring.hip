// Instances of the tiles of gemm_ring.hpp
#include "gemm_ring.hpp"

namespace mi355
{
// (KD: wave groups of the dense kernels, KC: of the convolutions; 0: not built for these)
template <int BM, int BN, int BK, int NS, int KG, int E, bool F, int MODE>
static const void *ring_fn()
{
    if constexpr (KG == 0)
        return nullptr;
    else
        return (const void *)gemm_ring_kernel<BM, BN, BK, NS, KG, E, F, MODE>;
}
#define MI355_REPI(BM, BN, BK, NS, KD, KC, E)                                                                                \
    {                                                                                                                        \
        {ring_fn<BM, BN, BK, NS, KD, E, false, RING_DENSE>(), ring_fn<BM, BN, BK, NS, KC, E, false, RING_CONV>()},           \
            {ring_fn<BM, BN, BK, NS, KD, E, true, RING_DENSE>(), ring_fn<BM, BN, BK, NS, KC, E, true, RING_CONV>()},         \
    }
#define MI355_RCFG(NAME, BM, BN, BK, NS, KD, KC)                                                                             \
    {                                                                                                                        \
        {NAME, BM, BN, BK}, {NS *(BM + BN) * BK, NS *(BM + BN) * BK + 1024}, {KD * 256, KC * 256},                           \
            {MI355_REPI(BM, BN, BK, NS, KD, KC, 0), MI355_REPI(BM, BN, BK, NS, KD, KC, 1), MI355_REPI(BM, BN, BK, NS, KD, KC, 2)} \
    }
// (128 x 128 tiles of this form, one workgroup per compute unit for their registers, were slower than these or than the copy and
// its tiles on all of 69 shapes: 4096 x 4096 x 4095 171 us, 64 x 64 164, with the copy 78)
#define MI355_RBYTES(E) {ring_fn<64, 64, 128, 3, 1, E, false, RING_BYTES>(), ring_fn<64, 64, 128, 3, 1, E, true, RING_BYTES>()}
const void *const g_ring_bytes[3][2] = {MI355_RBYTES(0), MI355_RBYTES(1), MI355_RBYTES(2)};
const RingEntry g_ring[] = {
    MI355_RCFG("pp_128x128x128_s3", 128, 128, 128, 3, 1, 2),
    MI355_RCFG("pp_128x64x128_s3", 128, 64, 128, 3, 1, 1),
    MI355_RCFG("pp_64x64x128_s3", 64, 64, 128, 3, 1, 1),
    MI355_RCFG("pp_64x64x128_s6", 64, 64, 128, 6, 1, 0),
    MI355_RCFG("pp_128x64x256_s3", 128, 64, 256, 3, 2, 0),
    MI355_RCFG("pp_128x128x128_s2", 128, 128, 128, 2, 1, 1),
    MI355_RCFG("pp_64x64x256_s2", 64, 64, 256, 2, 2, 2),
};
static_assert(sizeof(g_ring) / sizeof(g_ring[0]) == 7, "dma_launch and its prices know 7");
const int g_ring_count = (int)(sizeof(g_ring) / sizeof(g_ring[0]));
} // namespace mi355
