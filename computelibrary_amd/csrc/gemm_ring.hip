// Instances of the tiles of gemm_ring.hpp
#include "gemm_ring.hpp"

namespace mi355
{
#define MI355_RFN(BM, BN, BK, NS, KG, E, F, C) (const void *)gemm_ring_kernel<BM, BN, BK, NS, KG, E, F, C>
// (KD: wave groups of the dense kernels, KC: of the convolutions)
#define MI355_REPI(BM, BN, BK, NS, KD, KC, E)                                                                \
    {                                                                                                        \
        {MI355_RFN(BM, BN, BK, NS, KD, E, false, 0), MI355_RFN(BM, BN, BK, NS, KC, E, false, 1)},             \
            {MI355_RFN(BM, BN, BK, NS, KD, E, true, 0), MI355_RFN(BM, BN, BK, NS, KC, E, true, 1)},           \
    }
#define MI355_RCFG(NAME, BM, BN, BK, NS, KD, KC)                                                                                     \
    {                                                                                                                                \
        {NAME, BM, BN, BK}, {NS *(BM + BN) * BK, NS *(BM + BN) * BK + 1024}, {KD * 256, KC * 256},                                                          \
            {MI355_REPI(BM, BN, BK, NS, KD, KC, 0), MI355_REPI(BM, BN, BK, NS, KD, KC, 1), MI355_REPI(BM, BN, BK, NS, KD, KC, 2)}       \
    }
const RingEntry g_ring[] = {
    MI355_RCFG("pp_128x128x128_s3", 128, 128, 128, 3, 1, 2),
    MI355_RCFG("pp_128x64x128_s3", 128, 64, 128, 3, 1, 1),
    MI355_RCFG("pp_64x64x128_s3", 64, 64, 128, 3, 1, 1),
    MI355_RCFG("pp_64x64x128_s6", 64, 64, 128, 6, 1, 2),
    MI355_RCFG("pp_128x64x256_s3", 128, 64, 256, 3, 2, 2),
    MI355_RCFG("pp_128x128x128_s2", 128, 128, 128, 2, 1, 1),
    MI355_RCFG("pp_64x64x256_s2", 64, 64, 256, 2, 2, 2),
};
static_assert(sizeof(g_ring) / sizeof(g_ring[0]) == 7, "dma_launch and its prices know 7");
const int g_ring_count = (int)(sizeof(g_ring) / sizeof(g_ring[0]));
} // namespace mi355
