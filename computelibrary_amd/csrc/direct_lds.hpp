// Direct-to-LDS loads and the waits that go with them, issued by hand: the compiler cannot tell which LDS bytes such a load
// writes and would wait for all of them in front of every LDS read. Nor does it keep the distances that the hardware asks for inside such a
// block: one instruction between a write of M0 and a load to LDS, and five between a vector instruction that writes a scalar register
// (a spilled one that comes back by v_readlane) and a load that takes its address from there. So the base goes through a scalar
// copy, which hardware does hold back, and the copy is what stands behind the write of M0.
#pragma once
#include "mfma_common.hpp"

namespace mi355
{
// one wave instruction: 64 lanes x 16 bytes from the lanes' addresses to 1 KiB of LDS at lds_addr
__device__ __forceinline__ void dma16(const void *gptr, uint32_t lds_addr)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "s"(lds_addr) : "memory");
}

// scalar-base form: address = sbase (SGPR pair, wave-uniform) + zero-extended per-lane 32-bit offset
__device__ __forceinline__ void dma16s(const void *sbase, uint32_t voff, uint32_t lds_addr)
{
    uint64_t base;
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\tglobal_load_lds_dwordx4 %1, %0" : "=&s"(base) : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}

// ... for the lanes in `lanes` (not none), while those in `others` write `pad` to LDS at slot + off. All 64 lanes are active.
__device__ __forceinline__ void dma16s_or_pad(const void *sbase, uint32_t voff, uint32_t lds_addr, uint64_t lanes, uint64_t others, uint32_t slot,
                                              int off, v4i pad)
{
    uint64_t base;
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\ts_mov_b64 exec, %4\n\tglobal_load_lds_dwordx4 %1, %0\n\ts_mov_b64 exec, %5\n\t"
                 "ds_write_b128 %6, %7 offset:%8\n\ts_mov_b64 exec, -1"
                 : "=&s"(base)
                 : "v"(voff), "s"(sbase), "s"(lds_addr), "s"(lanes), "s"(others), "v"(slot), "v"(pad), "n"(off)
                 : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void block_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
} // namespace mi355
