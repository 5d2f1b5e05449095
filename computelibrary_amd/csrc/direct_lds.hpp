// Direct-to-LDS loads and the waits that go with them, issued by hand: the compiler cannot tell which LDS bytes such a load
// writes and would wait for all of them in front of every LDS read. Nor does it keep the distances that the hardware asks for inside such a
// block: one instruction between a write of M0 and a load to LDS, and five between a vector instruction that writes a scalar register
// (a spilled one that comes back by v_readlane) and a load that takes its address from there.
#pragma once
#include "mfma_common.hpp"

namespace mi355
{
// one wave instruction: 64 lanes x 16 bytes from the lanes' addresses to 1 KiB of LDS at lds_addr
__device__ __forceinline__ void dma16(const void *gptr, uint32_t lds_addr)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "s"(lds_addr) : "memory");
}

// scalar-base form: address = sbase (SGPR pair, wave-uniform) + zero-extended per-lane 32-bit offset; to LDS at lds_addr + off, added up on
// the way into M0 (with the s_nop that is one instruction, the K step of a 64 x 64 tile is as long as without either). For kernels that
// spill no scalars
__device__ __forceinline__ void dma16s(const void *sbase, uint32_t voff, uint32_t lds_addr, int off)
{
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr), "n"(off) : "memory", "scc");
}

// ... and for those that do: the base goes through a scalar copy, which the hardware does hold back, in the place of the s_nop. (Used
// everywhere it costs 64 x 64 tiles 3 to 5 % of a K step: 473 x 1600 x 3008 7.35 -> 7.83 us.)
__device__ __forceinline__ void dma16s_copied(const void *sbase, uint32_t voff, uint32_t lds_addr)
{
    uint64_t base;
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\tglobal_load_lds_dwordx4 %1, %0" : "=&s"(base) : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}

// ... for the lanes in `lanes` (not none), while those in `others` write `pad` to LDS at slot + off. All 64 lanes are active.
__device__ __forceinline__ void dma16s_or_pad(const void *sbase, uint32_t voff, uint32_t lds_addr, uint64_t lanes, uint64_t others, uint32_t slot,
                                              int off, v4i pad)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, %4\n\tds_write_b128 %5, %6 offset:%7\n\t"
                 "s_mov_b64 exec, -1" ::"v"(voff),
                 "s"(sbase), "s"(lds_addr), "s"(lanes), "s"(others), "v"(slot), "v"(pad), "n"(off)
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
