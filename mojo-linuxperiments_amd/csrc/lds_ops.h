// Instruction-level pieces of the kernels that stream operands through LDS: waits, LDS fragment reads and direct-to-LDS loads.
#pragma once
#include "common.h"

namespace mi {

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

template <int N>
__device__ __forceinline__ void wait_lgkm()
{
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
template <int OFF>
__device__ __forceinline__ void ds_read128(v4i &dst, unsigned addr)
{
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
// Direct-to-LDS loads of 16 and of 4 bytes per lane: global address = sbase + voff, LDS address = ldsaddr + 16 (4) * lane.  A
// file that uses them is built with the check for spilled scalars: the compiler does not pad a base that it brings back with a
// vector instruction for a load that it cannot see.
__device__ __forceinline__ void dma16(const int8_t *sbase, unsigned voff, unsigned ldsaddr)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(ldsaddr)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma4(const float *sbase, unsigned voff, unsigned ldsaddr)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(ldsaddr)
                 : "memory", "m0");
}
// the value of lane ^ 8 of the same 16
__device__ __forceinline__ int ror8(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false); }

}  // namespace mi
