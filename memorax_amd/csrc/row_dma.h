// Rows from memory to LDS without passing through registers, each wave counting its own requests.
#pragma once
#include "common.h"

namespace mrx {
namespace {

// All but the last N vector memory operations of this wave are done (they end in order).
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory"); }
// 16 (4) bytes for each lane from base + off to LDS, lane by lane from `lds` on.  The compiler does not see these, or it would wait for
// all of them before every read of LDS: whoever reads what they bring waits by wait_vm first, and for the other waves' by a barrier; and
// a workgroup waits for all of its own before it ends, when its LDS goes to another.  The address of the first lane's goes by m0, which
// the compiler writes as an operand: it knows what the register holds before and after.
__device__ __forceinline__ void dma16(const void *base, uint32_t off, uint32_t lds)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void dma4(const void *base, uint32_t off, uint32_t lds)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %1, %2" ::"{m0}"(lds), "v"(off), "s"(base) : "memory");
}
// Where a workgroup's dynamic LDS starts, as those count it.
__device__ __forceinline__ uint32_t lds_address(unsigned char *smem)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
}

}  // namespace
}  // namespace mrx
