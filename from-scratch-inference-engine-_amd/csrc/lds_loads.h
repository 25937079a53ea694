// Loads from memory to LDS that go through no register (buffer loads with the lds bit), for the products that bring both operands so.
#pragma once
#include "common.h"

namespace fsie_lds {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes a lane from memory to LDS, lane i's at lds + 16 i (m0 is an operand; the wait state behind its write is not the compiler's to
// put inside an asm statement).
__device__ __forceinline__ void load_to_lds(u32x4 rsrc, uint32_t lds, uint32_t offset, uint32_t k_offset) {
    asm volatile(
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen lds"
        :
        : "{m0}"(lds), "v"(offset), "s"(rsrc), "s"(k_offset)
        : "memory");
}
// Four bytes a lane, as above.
__device__ __forceinline__ void touch(u32x4 rsrc, uint32_t lds, uint32_t offset, uint32_t k_offset) {
    asm volatile(
        "s_nop 0\n\t"
        "buffer_load_dword %1, %2, %3 offen lds"
        :
        : "{m0}"(lds), "v"(offset), "s"(rsrc), "s"(k_offset)
        : "memory");
}

// A buffer descriptor of `bytes` bytes from `base` on, in scalar registers.
__device__ __forceinline__ u32x4 rows_from(const void* base, uint32_t bytes) {
    const uint64_t at = reinterpret_cast<uint64_t>(base);
    u32x4 r;
    r[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at));
    r[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at >> 32));
    r[2] = __builtin_amdgcn_readfirstlane(bytes);
    r[3] = 0x00020000u;
    return r;
}

}  // namespace fsie_lds
