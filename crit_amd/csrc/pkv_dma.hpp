// Loads that the memory pipe writes into LDS itself (no register holds what is in flight), their waits, and reads that LDS
// transposes.
#pragma once
#include "pkv_common.hpp"

namespace pkv {

// 64 lanes x 16 bytes from base + offset (a lane's own) to LDS bytes lds .. lds + 1023 (ONCE: not kept in the caches), and
// 4 bytes a lane to lds + 4 lane. Spelled in assembly so that the compiler neither counts these loads nor waits for them:
// the waits are the kernel's own (wait_dma), and "memory" clobbers, which keeps the reads of LDS behind them.
template <bool ONCE>
PKV_DEV void dma_rows(uint32_t offset, const uint8_t* base, unsigned lds) {
    lds = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);      // (uniform; it may have been kept in a vector register)
    if constexpr (ONCE) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(offset), "s"(base), "s"(lds));
    else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds));
}
PKV_DEV void dma_any(const uint8_t* from, unsigned lds) {      // (each lane from its own address)
    lds = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds));
}
PKV_DEV void dma_words(const float* from, unsigned lds) {
    lds = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(from), "s"(lds));
}
template <int N>
PKV_DEV void wait_dma() {
    static_assert(N >= 0 && N < 64, "vmcnt is six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// The wavefront's own LDS reads have returned: what they read may be overwritten.
PKV_DEV void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// 4 consecutive rows of one value, transposed on the way out of LDS: lane 4 j + c of a 16-lane group points at row j's
// values 4 c .. 4 c + 3; lane i of the group receives value i of rows 0 .. 3.
PKV_DEV u32x2 read_transposed(const uint8_t* p) {
    typedef short v4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4*)(p)));
}

}   // namespace pkv
