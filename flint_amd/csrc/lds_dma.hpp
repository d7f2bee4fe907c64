// Direct-to-LDS loads (gfx950): 16 bytes per lane from memory into LDS without
// passing through registers.  Lane i's bytes go to LDS byte l + 16 i (l the
// same in every lane).  Written in assembly, which names no result register:
// with the builtin the compiler waits for every load in flight before the
// next LDS read, as it cannot tell one stage of a ring from another.  The
// caller waits itself (wait_vm) before it reads what a load brought, and
// orders a request behind the reads of what it overwrites.
#pragma once

#include <cstdint>

namespace thb {

// NT: non-temporal, for bytes that are read once (they would take the place of
// what the next kernel finds in L2: its code, its tables, its inputs).
template <bool NT = false>
__device__ inline void dma16(const void* g, uint32_t l) {
    if constexpr (NT)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(g), "s"(l)
                     : "m0", "memory");
    else
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(l)
                     : "m0", "memory");
}

// The same from byte `off` (per lane) past a base the lanes share.
template <bool NT = false>
__device__ inline void dma16_from(const void* base, uint32_t off, uint32_t l) {
    if constexpr (NT)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(base), "s"(l)
                     : "m0", "memory");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(l)
                     : "m0", "memory");
}

__device__ inline uint32_t lds_offset(const void* l) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)l));
}

// Waits until at most N of this wave's loads are in flight and its LDS
// accesses are done (s_waitcnt, gfx9 encoding: vmcnt in bits 3:0 and 15:14,
// expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ inline void wait_vm() {
    static_assert(N < 64, "vmcnt");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
    asm volatile("" ::: "memory");
}

}  // namespace thb
