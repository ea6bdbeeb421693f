// Loads from memory straight into LDS for the matrix-core kernels, as assembly.
//
// The compiler knows the builtin's write to LDS, but not which of the kernel's waits it is covered by, and puts an
// "s_waitcnt vmcnt(0)" before reads from LDS that may follow it: which reads these are changes with the code around, and
// one of them, right behind the loads of the next stage, made the walks of these kernels idle for a memory latency every
// fourth stage.  Here it sees no write, only a barrier for its own memory operations; the waits are the kernel's
// (s_waitcnt vmcnt, which counts these loads in the order they were sent in).  No register is written, so nothing can
// arrive in one that has been given to somebody else.
//
// `to` and the base are uniform over the wave (uniform_address); lane l's bytes land at to + l * size.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi355 {

typedef const uint8_t __attribute__((address_space(1))) *lds_load_from;

__device__ __forceinline__ uint32_t lds_load_place(const void *to) {
    return (uint32_t)(uintptr_t)(const uint8_t __attribute__((address_space(3))) *)to;
}

// an address that is the same in every lane, in scalar registers
__device__ __forceinline__ lds_load_from uniform_address(lds_load_from p) {
    const uint64_t bits = (uint64_t)(uintptr_t)p;
    const uint32_t low = __builtin_amdgcn_readfirstlane((int)(uint32_t)bits), high = __builtin_amdgcn_readfirstlane((int)(uint32_t)(bits >> 32));
    return (lds_load_from)(uintptr_t)((uint64_t)high << 32 | low);
}

// sixteen or two bytes per lane, from a uniform address and a lane's 32-bit offset
//
// A memory instruction may read a scalar register five wait states after a vector instruction has written it (a
// readfirstlane, or the readlane of a spilled one) and no sooner, which the compiler sees to for instructions that it knows.
// Here the load's base is a copy that a scalar instruction makes: that one waits for vector writes by itself, and nobody has
// to wait for what it writes.  It is also the one wait state that a load into LDS wants after the write of m0.
template <int SIZE> __device__ __forceinline__ void load_to_lds(lds_load_from base, uint32_t offset, const void *to) {
    static_assert(SIZE == 16 || SIZE == 2, "");
    uint64_t copy;
    if (SIZE == 16)
        asm volatile("s_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(copy) : "{m0}"(lds_load_place(to)), "v"(offset), "s"(base) : "memory");
    else
        asm volatile("s_mov_b64 %0, %3\n\tglobal_load_lds_ushort %2, %0" : "=&s"(copy) : "{m0}"(lds_load_place(to)), "v"(offset), "s"(base) : "memory");
}

// the same with a 64-bit offset
template <int SIZE> __device__ __forceinline__ void load_to_lds(lds_load_from base, uint64_t offset, const void *to) {
    static_assert(SIZE == 16 || SIZE == 2, "");
    const uint64_t at = (uint64_t)(uintptr_t)base + offset;
    if (SIZE == 16)
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds_load_place(to)), "v"(at) : "memory");
    else
        asm volatile("s_nop 0\n\tglobal_load_lds_ushort %1, off" ::"{m0}"(lds_load_place(to)), "v"(at) : "memory");
}

}  // namespace mi355
