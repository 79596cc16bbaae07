// Global-to-LDS DMA and the waits and barriers that order it, shared by the
// GEMM kernels whose tiles are staged without passing through registers.
#pragma once

#include "common.cuh"

namespace smg {

// LDS DMA: each lane's 16 (4) bytes from sbase + voff land at M0 + 16 (4) *
// lane; sbase is wave-uniform (scalar registers), voff the lane's 32-bit byte
// offset, so a step's addresses cost no vector instructions. The instructions
// are issued from inline asm so that the compiler neither tracks them nor adds
// waits of its own (it cannot tell which stage a DMA fills); the kernel's
// explicit vmcnt waits and barriers order them. The "memory" clobber keeps LDS
// reads from moving across an issue; s_nop covers the M0 write hazard. lds is a
// wave-uniform LDS byte address. (M0 has no other user in these kernels, so
// clobbering it is safe.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void *sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase),
                 "s"(lds)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void *sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase),
                 "s"(lds)
                 : "memory", "m0");
}
// The same through a buffer resource (make_rsrc4): the 16 bytes at voff, zeros
// where that lies past the resource. (The whole offset is the lane's: the
// range check takes the resource's size less a scalar offset, which would wrap
// for one past the end.)
typedef int rsrc4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rsrc4_t make_rsrc4(const void *base, uint32_t bytes) {
    const uint64_t b = (uint64_t)base;
    return (rsrc4_t){__builtin_amdgcn_readfirstlane((int)b), __builtin_amdgcn_readfirstlane((int)(b >> 32) & 0xFFFF),
                     __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}
__device__ __forceinline__ void dma16_buf(const rsrc4_t &r, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)p;
}

// s_waitcnt vmcnt(n) (gfx9 encoding; expcnt and lgkmcnt left unwaited).
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier that orders LDS accesses without waiting on outstanding
// DMA (a release fence would wait for all of it): the empty asm statements keep
// the compiler from moving memory accesses across it; the caller first waits
// for the DMA the next step reads.
__device__ __forceinline__ void barrier_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) uint8_t lds_u8_t;
template <class T>
__device__ __forceinline__ T lds_load(uint32_t addr) {
    return *(const __attribute__((address_space(3))) T *)(lds_u8_t *)(uintptr_t)addr;
}

}  // namespace smg
