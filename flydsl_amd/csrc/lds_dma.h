// Global -> LDS copies by DMA (buffer_load ... lds), issued from inline assembly.
#pragma once
#include "psg_common.h"

namespace {

// descriptor built from values forced into scalar registers (an inline-asm "s" operand must not end up in vector registers)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc_uniform(const void* base, uint64_t bytes) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)rsrc_bytes(bytes));
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>((uintptr_t)(((uint64_t)hi << 32) | lo)), 0, (int)n, 0x00020000);
}

// One DMA instruction: 64 lanes x 16 bytes from (descriptor, voff + soff) to LDS [lds_addr, lds_addr + 1024).
// A vector memory instruction must stay five wait states behind a vector instruction that wrote one of its scalar operands, and the compiler
// does not know that this statement is one: where scalar registers run short it fetched `soff` back from a vector register (v_readlane)
// directly in front.  So the offset goes through a scalar move, which waits by itself and is at the same time the wait state behind
// the write of M0 (the s_nop it replaces: the statement is no longer than before).  The descriptor must come from make_rsrc_uniform and
// stay in scalar registers; tests/test_wait_states.py looks at what was built.
// The compiler does not know either that the statement writes LDS (it would put a full vmcnt wait in front of every LDS read that
// follows): kernels wait for it themselves.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
    int so;
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b32 %0, %4\n\tbuffer_load_dwordx4 %2, %3, %0 offen lds" : "=&s"(so) : "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voff), "s"(r), "s"(__builtin_amdgcn_readfirstlane((int)soff))
                 : "memory");
}

// 4 bytes per lane: 64 lanes x 4 bytes to LDS [lds_addr, lds_addr + 256)
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t r, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
    int so;
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b32 %0, %4\n\tbuffer_load_dword %2, %3, %0 offen lds" : "=&s"(so) : "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(voff), "s"(r), "s"(__builtin_amdgcn_readfirstlane((int)soff))
                 : "memory");
}

}  // namespace
