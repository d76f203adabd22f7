// Direct-to-LDS loads and the waits of a ring of LDS stages, shared by the GEMM with both tiles in LDS
// (tw4_gemm_lds.hip) and the dense fp16 kernel for small batches (tw4_dense.hip).
#pragma once

#include "tw4_common.h"

namespace tw4 {

typedef __attribute__((address_space(3))) const void lds_void;

// Direct-to-LDS loads: lane l's 16 (4) bytes at global `voff` (`src`) go to LDS byte address base + IMM + 16 l (4 l),
// base wavefront-uniform. Issued as inline assembly so that the compiler, which cannot tell the ring's slots apart for
// these loads, does not add a wait for every load in flight before each LDS read; the ring waits with explicit vmcnt
// counts instead, and the loop holds no other vector memory operation. M0 carries the LDS address, one wait state
// after it is written (the M0 -> LDS-DMA hazard).
// The 16-byte form goes through a buffer resource: the part of the address that moves with the stage is one 32-bit
// scalar offset, the lane's own offset is fixed for the whole kernel, and a resource of no records turns the load into
// one that reads nothing (zeros), which is how the stages past the end keep the loop's counts without a branch: the range
// check takes lane and scalar offset together, whatever the scalar one (no records at an offset of 4 KB: zeros; 4608 bytes: the first
// 512 from there).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register: the clobber is what tells the compiler
template <int IMM, bool NT = false>  // NT: non-temporal, data that is read once
__device__ __forceinline__ void lds_dma16(const u4& rsrc, uint32_t voff, uint32_t soff, uint32_t base) {
    if constexpr (NT)
        asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds"
                     :: "v"(voff), "s"(rsrc), "s"(soff), "s"(base), "n"(IMM) : "memory", "m0", "scc");
    else
        asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                     :: "v"(voff), "s"(rsrc), "s"(soff), "s"(base), "n"(IMM) : "memory", "m0", "scc");
}
template <int IMM>
__device__ __forceinline__ void lds_dma4(const void* src, uint32_t base) {
    asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
                 :: "v"(src), "s"(base), "n"(IMM) : "memory", "m0", "scc");
}
#pragma clang diagnostic pop

// Wait until at most N of this wavefront's vector memory operations are in flight and its LDS reads are done.
template <int N>
__device__ __forceinline__ void wait_stage() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(N) : "memory");
}

// A workgroup barrier that orders no memory by itself (the LDS data it guards was waited for with
// wait_stage): s_barrier between two compiler-only fences, so no LDS access moves across it.
__device__ __forceinline__ void ring_barrier() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A buffer resource over everything from `base` on (word 2: the records in bytes; 0 makes every load read nothing).
__device__ __forceinline__ u4 lds_rsrc(const void* base) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    return u4{static_cast<uint32_t>(b), static_cast<uint32_t>(b >> 32) & 0xFFFFu, 0xFFFFFFFFu, static_cast<uint32_t>(kBufferFlags)};
}

}  // namespace tw4
