// qh_lds.hpp -- loads from memory straight to LDS (gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qh {

// Buffer resource of `bytes` bytes at p (raw; word 3 as on the gfx9 family).
typedef uint32_t rsrc_v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ rsrc_v make_rsrc(const void* p, uint32_t bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    rsrc_v r = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b),
                (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(b >> 32) & 0xFFFFu)),
                (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    asm volatile("s_nop 4" : "+s"(r));  // the wait states of the loads that read it
    return r;
}

// 16 (or 4) bytes per lane from r + voff + soff to LDS at lds + lane * 16
// (or 4).  Out-of-range lanes write zeros.  The data has landed once the
// vector-memory counter says so (wait_vm below).
//
// Inline assembly, as the compiler's own form of these loads waits for all of
// them before every LDS access.  Its hazard pass does not look inside: the
// write of M0 gets its wait state here; an SGPR written by a vector
// instruction needs 5 before the load reads it, which make_rsrc gives the
// descriptor, and tests/test_lds_loads.py counts for every operand over the
// kernels' assembly.  (5 in front of each load cost the prefill GEMM 0.5-0.9 %.)
// M0 stays in the clobber list: it is not allocated, so there is nothing to
// preserve, and the compiler sets it right before its own uses; its warning
// about a reserved register is off for these statements alone.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load16(rsrc_v r, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(r), "s"(soff), "s"(lds)
                 : "memory", "m0");
}
__device__ __forceinline__ void lds_load4(rsrc_v r, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(r), "s"(soff), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
// Waits until at most N of this wave's vector-memory operations are in
// flight and all its LDS operations are done.
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}

// LDS address of a __shared__ object.
__device__ __forceinline__ uint32_t lds_address(void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)p;
}

}  // namespace qh
