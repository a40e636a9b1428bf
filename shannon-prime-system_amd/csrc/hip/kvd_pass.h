// kvd_pass.h -- what the kernels of a batched pass share: loads straight into
// LDS, and a prefill pass's pages and window starts.
#pragma once
#include "kvd_internal.h"

namespace kvd {

typedef int v4i __attribute__((ext_vector_type(4)));

// raw buffer descriptor of [base, base + bytes): reads past it return zero
__device__ __forceinline__ v4i rsrc_of(const void *base, uint32_t bytes) {
    const uint64_t b = (uint64_t)base;
    v4i r;
    r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    r.y = __builtin_amdgcn_readfirstlane((int)((uint32_t)(b >> 32) & 0xFFFFu));
    r.z = __builtin_amdgcn_readfirstlane((int)bytes);
    r.w = 0x00020000;                                  // 32-bit data format, stride 0
    return r;
}
// Loads straight into LDS (no registers): lane l's bytes at voff + soff go to
// LDS byte lds + 16 l (dma16) or, zero-extended, lds + 4 l (dma2).  The caller
// counts them (vmcnt) and waits before anyone reads the bytes.  Inline assembly,
// because the compiler waits for every load of its own builtin before any LDS
// read.  m0 is a reserved register (a clobber of it is refused): the compiler
// writes it itself right before its own uses, of which these kernels have none.
__device__ __forceinline__ void dma16(uint32_t lds, int voff, v4i rsrc, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 : : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void dma16(uint32_t lds, int voff, v4i rsrc) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 : : "s"(lds), "v"(voff), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void dma2(uint32_t lds, int voff, v4i rsrc, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_ushort %1, %2, %3 offen lds"
                 : : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

// the page of a position of the pass's session (every kv head's K rows, then V rows)
__device__ __forceinline__ const float *page_at(const AttnArgs &a, int pos) {
    const int lp = pos / PAGE;
    return gmem(a.pages)[a.ring_pages ? lp % a.ring_pages : lp];
}
// the first position token t of the pass attends
__host__ __device__ __forceinline__ int win_start(const AttnArgs &a, int t) {
    const int q = a.pos0 + t - a.win + 1;
    return a.win >= 0 && q > 0 ? q : 0;
}

}  // namespace kvd
