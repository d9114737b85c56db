// What the kernels with two groups of waves in alternating roles share (gemm_pingpong.hip, moe_pingpong.hip): pieces of a half-tile
// brought in by LDS-DMA, counted waits for them, barriers that nothing is moved across.
#pragma once
#include "common.h"

namespace dlia {

constexpr int kPPThreads = 512;
constexpr int kPPHalf = 16384;                   // bytes of one half-tile

// Two 1 KiB pieces, global -> LDS, under ONE setting of M0: lane l of piece i lands at
// lds_addr + 1024 i + 16 l and reads g_i + 16 bytes per lane as set up by the caller. The second
// piece uses the instruction's immediate offset, which advances the global AND the LDS address, so
// its source pointer is passed 1024 bytes low. Why one setting: a write to M0 waits until every
// earlier LDS-DMA instruction of the wave has read it, ~180 cycles after issue — with M0 written
// (and restored) around every piece a wave issues one piece per ~180 cycles and a CU takes 32 bytes
// per cycle from L2, with four pieces per setting 63 (bench/l2_lds_bw.hip). M0 is not restored:
// nothing else in this kernel uses it (no other LDS-DMA, no indexed register access).
__device__ __forceinline__ void pp_dma_pair(const void* g0, const void* g1_minus_1k, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
               "global_load_lds_dwordx4 %2, off offset:1024"
               :: "s"(lds_addr), "v"(g0), "v"(g1_minus_1k) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void pp_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}
// what the wave wrote to LDS is there, and everyone's behind the barrier (s_barrier alone does not wait for LDS writes)
__device__ __forceinline__ void pp_staged() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  pp_barrier();
}

}  // namespace dlia
