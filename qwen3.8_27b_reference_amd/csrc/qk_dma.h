// LDS-DMA building blocks shared by the streaming kernels (GEMV, GEMM): global memory into LDS without
// VGPRs, hand-counted waits and a barrier that leaves the DMAs in flight.
#pragma once

#include "qk_device.h"

namespace qk {

#define LDS_AS __attribute__((address_space(3)))

// Wait until at most N vector-memory operations of this wave are outstanding.  The compiler does
// not track LDS-DMA completion for later LDS reads, so the ring waits explicitly; the memory
// clobber keeps the compiler from moving LDS accesses across the wait.
template <int N>
__device__ inline void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int N>
__device__ inline void wait_vm_le(int n) {  // wait until at most n (<= N) operations are in flight
    if constexpr (N > 0) {
        if (n >= N) {
            wait_vm<N>();
            return;
        }
        wait_vm_le<N - 1>(n);
    } else {
        wait_vm<0>();
    }
}

template <int STEP>
__device__ inline void wait_vm_units(int k) {  // k = units still allowed in flight (0..2)
    if (k <= 0) wait_vm<0>();
    else if (k == 1) wait_vm<STEP>();
    else wait_vm<2 * STEP>();
}

__device__ inline uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(LDS_AS const void*)p; }

// Work-group barrier that waits only for this wave's LDS operations (not for its LDS-DMAs, as the
// release fence of __syncthreads() would); the empty asm keeps memory accesses on their side.
__device__ inline void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 16 bytes per lane from global memory into LDS (M0 + 16 * lane), without VGPRs.  Issued from inline
// assembly: the compiler then never holds a pending LDS-DMA, which it would otherwise wait out
// (vmcnt(0), the whole ring) before every LDS access it cannot prove disjoint from the destination,
// and before the lane-masked ones it could not count at all.  Every read of DMA'd bytes follows an
// explicit wait_vm*; an operation the compiler does not count only makes its own waits (for the
// loads it issued earlier) more conservative.  The LDS base goes in M0 (an input the compiler
// sets); s_nop: M0 written by the SALU needs one wait state before an LDS-DMA reads it.
__device__ inline void dma16(const void* g, uint8_t* lds) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds_addr(lds)) : "memory");
}
// The same for weight bytes, which a call reads exactly once: non-temporal, so that the stream does
// not push the activation (read by every CU) out of L2.  Measured on MI355X: the single-token GEMV
// takes 13.0 us instead of 14.4 (K=5120, N=17408) and 19.2 instead of 20.5 (K=17408, N=5120).
__device__ inline void dma16_stream(const void* g, uint8_t* lds) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(g), "{m0}"(lds_addr(lds)) : "memory");
}

// dma16_stream on lanes 0 .. LANES - 1 only, with the lane mask applied inside the assembly: a
// lane-masked call in C++ becomes an exec-skip branch around the DMA, and on that (never taken)
// path the vmcnt waits that count this DMA would no longer cover the loads they wait for, so the
// code could not be checked path by path.  exec is restored before the statement ends.
template <int LANES>
__device__ inline void dma16_stream_lanes(const void* g, uint8_t* lds) {
    static_assert(LANES > 0 && LANES < 64, "a partial wave");
    constexpr uint64_t MASK = (1ull << LANES) - 1;
    uint64_t saved;
    asm volatile("s_and_saveexec_b64 %0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt\n\ts_mov_b64 exec, %0"
                 : "=&s"(saved)
                 : "v"(g), "s"(MASK), "{m0}"(lds_addr(lds))
                 : "memory", "scc");
}

// One weight group into an LDS slot: 1 KiB per instruction, the last one on the lanes it needs
// (every instruction has live lanes, so each one counts once on vmcnt), with no branch.
template <int GB>
__device__ inline void dma_group(const uint8_t* G, uint8_t* slot, int lane) {
    static_assert(GB % 16 == 0, "16-byte pieces");
    constexpr int FULL = GB / 1024, TAIL = (GB % 1024) / 16;
#pragma unroll
    for (int c = 0; c < FULL; c++) dma16_stream(G + c * 1024 + 16 * lane, slot + c * 1024);
    if constexpr (TAIL > 0) dma16_stream_lanes<TAIL>(G + FULL * 1024 + 16 * lane, slot + FULL * 1024);
}

}  // namespace qk
