// Loads that go straight into LDS, and the waits for them.
#pragma once
#include "common.hpp"

namespace lsa {

typedef __attribute__((address_space(3))) unsigned char* lds_ptr_t;

// One load of a wavefront straight into LDS: lane i's 16 bytes go to `lds_address` + 16 i (a byte address in LDS, the
// same for all lanes).  Written out rather than called as a builtin: the compiler makes every later LDS read wait for
// all loads it knows to write LDS, and these are meant to stay in flight while the steps before them are read.
// A load that takes its LDS address from m0 wants one wait state behind the scalar instruction that wrote it; the compiler puts
// it there for its own loads (s_nop 0) and does not look into an asm block.
__device__ __forceinline__ void load_16_bytes_a_lane_to_lds(const void* source, unsigned lds_address) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(source), "s"(lds_address) : "memory", "m0");
}
// The same with one base for all lanes and a byte offset per lane.
__device__ __forceinline__ void load_16_bytes_a_lane_to_lds(const void* base, unsigned offset, unsigned lds_address) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_address) : "memory", "m0");
}

// Waits until at most PENDING of this wavefront's loads are still under way (they land in the order they were
// issued), then for the workgroup.  Written out because __syncthreads() would wait for every load, also for those
// of the steps ahead, which are meant to stay in flight across the barrier.
template <int PENDING>
__device__ __forceinline__ void loads_landed_then_barrier() {
    static_assert(PENDING >= 0 && PENDING < 64, "the counter of loads in flight has six bits");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PENDING) : "memory");
}

}  // namespace lsa
