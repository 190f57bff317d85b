// Memory straight into LDS, and what goes with it: buffer loads that write LDS by themselves, a
// barrier that leaves the newest of them on their way, and the order in which rows lie there.
#pragma once

#include "hal_common.h"

typedef __amdgpu_buffer_rsrc_t hal_memory;

// `bytes` bytes from p on (the same in all lanes); what lies past them reads as 0 and is not written
__device__ __forceinline__ hal_memory hal_memory_at(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// 16 bytes a lane: from byte `each` (a lane's own) + `all` of `from`, lane l's to `to` (the same in all lanes) + 16 l.
// (Buffer loads: the compiler waits for every load where it meets one in the flat form that goes into LDS.
// And buffers in LDS are arrays of their own, so that it can tell a load into one from a read of another.)
// HAL_ONCE: for what one workgroup reads, once, in whole lines, and nobody after it: caches pass it on.  (537 MB in runs of 32 KB a wave
// 91 us, 84 with it; in half lines, the other half of which then comes from memory again, 110 and 144.)
#define HAL_ONCE 2
template <int HOW = 0>
__device__ __forceinline__ void hal_load_lds(hal_memory from, uint32_t each, uint32_t all, void* to) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)to, 16, each, all, 0, HOW);
}

// Until all but the last `LEFT` accesses to memory of this wave are done, and then until every wave is here.
template <int LEFT>
__device__ __forceinline__ void hal_meet() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// LDS holds 8 rows x 64 k of bf16 as one KiB, eight lanes of a load a row: the piece of eight k that lies
// at place p of row r is piece p ^ hal_turn(r % 16).  A 16-byte read of a wave goes through LDS in turns of
// sixteen lanes, lanes 0-3, 12-15 and 20-27 in one and 4-11, 16-19 and 28-31 in the next (and so on from
// lane 32); each turn then meets all 64 banks once.
__device__ __forceinline__ int hal_turn(int r) { return ((r >> 1) & 1) | ((r >> 2) & 2) | (((r >> 1) ^ r) & 4); }
