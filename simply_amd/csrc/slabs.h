// What the kernels share that bring operands into LDS by loads of their own count: waits for the loads under way, and a barrier that
// waits for nothing else.
#pragma once
#include "common.h"

namespace sa {
namespace slabs {

// s_waitcnt for "at most n vector-memory loads outstanding" and nothing else (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4, lgkmcnt 11:8)
constexpr int waitcnt_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// The workgroup barrier alone; the empty statements and the scheduling barriers keep the compiler from moving memory
// accesses across it.
__device__ inline void bare_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

}  // namespace slabs
}  // namespace sa
