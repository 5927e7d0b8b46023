// Direct global -> LDS pipelines of the prefill GEMMs: the 16-byte direct
// load, the partial vmcnt wait that proves a stage landed (loads of one size
// complete in issue order) and the barrier for LDS data alone.
#pragma once
#include "common.hpp"

namespace w4a16 {

// s_waitcnt immediate for vmcnt <= n with expcnt and lgkmcnt not waited for
// (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
constexpr int px_vm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// s_waitcnt vmcnt(n) for a wavefront-uniform n <= 15 (more waits for all)
__device__ __forceinline__ void px_wait_vm(int n) {
  switch (n) {
    case 1: __builtin_amdgcn_s_waitcnt(px_vm_wait(1)); break;
    case 2: __builtin_amdgcn_s_waitcnt(px_vm_wait(2)); break;
    case 3: __builtin_amdgcn_s_waitcnt(px_vm_wait(3)); break;
    case 4: __builtin_amdgcn_s_waitcnt(px_vm_wait(4)); break;
    case 5: __builtin_amdgcn_s_waitcnt(px_vm_wait(5)); break;
    case 6: __builtin_amdgcn_s_waitcnt(px_vm_wait(6)); break;
    case 7: __builtin_amdgcn_s_waitcnt(px_vm_wait(7)); break;
    case 8: __builtin_amdgcn_s_waitcnt(px_vm_wait(8)); break;
    case 9: __builtin_amdgcn_s_waitcnt(px_vm_wait(9)); break;
    case 10: __builtin_amdgcn_s_waitcnt(px_vm_wait(10)); break;
    case 11: __builtin_amdgcn_s_waitcnt(px_vm_wait(11)); break;
    case 12: __builtin_amdgcn_s_waitcnt(px_vm_wait(12)); break;
    case 13: __builtin_amdgcn_s_waitcnt(px_vm_wait(13)); break;
    case 14: __builtin_amdgcn_s_waitcnt(px_vm_wait(14)); break;
    case 15: __builtin_amdgcn_s_waitcnt(px_vm_wait(15)); break;
    default: __builtin_amdgcn_s_waitcnt(px_vm_wait(0)); break;
  }
}

// Workgroup barrier for LDS data only: each wavefront waits for its own LDS
// operations, then meets the others.  (__syncthreads() would also wait for
// every global load in flight, the direct LDS loads of the next stages
// included.)  The wait is the builtin, not part of the asm, so that the
// compiler knows the LDS reads before it are done: without that a register
// read before the barrier makes it wait for the reads issued after it too.
__device__ __forceinline__ void px_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
}

// direct global -> LDS load: lane l's 16 bytes land at lds_dst + 16 l
__device__ __forceinline__ void px_dma16(__amdgpu_buffer_rsrc_t rsrc, int voff, int soff, void* lds_dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds_dst, 16,
                                          voff, soff, 0, 0);
}

}  // namespace w4a16
