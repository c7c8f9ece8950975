// Staging of global memory into LDS, shared by the kernels that keep a ring of
// stages there (uqm_mfma.hip, uqm_dense.hip, uqm_prefill.hip).
#pragma once

#include "uqm_device.h"

namespace uqm {

// s_waitcnt with only vmcnt limited (gfx9 encoding: vmcnt bits 3:0 and 15:14):
// at most N of this wave's loads outstanding.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N <= 63, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// This wave's LDS reads complete, then the workgroup barrier. (Its loads into
// LDS are waited for separately, by stage; a plain __syncthreads would wait for
// all of them.)
__device__ __forceinline__ void stage_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), vmcnt and expcnt unlimited
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

// 16 or 4 bytes per lane from global memory into LDS at a wave-uniform LDS byte
// address (lane l's bytes at lds_addr + 16 l or + 4 l). (Helpers of their own:
// with the builtin written in a kernel's body the host compilation drops the
// kernel's launch stub.)
typedef __attribute__((address_space(3))) void stage_lds_t;

__device__ __forceinline__ void dma16_to(const void* src, uint32_t lds_addr) {
  __builtin_amdgcn_global_load_lds(src, reinterpret_cast<stage_lds_t*>(static_cast<uintptr_t>(lds_addr)), 16, 0, 0);
}
__device__ __forceinline__ void dma4_to(const void* src, uint32_t lds_addr) {
  __builtin_amdgcn_global_load_lds(src, reinterpret_cast<stage_lds_t*>(static_cast<uintptr_t>(lds_addr)), 4, 0, 0);
}

}  // namespace uqm
