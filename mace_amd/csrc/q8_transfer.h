// Transfers from global memory straight into LDS, and the wait for them, as the uint8 GEMM and convolution
// kernels use them.
#pragma once

#include "common.h"

namespace {

// global_load_lds: every lane fetches 16 bytes from its own address; the wavefront's 64 x 16 bytes land
// contiguously from lds_wave_base (the same in every lane) on.
__device__ inline void dma_16B(const uint8_t *g, uint8_t *lds_wave_base) {
  __builtin_amdgcn_global_load_lds(
      (const void __attribute__((address_space(1))) *)g,
      (void __attribute__((address_space(3))) *)lds_wave_base, 16, 0, 0);
}

// The same transfer addressed through a buffer descriptor: base (wave-uniform) + lane offset + scalar
// offset.  Preferred where the rows can be addressed this way: the compiler treats the global
// form as a FLAT access that may return through the LDS counter and then waits for ALL outstanding
// LDS reads (lgkmcnt(0)) wherever it needs one of them, for as long as a transfer is in flight,
// i.e. throughout the loops below; with the buffer form its waits name the read they need.
typedef __amdgpu_buffer_rsrc_t mh_rsrc;
__device__ inline mh_rsrc dma_rsrc(const uint8_t *base) {
  // raw buffer: stride 0, every 32-bit offset in range, DATA_FORMAT = 32-bit
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, -1, 0x00020000);
}
__device__ inline void dma_16B(mh_rsrc rs, uint32_t lane_off, uint32_t uniform_off, uint8_t *lds_wave_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (void __attribute__((address_space(3))) *)lds_wave_base,
                                           16, (int)lane_off, (int)uniform_off, 0, 0);
}

// s_waitcnt vmcnt(N) alone (expcnt / lgkmcnt fields left at "no wait"), or with LDS for the wavefront's LDS
// accesses too (lgkmcnt(0))
template <int N, bool LDS = false>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
  __builtin_amdgcn_s_waitcnt((LDS ? 0x0070 : 0x0f70) | (N & 15) | ((N >> 4) << 14));
}

}  // namespace
