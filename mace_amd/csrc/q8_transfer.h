// Transfers from global memory straight into LDS, and the wait for them, as the uint8 GEMM and convolution
// kernels use them; pieces that end with their operand.
#pragma once

#include "common.h"
#include "q8_requant.h"

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

// A piece of which less than 16 bytes are left in the operand was loaded `early` (below 16) bytes before its place: moved
// down to it, zeros behind.
__device__ __forceinline__ v4i moved_down(const v4i &v, uint32_t early) {
  const bool two = (early & 8) != 0, one = (early & 4) != 0;
  const uint32_t a0 = (uint32_t)(two ? v.z : v.x), a1 = (uint32_t)(two ? v.w : v.y), a2 = two ? 0u : (uint32_t)v.z,
                 a3 = two ? 0u : (uint32_t)v.w;
  const uint32_t b0 = one ? a1 : a0, b1 = one ? a2 : a1, b2 = one ? a3 : a2, b3 = one ? 0u : a3;
  const uint32_t by = early & 3;
  return v4i{(int)__builtin_amdgcn_alignbyte(b1, b0, by), (int)__builtin_amdgcn_alignbyte(b2, b1, by),
             (int)__builtin_amdgcn_alignbyte(b3, b2, by), (int)__builtin_amdgcn_alignbyte(0u, b3, by)};
}

// s_waitcnt vmcnt(N) alone (expcnt / lgkmcnt fields left at "no wait"), or with LDS for the wavefront's LDS
// accesses too (lgkmcnt(0))
template <int N, bool LDS = false>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
  __builtin_amdgcn_s_waitcnt((LDS ? 0x0070 : 0x0f70) | (N & 15) | ((N >> 4) << 14));
}

}  // namespace
