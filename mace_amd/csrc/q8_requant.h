// Device side of the requantization shared by the uint8 GEMM and convolution kernels: one 64-bit
// multiply-add per output.  (Host side: RequantFixed, mh_make_requant in common.h; parameters outside
// this form take mh_requant_fixed there.)
#pragma once

#include "common.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

// ---- requantization by one 64-bit multiply-add per output ---------------------------------------
//
// clamp(RDivPOT(SRDHM(x, m), s) + zp, lo, hi) with m > 0 and s >= 1.  SRDHM(x, m) is
// y = floor((x m + 2^30) / 2^31), RDivPOT(y, s) is floor((y + 2^(s-1) - [y < 0]) / 2^s), and [x < 0]
// does for [y < 0] (where x < 0 and y = 0 both give 0).  A floor of a floor is a floor, so all of
// it is
//   z + zp = floor((x m + C - [x < 0] 2^31) / 2^(31+s)),   C = 2^30 + 2^(30+s) + zp 2^(31+s),
// a v_mad_i64_i32 (2.2 ns per wavefront on a SIMD; a 32-bit add takes 1.1) whose high dword, shifted
// right by s - 1 more, is the unclamped output.  v_ashr_pk_u8_i32 does that shift, the clamp to 0..255 and the packing of two outputs at once.  Outputs that zp and the clamp keep
// from ever being a z below 1 (zp = 0: a quantized ReLU) need no sign term: 1.5 instructions per
// output beside the correction terms' addition, 3.5 with it, 4.5 with a narrower clamp (the high
// dword is clamped to lo 2^(s-1) .. hi 2^(s-1)), against 7.75 and an LDS read by the table, which
// also had to be staged by every workgroup.  MobileNet's five pointwise layers at batch 64 85.2 ->
// 78.3 us, five spatial layers 121.0 -> 115.3, ten layers of one image 60.7 -> 59.5, 8192^3 499.6 ->
// 496.0.
// Exact for every x: with |x m| < 2^62 and (2 |zp| + 1) 2^(30+s) <= 2^62 no sum leaves 64 bits.
//
// s = 0 (a real multiplier of 1/2 and more) has no rounding shift: z = floor((2 x m + 2^31) / 2^32), no
// sign term and no shift of the high dword.  Where 2 m leaves 31 bits, x (2 m - 2^32) + 2^32 x stands for
// it: the high dword of the multiply-add by the wrapped 2 m, plus x, saturating.  At a multiplier of 0.7,
// batch 64: 224 x 224 x 3 -> 32 in the strip kernel 16.4 us (67.3 in the kernel that takes any
// parameters, 18.2 by the table), 56 x 56 x 32 -> 64 3 x 3 14.8 (22.9, 15.4).
//
// What this leaves out, offsets too large for the shift (128 from s = 24 on, where an output moves by at
// most one unit in 2^23), takes mh_requant_fixed in the kernels that have it.
struct RequantMad {
  int64_t c;
  int32_t mult, sh;
  int32_t lo, hi;        // bounds of the high dword
  bool no_sign, plus_x;  // no sign term needed; s = 0: the high dword lacks x
  bool clamp;            // a clamp narrower than 0..255
  bool more;             // plus_x or clamp: what most calls do without
};
__host__ __device__ inline bool requant_by_mad(const RequantFixed &rq) {
  if (rq.mult <= 0 || rq.shift < 0 || rq.shift > 31 || rq.blo < -32768 || rq.bhi > 32768) return false;
  const int64_t lo = (int64_t)rq.blo + rq.zp, hi = (int64_t)rq.bhi + rq.zp, away = rq.zp < 0 ? -(int64_t)rq.zp : rq.zp;
  if (lo < 0 || hi > 255) return false;
  if (rq.shift == 0) return true;
  // (the lower clamp must be reachable in the high dword; above its top nothing ever comes)
  return 2 * away + 1 <= ((int64_t)1 << (32 - rq.shift)) && (lo << (rq.shift - 1)) <= INT32_MAX;
}
__host__ __device__ inline RequantMad requant_mad(const RequantFixed &rq) {
  RequantMad m;
  const int s = rq.shift;
  const int lo = rq.blo + rq.zp, hi = rq.bhi + rq.zp;
  m.sh = s ? s - 1 : 0;
  m.mult = s ? rq.mult : (int32_t)((uint32_t)rq.mult << 1);
  m.plus_x = s == 0 && rq.mult >= (1 << 30);
  m.c = s ? ((int64_t)1 << 30) + ((int64_t)1 << (30 + s)) + (int64_t)rq.zp * ((int64_t)1 << (31 + s))
          : ((int64_t)1 << 31) + (int64_t)rq.zp * ((int64_t)1 << 32);
  const int64_t top = (int64_t)hi << m.sh;
  m.hi = top > INT32_MAX ? INT32_MAX : (int32_t)top;
  m.lo = lo << m.sh;
  m.clamp = lo != 0 || hi != 255;
  m.no_sign = s == 0 || (rq.zp <= 0 && !m.clamp);
  m.more = m.plus_x || m.clamp;
  return m;
}
// One accumulator on the host, in the same steps (for the CPU-side tests of the form).
__host__ __device__ inline int32_t requant_mad_one(int32_t x, const RequantMad &m) {
  int64_t w = (int64_t)x * m.mult + m.c;
  if (!m.no_sign && x < 0) w -= (int64_t)1 << 31;
  int64_t h = w >> 32;
  if (m.plus_x) h += x;
  h = h < INT32_MIN ? INT32_MIN : (h > INT32_MAX ? INT32_MAX : h);
  if (m.clamp) h = h < m.lo ? m.lo : (h > m.hi ? m.hi : h);
  h >>= m.sh;
  return (int32_t)(h < 0 ? 0 : (h > 255 ? 255 : h));
}
// Sixteen high dwords -> their bytes in four dwords: shifted right, clamped to 0..255, packed.
// Lower halves first, then the upper ones (op_sel: the result goes to the upper half and the lower
// half is kept).  Every caller swaps halves of the packed dwords next: a v_permlane32_swap must come
// at least two wait states after the vector instruction that writes an operand of it, and what the
// upper-half form writes may be read one after.  The compiler keeps those distances for instructions
// of its own but not for assembly, so the wait stands in the block, behind all eight.
__device__ __forceinline__ void requant_pack_16(const int32_t (&h)[16], int32_t sh, uint32_t (&packed)[4]) {
#if defined(__HIP_DEVICE_COMPILE__)   // (GPU instructions; the host pass never runs this)
  asm("v_ashr_pk_u8_i32 %0, %4, %5, %20\n\t"
      "v_ashr_pk_u8_i32 %1, %8, %9, %20\n\t"
      "v_ashr_pk_u8_i32 %2, %12, %13, %20\n\t"
      "v_ashr_pk_u8_i32 %3, %16, %17, %20\n\t"
      "v_ashr_pk_u8_i32 %0, %6, %7, %20 op_sel:[0,0,0,1]\n\t"
      "v_ashr_pk_u8_i32 %1, %10, %11, %20 op_sel:[0,0,0,1]\n\t"
      "v_ashr_pk_u8_i32 %2, %14, %15, %20 op_sel:[0,0,0,1]\n\t"
      "v_ashr_pk_u8_i32 %3, %18, %19, %20 op_sel:[0,0,0,1]\n\t"
      "s_nop 1"
      : "=&v"(packed[0]), "=&v"(packed[1]), "=&v"(packed[2]), "=&v"(packed[3])
      : "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(h[3]), "v"(h[4]), "v"(h[5]), "v"(h[6]), "v"(h[7]), "v"(h[8]),
        "v"(h[9]), "v"(h[10]), "v"(h[11]), "v"(h[12]), "v"(h[13]), "v"(h[14]), "v"(h[15]), "s"(sh));
#else
  for (int q = 0; q < 4; ++q) packed[q] = 0;
#endif
}
// Sixteen accumulators -> sixteen output bytes in four dwords.
__device__ __forceinline__ void requant_16_by_mad(const int32_t (&v)[16], const RequantMad &m,
                                                  uint32_t (&packed)[4]) {
  int32_t h[16];
#if defined(__HIP_DEVICE_COMPILE__)
  auto clamp = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      asm("v_med3_i32 %0, %1, %2, %3" : "=v"(h[r]) : "v"(h[r]), "s"(m.lo), "v"(m.hi));
  };
  if (m.no_sign) {
#pragma unroll
    for (int r = 0; r < 16; ++r) h[r] = (int32_t)(((int64_t)v[r] * m.mult + m.c) >> 32);
    if (__builtin_expect(m.more, 0)) {
      if (m.plus_x) {
#pragma unroll
        for (int r = 0; r < 16; ++r) h[r] = __builtin_elementwise_add_sat(h[r], v[r]);
      }
      clamp();
    }
  } else {
    int32_t k = INT32_MIN;
    asm("" : "+s"(k));   // opaque: a multiplication by it must stay the multiply-add it is
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t c = (int64_t)(int32_t)((uint32_t)v[r] >> 31) * k + m.c;
      h[r] = (int32_t)(((int64_t)v[r] * m.mult + c) >> 32);
    }
    if (m.clamp) clamp();
  }
#endif
  requant_pack_16(h, m.sh, packed);
}

}  // namespace
