// Device side of the requantization shared by the uint8 GEMM and convolution kernels: the 64-bit
// multiply-add form that nearly every call takes, and for parameters outside it the comparison table
// in LDS with the sixteen-at-a-time look-up.  (Host side: RequantFixed, mh_make_requant,
// mh_requant_table_cached in common.h.)
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
// a v_mad_i64_i32 (full rate here: 4.9 cycles per wavefront measured, a 32-bit add 4.6) whose high
// dword, shifted right by s - 1 more, is the unclamped output.  v_ashr_pk_u8_i32 does that shift,
// the clamp to 0..255 and the packing of two outputs at once.  Outputs that zp and the clamp keep
// from ever being a z below 1 (zp = 0: a quantized ReLU) need no sign term: 1.5 instructions per
// output beside the correction terms' addition, 3.5 with it, 4.5 with a narrower clamp (the high
// dword is clamped to lo 2^(s-1) .. hi 2^(s-1)), against 7.75 and an LDS read by the table, which
// also had to be staged by every workgroup.  MobileNet's five pointwise layers at batch 64 85.2 ->
// 78.3 us, five spatial layers 121.0 -> 115.3, ten layers of one image 60.7 -> 59.5, 8192^3 499.6 ->
// 496.0.
// Exact for every x: |x m| < 2^62 and, with |zp| 2^(31+s) <= 2^61, no sum leaves 64 bits.
struct RequantMad {
  int64_t c;
  int32_t mult, sh;
  int32_t lo, hi;        // bounds of the high dword
  bool positive, clamp;  // no sign term needed; a clamp narrower than 0..255
};
__host__ __device__ inline bool requant_by_mad(const RequantFixed &rq) {
  if (rq.mult <= 0 || rq.shift < 1 || rq.shift > 30 || rq.blo < -32768 || rq.bhi > 32768) return false;
  const int64_t room = (int64_t)1 << (30 - rq.shift);
  const int64_t lo = (int64_t)rq.blo + rq.zp, hi = (int64_t)rq.bhi + rq.zp;
  // (the lower clamp must be reachable in the high dword; above its top nothing ever comes)
  return rq.zp <= room && -(int64_t)rq.zp <= room && lo >= 0 && hi <= 255 &&
         (lo << (rq.shift - 1)) <= INT32_MAX;
}
__host__ __device__ inline RequantMad requant_mad(const RequantFixed &rq) {
  RequantMad m;
  const int s = rq.shift;
  m.mult = rq.mult;
  m.sh = s - 1;
  m.c = ((int64_t)1 << 30) + ((int64_t)1 << (30 + s)) + (int64_t)rq.zp * ((int64_t)1 << (31 + s));
  const int lo = rq.blo + rq.zp, hi = rq.bhi + rq.zp;
  const int64_t top = (int64_t)hi << m.sh;
  m.hi = top > INT32_MAX ? INT32_MAX : (int32_t)top;
  m.lo = lo << m.sh;
  m.clamp = lo != 0 || hi != 255;
  m.positive = rq.zp <= 0 && lo == 0 && !m.clamp;
  return m;
}
// One accumulator on the host, in the same steps (for the CPU-side tests of the form).
__host__ __device__ inline int32_t requant_mad_one(int32_t x, const RequantMad &m) {
  int64_t w = (int64_t)x * m.mult + m.c;
  if (!m.positive && x < 0) w -= (int64_t)1 << 31;
  int32_t h = (int32_t)(w >> 32);
  if (m.clamp) h = h < m.lo ? m.lo : (h > m.hi ? m.hi : h);
  h >>= m.sh;
  return h < 0 ? 0 : (h > 255 ? 255 : h);
}
// Sixteen accumulators -> sixteen output bytes in four dwords.
__device__ __forceinline__ void requant_16_by_mad(const int32_t (&v)[16], const RequantMad &m,
                                                  uint32_t (&packed)[4]) {
#if defined(__HIP_DEVICE_COMPILE__)   // (GPU instructions; the host pass never runs this)
  int32_t h[16];
  if (m.positive) {
#pragma unroll
    for (int r = 0; r < 16; ++r) h[r] = (int32_t)(((int64_t)v[r] * m.mult + m.c) >> 32);
  } else {
    int32_t k = INT32_MIN;
    asm("" : "+s"(k));   // opaque: a multiplication by it must stay the multiply-add it is
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t c = (int64_t)(int32_t)((uint32_t)v[r] >> 31) * k + m.c;
      h[r] = (int32_t)(((int64_t)v[r] * m.mult + c) >> 32);
    }
    if (m.clamp) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        asm("v_med3_i32 %0, %1, %2, %3" : "=v"(h[r]) : "v"(h[r]), "s"(m.lo), "v"(m.hi));
    }
  }
  // Lower halves first, then the upper ones (op_sel: the result goes to the upper half and the lower
  // half is kept).  Every caller swaps halves of the packed dwords next: a v_permlane32_swap must come
  // at least two wait states after the vector instruction that writes an operand of it, and what the
  // upper-half form writes may be read one after.  The compiler keeps those distances for instructions
  // of its own but not for assembly, so the wait stands in the block, behind all eight.
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
        "v"(h[9]), "v"(h[10]), "v"(h[11]), "v"(h[12]), "v"(h[13]), "v"(h[14]), "v"(h[15]), "s"(m.sh));
#else
  for (int q = 0; q < 4; ++q) packed[q] = 0;
#endif
}

// Comparison table of the threshold requantization (RequantFixed::table), passed as the kernel
// argument that follows the parameter struct.  The kernels never name it: they read it from the
// argument segment, right after their parameters, with a lane-dependent index.
struct RequantTable {
  int32_t t[MH_REQUANT_TABLE_MAX];
};

// The comparison table as the kernels keep it in LDS: entry c (8 bytes) = {largest accumulator
// that does not reach step c + 1, output value of step c}.  A kernel argument (RequantTable) holds the
// first halves (see mh_requant_table_entry); the kernels read it from the argument segment with a
// lane-dependent index (indexing a by-value copy that way would spill it).
constexpr int MH_REQUANT_PAIRS_BYTES = 8 * (MH_REQUANT_TABLE_MAX - 1);
__device__ inline void stage_requant_pairs_from(const int32_t *arg_tab, int32_t *pairs,
                                                const RequantFixed &rq, int tid, int nthreads) {
  for (int c = tid; c <= rq.n; c += nthreads) {
    pairs[2 * c] = arg_tab[c + 1];
    pairs[2 * c + 1] = rq.lo + c;
  }
}
// The float estimate of the step index with the table's LDS address folded in: the mantissa trick
// of mh_requant_step_estimate yields 8 * (step index) as the low bits of the float; adding the
// table's address / 8 to the offset and to both clamp bounds makes those bits the entry's LDS
// address itself, so the look-up needs no address arithmetic (a vector add per output otherwise).
// All values stay integers (+ 7/8) below 2^21, where a float's last bit is worth 1/8: exact.
struct RequantLds {
  float inv, off, lo, top;
};
__device__ __forceinline__ RequantLds requant_lds(const RequantFixed &rq, const int32_t *pairs) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t addr = (uint32_t)(const __attribute__((address_space(3))) int32_t *)pairs;
#else
  const uint32_t addr = 0;
#endif
  const float t0 = (float)(addr >> 3);   // the table is 8-byte aligned; LDS addresses are below 2^18
  return RequantLds{rq.inv, rq.off + t0, MH_REQUANT_MAGIC + t0, rq.top + t0};
}
// Sixteen accumulators -> sixteen output bytes in four dwords.  Estimates first, then all
// look-ups, then the compares: sixteen LDS reads in flight instead of one round trip per element.
__device__ __forceinline__ void requant_16_by_table(const int32_t (&v)[16], const RequantLds &rq,
                                                    uint32_t (&packed)[4]) {
  typedef int pair_t __attribute__((ext_vector_type(2)));
  uint32_t a[16];
  pair_t e[16];
#pragma unroll
  for (int r = 0; r < 16; ++r)
    a[r] = __float_as_uint(__builtin_amdgcn_fmed3f(__fmaf_rn((float)v[r], rq.inv, rq.off), rq.lo,
                                                   rq.top)) & 0x3FFF8u;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
#if defined(__HIP_DEVICE_COMPILE__)   // (an LDS pointer is 32 bits wide in the device pass only)
    e[r] = *(const __attribute__((address_space(3))) pair_t *)a[r];
#else
    e[r] = pair_t{0, 0};
#endif
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t o[4];
#if defined(__HIP_DEVICE_COMPILE__)
    // o = out + (v > limit), four at a time: the compares first, each into a lane mask of its own,
    // then the four additions with the mask as carry.  A compare's mask cannot be consumed by the
    // very next instructions (the compiler, left alone, reuses one mask register and waits
    // between every compare and its addition).
    uint64_t m0, m1, m2, m3;
    asm("v_cmp_gt_i32_e64 %4, %8, %12\n\t"
        "v_cmp_gt_i32_e64 %5, %9, %13\n\t"
        "v_cmp_gt_i32_e64 %6, %10, %14\n\t"
        "v_cmp_gt_i32_e64 %7, %11, %15\n\t"
        "v_addc_co_u32_e64 %0, %4, 0, %16, %4\n\t"
        "v_addc_co_u32_e64 %1, %5, 0, %17, %5\n\t"
        "v_addc_co_u32_e64 %2, %6, 0, %18, %6\n\t"
        "v_addc_co_u32_e64 %3, %7, 0, %19, %7"
        : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3]), "=&s"(m0), "=&s"(m1), "=&s"(m2), "=&s"(m3)
        : "v"(v[4 * q]), "v"(v[4 * q + 1]), "v"(v[4 * q + 2]), "v"(v[4 * q + 3]), "v"(e[4 * q].x),
          "v"(e[4 * q + 1].x), "v"(e[4 * q + 2].x), "v"(e[4 * q + 3].x), "v"(e[4 * q].y),
          "v"(e[4 * q + 1].y), "v"(e[4 * q + 2].y), "v"(e[4 * q + 3].y));
#else
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (uint32_t)(e[4 * q + i].y + (v[4 * q + i] > e[4 * q + i].x ? 1 : 0));
#endif
    // bytes 0 of o[0..3] side by side (v_perm_b32: selector 0..3 = bytes of the second operand,
    // 4..7 of the first, 0x0c = zero)
    const uint32_t p10 = __builtin_amdgcn_perm(o[1], o[0], 0x0c0c0400u);
    const uint32_t p32 = __builtin_amdgcn_perm(o[3], o[2], 0x0c0c0400u);
    packed[q] = (p32 << 16) | p10;
  }
}

}  // namespace
