// fp32 Gemm / Gemv on CDNA4.
//
// Gemm replaces delegator::Gemm for float (contract mace/ops/delegator/gemm.h:42-69,
// semantics mace/ops/ref/gemm.cc:58-146; the NEON implementation it stands in for is
// mace/ops/arm/base/gemm.cc:520-683): out[b] = lhs[b or 0] * rhs[b or 0] with each of the
// three matrices RowMajor or ColMajor.  The NEON kernel packs both operands into cache
// panels; here the panels are LDS tiles of the operands' three bf16 parts (below).  Products are
// good to binary32 and sums are binary32; the summation order differs from the reference's serial k
// loop, which the reference's own tolerance (1e-4 relative + 1e-2 absolute) covers.
//
// Gemv replaces delegator::Gemv for float (mace/ops/delegator/gemv.h:35-44,
// mace/ops/ref/gemv.cc:46-81): rows in slices by 16-byte pieces, up to 16 vectors a pass, or one row a wavefront.
#include <math.h>

#include <type_traits>

#include "common.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int TM = 128, TN = 128, TK = 16;   // (TK: the unit a k split deals out)

struct F32GemmParams {
  const float *lhs, *rhs;
  float *out;
  int64_t lrs, lcs;   // lhs element strides for (row, depth)
  int64_t rrs, rcs;   // rhs element strides for (depth, col)
  int64_t ors, ocs;   // out element strides for (row, col)
  int64_t lbs, rbs, obs;
  int M, N, K;
  int flat;   // columns per batch where the columns of all batches are one long row of N (0: not so)
  const float *bias_row;   // added per result row (a convolution's output channel), or nullptr
  const float *bias_col;   // added per result column (MatMul's bias), or nullptr
  int act;
  float limit;
  int tiles_m;
  // k split: blockIdx.y takes k tiles [y kt_split, (y + 1) kt_split) and
  // stores its raw sums into part[y part_stride + ...] with the result's own strides;
  // f32_ksplit_reduce_kernel adds the parts in the order of y and applies bias and activation.
  // kt_split = 0: no split.
  float *part;
  int64_t part_stride;   // elements of one part: the whole result
  int kt_split;
};

// Which tile of which batch a workgroup computes.  Workgroup ids (tiles of a batch first, then the
// batches) go round-robin to the 8 XCDs, each with an L2 of its own: left alone every XCD would
// hold a few tiles of every batch and pull all operands through its L2.  Every XCD gets a
// contiguous span of (batch, tile) instead.
__device__ inline void span_of_block(int *bid, int *b) {
  *bid = blockIdx.x;
  *b = blockIdx.z;
  const int nwg = gridDim.x * gridDim.z;
  if (nwg % 8 != 0) return;
  int wg = blockIdx.x + gridDim.x * blockIdx.z;
  wg = (wg % 8) * (nwg / 8) + wg / 8;
  *b = wg / gridDim.x;
  *bid = wg - *b * gridDim.x;
}

__device__ inline float apply_act(float v, int act, float limit) {
  // mace/ops/ref/activation.cc:61-75
  if (act == MACE_HIP_ACT_RELU) return fmaxf(0.f, v);
  if (act == MACE_HIP_ACT_RELUX) return fmaxf(0.f, fminf(limit, v));
  return v;
}

// ---- the tile kernels: binary32 products out of bf16 matrix instructions --------------------------
//
// v_mfma_f32_32x32x2_f32 multiplies 64 binary32 pairs per cycle and SIMD, v_mfma_f32_32x32x16_bf16
// sixteen times as many bf16 pairs into the same binary32 accumulators.  A binary32 number is the
// sum of three bf16 numbers, EXACTLY: hi = bf16(x) (to nearest), mid = bf16(x - hi),
// lo = x - hi - mid; x - hi has at most 16 significant bits, what mid leaves of it at most 7.  Of the
// nine products of two such sums the kernels form the six largest and leave out mid lo, lo mid and
// lo lo: with |mid| <= 2^-8 |x| and |lo| <= 2^-17 |x| (to nearest, so of either sign) that is at most
// 2^-24 |a b|.  The six go into one binary32 accumulator, sixteen depths per instruction, so the running
// sum is rounded less often than with two depths per instruction.  2-norm error against binary64, the
// binary32 instruction's first: 4 x 1024^3, normal operands, 4.1e-7 and 1.9e-7; 2304 x 2200 outputs (four
// wavefronts) 1.0e-7 and 6.9e-8 at depth 32, 7.4e-8 and 3.4e-8 at 16, 3.6e-8 and 3.3e-8 at 3, 3.1e-8 and
// 3.4e-8 at 2.  One product alone is off by up to 0.9 units in the last place with eight wavefronts and 1.4
// with four, where the binary32 instruction rounds it to nearest: depths 1 and 2 go to f32_fill_kernel
// for that.  (Rows with one entry other than zero keep it; where that entry is a power of two the product
// is exact.)  In time, 4 x 1024^3 against transposed weights 86.0 -> 50.0 us, MobileNet's five pointwise layers
// at batch 64 688 -> 291 us.  The matrix cores are busy 42 - 51 % of 4 x 1024^3 and 12 - 35 % of the pointwise
// layers; the rest is each k tile's chain of LDS reads, MFMAs, LDS writes and barrier (one to three workgroups
// per CU overlap) and, at short depths, the first loads and the stores of every tile.
//
// Both operands are multiplied by 2^23 before the split and the sums by 2^-46 behind it, all exact: the
// last bit of the smallest subnormal number then lies at 2^-126, so every part of every number is a
// normal bf16 number or zero, and values of any smallness (the tails of a softmax) go at one speed.
// That replaces a test for bits the split would lose: the loop takes as long as with it (4 x 1024^3 50.4
// and 50.1 us, 2304 x 512 x 2304 45.7 and 44.4).
//
// What the scaled split cannot take are operands from about 2^105 on, sums from 2^82 on, and numbers that
// are not finite.  They leave a sum that is not finite, and the workgroup computes its tile again with
// the binary32 instruction (`again` in f32_tile): with an infinity in every tile 4 x 1024^3 takes 140 us.
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t bf16_pair(float x, float y) {   // to nearest even; x in the low half
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t d;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(d) : "v"(x), "v"(y));
  return d;
#else
  return 0;
#endif
}
__device__ __forceinline__ float bf16_low(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_high(uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); }

constexpr float SPLIT_SCALE = 0x1p23f, SUM_SCALE = 0x1p-46f;

// Eight consecutive depths of one row (or column) as three 16-byte pieces: an MFMA fragment each.
__device__ __forceinline__ void split_8(const float (&x)[8], u4v (&part)[3]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x0 = x[2 * e] * SPLIT_SCALE, x1 = x[2 * e + 1] * SPLIT_SCALE;
    const uint32_t hi = bf16_pair(x0, x1);
    const float r0 = x0 - bf16_low(hi), r1 = x1 - bf16_high(hi);
    const uint32_t mid = bf16_pair(r0, r1);
    const float s0 = r0 - bf16_low(mid), s1 = r1 - bf16_high(mid);
    part[0][e] = hi;
    part[1][e] = mid;
    part[2][e] = bf16_pair(s0, s1);
  }
}

// A TMT x 128 tile of the result per workgroup.  LK / RK: the operand is contiguous along depth (true)
// or along its outer index (false).  SPLIT = 1: four wavefronts of 64 x 64 (TMT = 64: of 64 x 32), k
// tiles of 16, up to three workgroups per CU; SPLIT = 2: eight wavefronts of 64 x 32, k tiles of 32,
// for launches of at most one tile per CU, where one wavefront per SIMD would leave every LDS wait
// exposed.
// GUARD: depths that are not whole k tiles of 16, or an operand that is contiguous along depth in
// rows that are not aligned 16-byte pieces: the same loads at any address; a unit that the depth ends in is read early
// and moved down to its place in the last k tile (depths below 8, one k tile: single loads, each checked).  With every load
// checked by itself, us, before and now: 3000 x 1000 x 1200 75 and 53 (1008 deep 51), 3000 x 1001 x 1201 against
// transposed weights 104 and 50, 5000 x 300 x 2000 96 and 48, 627 x 1603 x 832 39 and 25.  Behind the last k tile
// nothing is split, stored or requested, and depths below 8 load no other: 1288 x 9 x 1554 10.9 -> 7.8, 1252 x 5 x 800
// 8.9 -> 6.2, 3615 x 20 x 490 against transposed weights 10.0 -> 7.3.
//
// A thread's unit is eight consecutive depths of one row: two 16-byte loads where depth is
// contiguous, else eight 4-byte loads, each coalesced over the wavefront's 64 rows (so rows of any
// length and alignment).  It splits them (about 6 vector instructions per element, once per tile that
// reads the element) and stores three 16-byte pieces, [part][8-depth piece][row] in LDS: lanes write
// and read consecutive 16-byte pieces.  Two LDS stages and two register sets: k tile t + 3 is
// requested, and k tile t + 1 split and stored, while k tile t is multiplied (a load has two k tiles
// of time to arrive), the split's instructions dealt out between the MFMAs.
template <bool LK, bool RK, int SPLIT, bool GUARD, int TMT>
__device__ __forceinline__ void f32_tile(const F32GemmParams &p) {
  constexpr int NT = 256 * SPLIT;
  constexpr int BKT = 16 * SPLIT;          // depths per k tile
  constexpr int KC = BKT / 8;              // 8-depth pieces per row
  constexpr int WM = TMT / 64, WN = NT / 64 / WM;   // wavefronts along m and n
  constexpr int FM = 2, FN = TN / 32 / WN;
  static_assert(TN * KC == NT && TMT * KC <= NT, "at most one unit of either operand per thread");
  // (PAD: where depth is contiguous 16 lanes write 16 / KC rows of all KC pieces, which a pitch of a
  // whole 256 bytes would put into the same banks.  With it conflicts take 13 % of the cycles of 4 x 1024^3 where
  // both operands lie so, 6 % where one does.)
  constexpr int PAD = 16 / KC, PA_ = TMT + PAD, PB_ = TN + PAD;
  __shared__ __align__(16) u4v sA[2][3][KC][PA_];
  __shared__ __align__(16) u4v sB[2][3][KC][PB_];
  __shared__ __align__(16) float s_bias[TMT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  int bid, b;
  span_of_block(&bid, &b);
  const int m0 = (bid % p.tiles_m) * TMT, n0 = (bid / p.tiles_m) * TN;
  const float *A = p.lhs + (int64_t)b * p.lbs;
  const float *B = p.rhs + (int64_t)b * p.rbs;

  // Element offset of column n of an operand or of the result: columns of all batches side by side
  // where the launch is flat (p.flat: columns per batch).
  auto col_at = [&](int n, int64_t step, int64_t batch_step) -> int64_t {
    if (!p.flat) return (int64_t)n * step;
    const int img = n / p.flat;
    return img * batch_step + (int64_t)(n - img * p.flat) * step;
  };
  // this thread's unit of either operand (rows past the end repeat the last one; not stored)
  const bool has_a = TMT * KC == NT || tid < TMT * KC;
  const int am = LK ? tid / KC : tid % TMT, ac = LK ? tid % KC : tid / TMT;
  const int bn = RK ? tid / KC : tid % TN, bc = RK ? tid % KC : tid / TN;
  const float *pa = A + (int64_t)min(m0 + am, p.M - 1) * p.lrs;
  const float *pb = B + col_at(min(n0 + bn, p.N - 1), p.rcs, p.rbs);
  u4v *const da = &sA[0][0][has_a ? ac : 0][has_a ? am : 0], *const db = &sB[0][0][bc][bn];

  const int kt0 = p.kt_split * (int)blockIdx.y * TK;
  const int kend = p.kt_split ? min(kt0 + p.kt_split * TK, p.K) : p.K;
  const int nk = (kend - kt0 + BKT - 1) / BKT;
  // No load sits under a condition (the waits in front of their use then leave younger requests in
  // flight): units past the depth re-read its last eight, single elements past it the last one.
  auto load_unit = [&](auto contig, const float *at, int64_t step, int kk, float (&x)[8]) __attribute__((always_inline)) {
    kk = min(kk, kend - 8);
    if constexpr (decltype(contig)::value) {
      if constexpr (GUARD) {
        __builtin_memcpy(&x[0], at + kk, 16);
        __builtin_memcpy(&x[4], at + kk + 4, 16);
      } else {
        const f4v v0 = *(const f4v *)(at + kk), v1 = *(const f4v *)(at + kk + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[e] = v0[e]; x[4 + e] = v1[e]; }
      }
    } else {
      const float *q = at + (int64_t)kk * step;
#pragma unroll
      for (int e = 0; e < 8; ++e) { x[e] = *q; q += step; }
    }
  };
  float xa[2][8], xb[2][8];
  auto load_tile = [&](auto set, int kt) __attribute__((always_inline)) {
    constexpr int S = decltype(set)::value;
    load_unit(std::integral_constant<bool, LK>{}, pa, p.lcs, kt0 + kt * BKT + ac * 8, xa[S]);
    load_unit(std::integral_constant<bool, RK>{}, pb, p.rrs, kt0 + kt * BKT + bc * 8, xb[S]);
  };
  // depths below 8: the one k tile there is, what lies past the depth as zeros
  auto load_shallow = [&](auto contig, const float *at, int64_t step, int kk, float (&x)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = at[min(kk + e, kend - 1) * (decltype(contig)::value ? 1 : step)];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = kk + e < kend ? x[e] : 0.f;
  };
  auto clear_past_depth = [&](auto set, int kt) __attribute__((always_inline)) {
    if constexpr (GUARD) {
      constexpr int S = decltype(set)::value;
      if (kt0 + (kt + 1) * BKT <= kend) return;
      // the last k tile: units that were read early move down to their place; what lies past the depth counts as zero
      auto settle = [&](int kk, float (&x)[8]) __attribute__((always_inline)) {
        const int early = max(kk - (kend - 8), 0);
#pragma unroll
        for (int by = 4; by > 0; by >>= 1)
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = early & by ? (e + by < 8 ? x[e + by] : 0.f) : x[e];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = kk + e < kend ? x[e] : 0.f;
      };
      settle(kt0 + kt * BKT + ac * 8, xa[S]);
      settle(kt0 + kt * BKT + bc * 8, xb[S]);
    }
  };
  auto store_tile = [&](auto set, int kt, int buf, auto last) __attribute__((always_inline)) {
    constexpr int S = decltype(set)::value;
    if constexpr (decltype(last)::value) clear_past_depth(set, kt);
    u4v part[3];
    split_8(xa[S], part);
    if (has_a) {
#pragma unroll
      for (int q = 0; q < 3; ++q) da[(buf * 3 + q) * KC * PA_] = part[q];
    }
    split_8(xb[S], part);
#pragma unroll
    for (int q = 0; q < 3; ++q) db[(buf * 3 + q) * KC * PB_] = part[q];
  };

  // the running sum of hi hi; with eight wavefronts, whose registers allow it, the five smaller
  // products have one of their own, so that they do not each round the large one
  constexpr int NACC = SPLIT == 2 ? 2 : 1;
  v16f acc[NACC][FM * FN];
#pragma unroll
  for (int s = 0; s < NACC; ++s)
#pragma unroll
    for (int t = 0; t < FM * FN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[s][t][r] = 0.f;
  auto multiply = [&](auto steps, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < decltype(steps)::value; ++ks) {
      const int kc = 2 * ks + (lane >> 5);
      b8v a[FM][3], bb[FN][3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i][q] = __builtin_bit_cast(b8v, sA[buf][q][kc][wm * 64 + i * 32 + (lane & 31)]);
#pragma unroll
        for (int j = 0; j < FN; ++j) bb[j][q] = __builtin_bit_cast(b8v, sB[buf][q][kc][(wn * FN + j) * 32 + (lane & 31)]);
      }
      // smallest products first
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            v16f &c = acc[t < 5 ? NACC - 1 : 0][i * FN + j];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][PA[t]], bb[j][PB[t]], c, 0, 0, 0);
          }
    }
  };

  constexpr std::integral_constant<int, 0> set0{};
  constexpr std::integral_constant<int, 1> set1{};
  const float bias_m = p.bias_row ? p.bias_row[min(m0 + tid % TMT, p.M - 1)] : 0.f;
  // (eight wavefronts: half a k tile at the end of a depth that has one; a guarded one is filled up
  // with zeros instead)
  const int nfull = GUARD ? nk : (kend - kt0) / BKT;
  // k tile t: its fragments read, the MFMAs with the split of tile t + 1 between them, then the request
  // for tile t + 3 into the registers that the split has freed
  auto step = [&](auto set, int kt, auto last) __attribute__((always_inline)) {
    constexpr int S = decltype(set)::value;   // tile kt + 1's registers
    multiply(std::integral_constant<int, BKT / 16>{}, S ^ 1);
    if constexpr (decltype(last)::value) {   // (of the last three k tiles: there is nothing to request any more)
      if (kt + 1 < nfull) store_tile(set, kt + 1, S, last);
      __syncthreads();
      return;
    }
    store_tile(set, kt + 1, S, last);
    constexpr int MFMAS = BKT / 16 * 6 * FM * FN;
#pragma unroll
    for (int i = 0; i < MFMAS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // an MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 144 / MFMAS, 0);   // vector instructions
    }
    load_tile(set, kt + 3);
    __syncthreads();
  };
  if (GUARD && p.K < 8) {   // (one k tile.  Apart: loads under a condition would make the usual ones wait for all of theirs)
    load_shallow(std::integral_constant<bool, LK>{}, pa, p.lcs, ac * 8, xa[0]);
    load_shallow(std::integral_constant<bool, RK>{}, pb, p.rrs, bc * 8, xb[0]);
    if (tid < TMT) s_bias[tid] = bias_m;
    store_tile(set0, 0, 0, std::false_type{});
    __syncthreads();
  } else {
    load_tile(set0, 0);
    load_tile(set1, 1);
    if (tid < TMT) s_bias[tid] = bias_m;
    store_tile(set0, 0, 0, std::true_type{});
    load_tile(set0, 2);
    __syncthreads();
    int kt = 0;
    for (; kt + (GUARD ? 3 : 1) < nfull; kt += 2) {
      step(set1, kt, std::false_type{});
      step(set0, kt + 1, std::false_type{});
    }
    if constexpr (GUARD) {
      for (; kt + 1 < nfull; kt += 2) {
        step(set1, kt, std::true_type{});
        step(set0, kt + 1, std::true_type{});
      }
    }
  }
  if constexpr (GUARD) {
    if (nfull & 1) multiply(std::integral_constant<int, BKT / 16>{}, 0);
  } else {
    if (nfull & 1) step(set1, nfull - 1, std::false_type{});
    if (BKT == 32 && nfull < nk) multiply(std::integral_constant<int, 1>{}, nfull & 1);
  }

  if constexpr (NACC == 2) {
#pragma unroll
    for (int t = 0; t < FM * FN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][t][r] = acc[0][t][r] + acc[1][t][r];
  }
  // The tile by the binary32 instruction: k tiles of the operands as they are in LDS, depth by depth,
  // the next k tile requested while one is multiplied.
  auto again = [&]() __attribute__((always_inline)) {
    // (opaque, so that nothing made up for this rare pass is kept in registers through the main loop)
    int t = tid, first = 0;
    asm("" : "+v"(t), "+s"(first));
    const int am = LK ? t / KC : t % TMT, ac = LK ? t % KC : t / TMT;
    const int bn = RK ? t / KC : t % TN, bc = RK ? t % KC : t / TN;
    const bool has_a = TMT * KC == NT || t < TMT * KC;
    float *const fa = (float *)sA + ac * 8 * PA_ + am, *const fb = (float *)sB + bc * 8 * PB_ + bn;
    static_assert(sizeof(sA) >= sizeof(float) * BKT * PA_ && sizeof(sB) >= sizeof(float) * BKT * PB_, "a k tile of binary32");
#pragma unroll
    for (int t = 0; t < FM * FN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][t][r] = 0.f;
    const bool shallow = GUARD && p.K < 8;   // (one k tile)
    if (shallow) {
      load_shallow(std::integral_constant<bool, LK>{}, pa, p.lcs, ac * 8, xa[0]);
      load_shallow(std::integral_constant<bool, RK>{}, pb, p.rrs, bc * 8, xb[0]);
    } else {
      load_tile(set0, first);
    }
    for (int kt = first; kt < nk; ++kt) {
      if (!shallow) clear_past_depth(set0, kt);
      __syncthreads();   // (nobody reads the k tile before any more)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (has_a) fa[e * PA_] = xa[0][e];
        fb[e * PB_] = xb[0][e];
      }
      if (!shallow) load_tile(set0, kt + 1);
      __syncthreads();
      const int depth = min(BKT, kend - kt0 - kt * BKT);
      for (int k = lane >> 5; k < depth + (lane >> 5); k += 2) {
        float a[FM], bb[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i] = ((const float *)sA)[k * PA_ + wm * 64 + i * 32 + (lane & 31)];
#pragma unroll
        for (int j = 0; j < FN; ++j) bb[j] = ((const float *)sB)[k * PB_ + (wn * FN + j) * 32 + (lane & 31)];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[0][i * FN + j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], bb[j], acc[0][i * FN + j], 0, 0, 0);
      }
    }
  };
  float worst = 0.f;   // not finite if one of the sums is not
#pragma unroll
  for (int t = 0; t < FM * FN; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      worst = __fmaf_rn(acc[0][t][r], 0.f, worst);
      acc[0][t][r] = acc[0][t][r] * SUM_SCALE;
    }
  if (__syncthreads_or(worst != 0.f)) again();

  const bool raw = p.kt_split != 0;   // a part of the k range: bias and activation come with the sum of the parts
  float *O = (raw ? p.part + (int64_t)blockIdx.y * p.part_stride : p.out) + (int64_t)b * p.obs;
  const bool whole = m0 + TMT <= p.M && n0 + TN <= p.N;
  // (Requested and back before the first store.  As a load under a condition between the stores it made each of them wait for
  // the one before it, in whichever copies below the compiler left it: 901 drawn calls of 200 to 600 tiles 0.87 of the time
  // in the geometric mean, 26 x 25 x 21 -> 557 at batch 8 11.0 -> 8.9 us, 4 x 1024^3 51.8 -> 50.9.)
  float bias_n[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = min(n0 + (wn * FN + j) * 32 + (lane & 31), p.N - 1);   // (of the long row of all batches, whose bias repeats)
    bias_n[j] = !raw && p.bias_col ? p.bias_col[p.flat ? col % p.flat : col] : 0.f;
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(bias_n[j]));
  // (one copy per activation, none of its tests per element)
  auto store = [&](auto act_tag) __attribute__((always_inline)) {
    constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + (wn * FN + j) * 32 + (lane & 31);
      float *oc = O + col_at(min(n, p.N - 1), p.ocs, p.obs);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int ml = wm * 64 + i * 32 + 4 * (lane >> 5);
        float *orow = oc + (int64_t)(m0 + ml) * p.ors;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f4v bias = *(const f4v *)&s_bias[ml + 8 * q];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = acc[0][i * FN + j][4 * q + e];
            if (!raw) {
              if (p.bias_row) v = v + bias[e];
              if (p.bias_col) v = v + bias_n[j];
            }
            v = apply_act(v, ACT, p.limit);
            if (whole || (m0 + ml + 8 * q + e < p.M && n < p.N)) *orow = v;
            orow += p.ors;
          }
          orow += 4 * p.ors;
        }
      }
    }
  };
  if (!raw && p.act == MACE_HIP_ACT_RELU) store(std::integral_constant<int, MACE_HIP_ACT_RELU>{});
  else if (!raw && p.act == MACE_HIP_ACT_RELUX) store(std::integral_constant<int, MACE_HIP_ACT_RELUX>{});
  else store(std::integral_constant<int, MACE_HIP_ACT_NOOP>{});
}

template <bool LK, bool RK, int SPLIT, int TMT>
__global__ __launch_bounds__(256 * SPLIT, SPLIT == 1 ? 3 : 1) void f32_gemm_vec_kernel(F32GemmParams p) {
  f32_tile<LK, RK, SPLIT, false, TMT>(p);
}
template <bool LK, bool RK, int SPLIT, int TMT>
__global__ __launch_bounds__(256 * SPLIT, SPLIT == 1 ? 3 : 1) void f32_gemm_kernel(F32GemmParams p) {
  f32_tile<LK, RK, SPLIT, true, TMT>(p);
}

// ---- a left-hand matrix that stays in LDS, columns streamed past it ----------------------------------
//
// A convolution's filter against the pixels of a batch is few rows against very many columns: per 128 x 128 tile the k loop
// is short, and every tile pays for its first loads, a barrier per 16 depths and its stores, in step with the others on its
// CU.  Here a workgroup keeps the three parts of 32 MI rows, all depths, in LDS as fragments (split once), and each of its
// eight wavefronts walks blocks of 32 columns by itself: eight 4-byte loads a k step, coalesced over 32 columns, straight
// into the fragment's registers and split there, no barrier.  The loads run D k steps ahead, on into the next block, so that
// a block's stores and the next one's loads overlap.  Products and their order are f32_tile's with four wavefronts: the same
// bits.
// What bounds it: the bytes up to about 128 depths (112 x 112 x 32 -> 64 at batch 64 4.9 TB/s, what a copy reaches), beyond
// that the vector ALU and the matrix cores, which take turns within a wavefront.  In tiles and here, batch 64, us: 112 x
// 112 x 32 -> 64 73.6 and 60.3, 56 x 56 x 128 -> 128 65.6 and 49.8, 28 x 28 x 256 -> 256 55.5 and 48.1, 56 x 56 x 100 -> 200
// 95.8 and 91.7, 56 x 56 x 24 -> 144 37.6 and 33.0.  Of 1500 drawn layers that come here 766 in whole k steps take 0.85 of the
// tiles' time in the geometric mean, 149 others of up to 32 rows 0.86, 325 of more rows and up to six broken k steps 0.97, but
// 260 of more than six 1.06 (28 x 28 x 333 -> 111 36.5 and 45.8): those were chosen against tiles that loaded depth by depth
// (56 us) and whose stores waited for each other, and tests name that plan.  (128 rows, eight wavefronts a CU: level at best,
// 36 % slower at 24 -> 144; a load under the epilogue's test for a bias per column made every block wait for all of its loads
// and stores: 78 us on 56 x 56 x 128.)
template <int MI, int D, bool GUARD>
__global__ __launch_bounds__(512, 4) void f32_gemm_panel_kernel(F32GemmParams p, int groups, int blocks) {
  extern __shared__ __align__(16) u4v panel[];     // [k step][part][32 rows][lane]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r32 = lane & 31;
  const int nks = (p.K + 15) >> 4;
  float *const s_bias = (float *)(panel + (size_t)nks * 3 * MI * 64);
  // Workgroup w runs on XCD w % 8: every XCD gets a contiguous span of (span of columns, rows), so that the
  // workgroups that read the same columns share an L2.
  int wg = blockIdx.x;
  {
    const int per = (int)gridDim.x >> 3, more = (int)gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, more) + (wg >> 3);
  }
  const int group = wg / p.tiles_m, m0 = (wg - group * p.tiles_m) * (32 * MI);
  const int b0 = (int)((int64_t)blocks * group / groups), b1 = (int)((int64_t)blocks * (group + 1) / groups);
  const float *const B = p.rhs;

  // byte offset of this lane's column of a block in the operand and in the result (there its half's first row)
  auto columns_of = [&](int block, uint32_t *in, uint32_t *out) __attribute__((always_inline)) {
    const int n = min(block * 32 + r32, p.N - 1);
    int64_t at = n, to = n;
    if (p.flat) {
      const int img = n / p.flat, in_img = n - img * p.flat;
      at = img * p.rbs + in_img;
      to = img * p.obs + in_img;
    }
    *in = (uint32_t)(at * 4);
    *out = (uint32_t)((to + (int64_t)(4 * h) * p.ors) * 4);
  };
  const int64_t row_bytes = p.rrs * 4;
  const uint32_t half_off = h ? (uint32_t)(8 * row_bytes) : 0u;
  float x[D][8];
  // (no load sits under a condition: see f32_tile)
  auto load = [&](int set, int ks, uint32_t off) __attribute__((always_inline)) {
    const char *row = (const char *)B + (int64_t)(16 * ks) * row_bytes;
    if constexpr (!GUARD) off += half_off;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (GUARD) {   // depths past the last re-read it; cleared when they are split
        const int left = p.K - 1 - (16 * ks + e);
        x[set][e] = *(const float *)(row + (off + (h ? (uint32_t)max(min(8, left), 0) * (uint32_t)row_bytes : 0u)));
        row += left > 0 ? row_bytes : 0;
      } else {
        x[set][e] = *(const float *)(row + off);
        row += row_bytes;
      }
    }
  };
  int block = b0 + wave;
  uint32_t in_off, out_off;
  columns_of(min(block, blocks - 1), &in_off, &out_off);
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, min(d, nks - 1), in_off);

  // the rows' three parts, once; rows past the last repeat it, depths past the last are zeros
  for (int u = tid; u < nks * 2 * 32 * MI; u += 512) {
    const int row = u % (32 * MI), piece = u / (32 * MI);
    const float *at = p.lhs + (int64_t)min(m0 + row, p.M - 1) * p.lrs + (int64_t)(8 * piece) * p.lcs;
    float v[8];
    if (p.lcs == 1 && 8 * piece + 8 <= p.K) {
      __builtin_memcpy(&v[0], at, 16);
      __builtin_memcpy(&v[4], at + 4, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int left = p.K - 1 - 8 * piece;      // (below 0: a piece of zeros)
        v[e] = at[(int64_t)min(e, left) * p.lcs];
        v[e] = e <= left ? v[e] : 0.f;
      }
    }
    u4v part[3];
    split_8(v, part);
#pragma unroll
    for (int q = 0; q < 3; ++q)
      panel[(((piece >> 1) * 3 + q) * MI + (row >> 5)) * 64 + (piece & 1) * 32 + (row & 31)] = part[q];
  }
  if (tid < 32 * MI) s_bias[tid] = p.bias_row ? p.bias_row[min(m0 + tid, p.M - 1)] : 0.f;
  __syncthreads();

  const int padded = (nks + D - 1) / D * D;
  if (block >= b1) return;
  do {   // (loops that run once at the least: no copies of registers whose loads are on their way)
    const int next = block + 8;
    uint32_t next_in, next_out;
    columns_of(next < b1 ? next : block, &next_in, &next_out);
    v16f acc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
    int ks0 = 0;
    do {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int ks = ks0 + d;
        u4v b[3];
        if constexpr (GUARD) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (16 * ks + 8 * h + e >= p.K) x[d][e] = 0.f;
        }
        split_8(x[d], b);
        const int ahead = ks + D;
        load(d, ahead < padded ? min(ahead, nks - 1) : min(ahead - padded, nks - 1), ahead < padded ? in_off : next_in);
        if (ks < nks) {
          const u4v *a = panel + (size_t)ks * (3 * MI * 64) + lane;
          u4v f[3][MI];
#pragma unroll
          for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int i = 0; i < MI; ++i) f[q][i] = a[(q * MI + i) * 64];
          constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};   // smallest products first
#pragma unroll
          for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int i = 0; i < MI; ++i)
              acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8v, f[PA[t]][i]),
                                                              __builtin_bit_cast(b8v, b[PB[t]]), acc[i], 0, 0, 0);
        }
      }
      ks0 += D;
    } while (ks0 < padded);
    float worst = 0.f;   // not finite if one of the sums is not
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        worst = __fmaf_rn(acc[i][r], 0.f, worst);
        acc[i][r] = acc[i][r] * SUM_SCALE;
      }
    if (__builtin_amdgcn_ballot_w64(worst != 0.f) != 0) {   // (see f32_tile)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
      for (int k0 = 0; k0 < p.K; k0 += 8) {
        float v[4], a[4][MI];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int64_t k = min(k0 + 2 * u + h, p.K - 1);
          v[u] = *(const float *)((const char *)(B + k * p.rrs) + in_off);
#pragma unroll
          for (int i = 0; i < MI; ++i) a[u][i] = p.lhs[(int64_t)min(m0 + i * 32 + r32, p.M - 1) * p.lrs + k * p.lcs];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bool in = k0 + 2 * u + h < p.K;
#pragma unroll
          for (int i = 0; i < MI; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? a[u][i] : 0.f, in ? v[u] : 0.f, acc[i], 0, 0, 0);
        }
      }
    }
    const int n = block * 32 + r32;
    const bool whole = m0 + 32 * MI <= p.M && block * 32 + 32 <= p.N;
    auto store = [&](auto act_tag) __attribute__((always_inline)) {
      constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f4v bias = *(const f4v *)&s_bias[i * 32 + 8 * q + 4 * h];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int m = m0 + i * 32 + 8 * q + e;          // (and 4 h)
            float v = acc[i][4 * q + e];
            if (p.bias_row) v = v + bias[e];
            v = apply_act(v, ACT, p.limit);
            if (whole || (m + 4 * h < p.M && n < p.N)) *(float *)((char *)(p.out + (int64_t)m * p.ors) + out_off) = v;
          }
        }
    };
    if (p.act == MACE_HIP_ACT_RELU) store(std::integral_constant<int, MACE_HIP_ACT_RELU>{});
    else if (p.act == MACE_HIP_ACT_RELUX) store(std::integral_constant<int, MACE_HIP_ACT_RELUX>{});
    else store(std::integral_constant<int, MACE_HIP_ACT_NOOP>{});
    block = next;
    in_off = next_in;
    out_off = next_out;
  } while (block < b1);
}

// ---- few tiles, or shallow ones: a wavefront per slice of a 32 x 32 FN tile's depth -----------------
//
// A call of few 128 x 128 tiles is the serial chain of one of them: its k tiles one after the other, two launches where
// they are dealt to several workgroups.  Here eight wavefronts share 8 / WK tiles of 32 rows x 32 FN columns; a
// wavefront loads its slice's operands straight into fragments (lane: row or column r, eight depths of half h), no LDS,
// splits them as f32_tile does and keeps the five smaller products in a sum of their own; the WK slices' sums meet
// in LDS and each of their wavefronts adds up, in the slices' order, and stores 16 FN / WK of the tile's registers.
// What bounds it: the launch and one load's latency up to a few k steps (pointwise 34 x 35 x 112 -> 91 on one image 9.7
// -> 4.2 us, 16 x 17 x 384 -> 320 14.3 -> 5.8, 8 x 8 x 963 -> 555 at batch 4 21.9 -> 8); beyond, the address path: a
// k step of a wavefront is 4 KiB in 2 to 16 loads, most of them 16 bytes of 64 rows, about 240 cycles of a CU (three or
// two steps ahead, 16 wavefronts a tile: within 5 %).  2-norm error against binary64: the tiles' up to one k step, 0.96 - 0.55 of it from 17
// to 200 depths, 0.6 - 0.9 beyond.
template <bool LK, bool RK, int FN, int WK>
__global__ __launch_bounds__(64 * (WK > 8 ? WK : 8), FN == 1 ? 4 : 2) void f32_gemm_slices_kernel(F32GemmParams p) {
  constexpr int NW = WK > 8 ? WK : 8, WT = NW / WK;   // wavefronts, tiles of a workgroup
  constexpr int REGS = 16 * FN, AHEAD = FN == 1 ? 3 : 2;   // k steps of operands on their way
  __shared__ float s_part[NW][REGS][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % WK, wt = wave / WK, h = lane >> 5, r32 = lane & 31;
  int bid, b;
  span_of_block(&bid, &b);
  const int tiles_n = (p.N + 32 * FN - 1) / (32 * FN), total = p.tiles_m * tiles_n;
  const int tile = bid * WT + wt;          // (past the last: computed again and not stored)
  const int tl = min(tile, total - 1), m0 = (tl % p.tiles_m) * 32, n0 = (tl / p.tiles_m) * (32 * FN);
  const float *A = p.lhs + (int64_t)b * p.lbs;
  const float *B = p.rhs + (int64_t)b * p.rbs;
  auto col_at = [&](int n, int64_t step, int64_t batch_step) -> int64_t {
    if (!p.flat) return (int64_t)n * step;
    const int img = n / p.flat;
    return img * batch_step + (int64_t)(n - img * p.flat) * step;
  };
  const float *pa = A + (int64_t)min(m0 + r32, p.M - 1) * p.lrs + (int64_t)(8 * h) * p.lcs;
  const float *pb[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
    pb[j] = B + col_at(min(n0 + 32 * j + r32, p.N - 1), p.rcs, p.rbs) + (int64_t)(8 * h) * p.rrs;
  const int nk = (p.K + 15) >> 4, k0 = nk * wk / WK, k1 = nk * (wk + 1) / WK, whole = p.K >> 4;

  // eight depths of a row: in two 16-byte loads (at any address) where they lie side by side
  auto load_unit = [&](auto contig, const float *at, int64_t step, int kt, float (&x)[8]) __attribute__((always_inline)) {
    if (kt < whole) {
      if constexpr (decltype(contig)::value) {
        __builtin_memcpy(&x[0], at + 16 * kt, 16);
        __builtin_memcpy(&x[4], at + 16 * kt + 4, 16);
      } else {
        const float *q = at + (int64_t)(16 * kt) * step;
#pragma unroll
        for (int e = 0; e < 8; ++e) { x[e] = *q; q += step; }
      }
    } else {   // the depth ends inside: what lies past it counts as zero
      const int left = p.K - 16 * kt - 8 * h;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] = at[(int64_t)(16 * kt + min(e, left - 1)) * step];
        x[e] = e < left ? x[e] : 0.f;
      }
    }
  };
  float xa[AHEAD][8], xb[AHEAD][FN][8];
  auto load = [&](int set, int kt) __attribute__((always_inline)) {   // (the set is a constant once unrolled)
    load_unit(std::integral_constant<bool, LK>{}, pa, p.lcs, kt, xa[set]);
#pragma unroll
    for (int j = 0; j < FN; ++j) load_unit(std::integral_constant<bool, RK>{}, pb[j], p.rrs, kt, xb[set][j]);
  };
  v16f acc[2][FN];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[s][j][r] = 0.f;
  auto multiply = [&](int set) __attribute__((always_inline)) {
    u4v a[3], bb[FN][3];
    split_8(xa[set], a);
#pragma unroll
    for (int j = 0; j < FN; ++j) split_8(xb[set][j], bb[j]);
    constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};   // smallest products first
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        v16f &c = acc[t < 5 ? 1 : 0][j];
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8v, a[PA[t]]), __builtin_bit_cast(b8v, bb[j][PB[t]]), c, 0, 0, 0);
      }
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u)
    if (k0 + u < k1) load(u, k0 + u);
  for (int kt = k0; kt < k1; kt += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (kt + u < k1) {
        multiply(u);
        if (kt + u + AHEAD < k1) load(u, kt + u + AHEAD);
      }
    }
  }
  // The slices' sums in their order: this wavefront's registers of the tile, REGS / WK of them.  What each addition
  // of the large sums rounds off is kept and joins the small ones (Knuth's two-sum), so that slices round no more often
  // than one accumulator does: the 2-norm error against binary64 was 25 % above the tiles' at two slices without.
  constexpr int MINE = REGS / WK;
  float v[MINE], off[MINE];
  auto gather = [&](const v16f (&sums)[FN], auto take) __attribute__((always_inline)) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) s_part[wave][j * 16 + r][lane] = sums[j][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MINE; ++i)
#pragma unroll
      for (int w = 0; w < WK; ++w) take(i, w, s_part[wt * WK + w][wk * MINE + i][lane]);
  };
  auto large = [&](int i, int w, float x) __attribute__((always_inline)) {
    if (w == 0) {
      v[i] = x;
      off[i] = 0.f;
    } else {
      const float s = v[i] + x, y = s - v[i];
      off[i] = off[i] + ((v[i] - (s - y)) + (x - y));
      v[i] = s;
    }
  };
  gather(acc[0], large);
  float small[MINE];
  gather(acc[1], [&](int i, int w, float x) __attribute__((always_inline)) { small[i] = w ? small[i] + x : x; });
  float worst = 0.f;   // not finite if one of the sums is not
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    v[i] = v[i] + (small[i] + off[i]);
    worst = __fmaf_rn(v[i], 0.f, worst);
    v[i] = v[i] * SUM_SCALE;
  }
  if (__syncthreads_or(worst != 0.f)) {   // (see f32_tile)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][j][r] = 0.f;
    for (int k = 16 * k0; k < min(16 * k1, p.K); k += 2) {
      const int at = k + h - 8 * h;        // (pa and pb begin at depth 8 h)
      const bool in = k + h < p.K;
      const float a = in ? pa[(int64_t)at * p.lcs] : 0.f;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const float x = in ? pb[j][(int64_t)at * p.rrs] : 0.f;
        acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, x, acc[0][j], 0, 0, 0);
      }
    }
    gather(acc[0], large);
#pragma unroll
    for (int i = 0; i < MINE; ++i) v[i] = v[i] * 0.f == 0.f ? v[i] + off[i] : v[i];
  }
  if (tile >= total) return;
  float *O = p.out + (int64_t)b * p.obs;
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    const int reg = wk * MINE + i, j = reg >> 4, r = reg & 15;   // (scalar)
    const int m = m0 + 8 * (r >> 2) + 4 * h + (r & 3), n = n0 + 32 * j + r32;
    if (m < p.M && n < p.N) {
      float x = v[i];
      if (p.bias_row) x = x + p.bias_row[m];
      if (p.bias_col) x = x + p.bias_col[p.flat ? n % p.flat : n];
      O[(int64_t)m * p.ors + col_at(n, p.ocs, p.obs)] = apply_act(x, p.act, p.limit);
    }
  }
}

// Depths of at most two: 0 (the reference's loop leaves sum = 0), and 1 and 2 by binary32 multiply-adds,
// because the tile kernels' products are not rounded to nearest (see there).  Bound by the stores: four
// neighbouring outputs per thread, so that divisions and loads are shared.  Against the tile kernels:
// 4096 x 1 x 4096 28.0 -> 16.6 us (column-major result 46.8 -> 16.6), two depths 28.1 -> 17.2.
template <typename Index>
__global__ __launch_bounds__(256) void f32_fill_kernel(F32GemmParams p, Index total) {
  // outputs in memory order: `in` runs fastest (columns of a row-major result, rows of a column-major one)
  const bool along_n = p.ocs == 1;
  const Index inner = (Index)(along_n ? p.N : p.M), outer = (Index)(along_n ? p.M : p.N);
  const float *const x = along_n ? p.rhs : p.lhs, *const y = along_n ? p.lhs : p.rhs;
  const int64_t xs = along_n ? p.rcs : p.lrs, ys = along_n ? p.lrs : p.rcs;
  const int64_t xk = along_n ? p.rrs : p.lcs, yk = along_n ? p.lcs : p.rrs;
  const int64_t xb = along_n ? p.rbs : p.lbs, yb = along_n ? p.lbs : p.rbs;
  const float *const bias_in = along_n ? p.bias_col : p.bias_row, *const bias_out = along_n ? p.bias_row : p.bias_col;
  const Index units = (total + 3) / 4;
  for (Index u = (Index)blockIdx.x * 256 + threadIdx.x; u < units; u += (Index)gridDim.x * 256) {
    const Index i = u * 4, line = i / inner;
    Index in = i - line * inner, b = line / outer, out = line - b * outer;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (in + 4 <= inner) {   // four of one line: one factor of each product is the same, the others lie side by side
      const float *const px = x + (int64_t)b * xb + (int64_t)in * xs, *const py = y + (int64_t)b * yb + (int64_t)out * ys;
      if (p.K > 0) {
        float f[2][4] = {};
        if (xs == 1) {
          __builtin_memcpy(f[0], px, 16);
          if (p.K > 1) __builtin_memcpy(f[1], px + xk, 16);
        } else {               // (two depths side by side)
          float pair[8];
          __builtin_memcpy(pair, px, 32);
#pragma unroll
          for (int e = 0; e < 4; ++e) { f[0][e] = pair[2 * e]; f[1][e] = pair[2 * e + 1]; }
        }
        const float y0 = py[0], y1 = p.K > 1 ? py[yk] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = __fmaf_rn(f[0][e], y0, v[e]);
          if (p.K > 1) v[e] = __fmaf_rn(f[1][e], y1, v[e]);
        }
      }
      const float bo = bias_out ? bias_out[out] : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {   // (a call has one bias or none)
        if (bias_in) v[e] = v[e] + bias_in[in + e];
        if (bias_out) v[e] = v[e] + bo;
        v[e] = apply_act(v[e], p.act, p.limit);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (i + e >= total) break;
        const float *const px = x + (int64_t)b * xb + (int64_t)in * xs, *const py = y + (int64_t)b * yb + (int64_t)out * ys;
        if (p.K > 0) v[e] = __fmaf_rn(px[0], py[0], v[e]);
        if (p.K > 1) v[e] = __fmaf_rn(px[xk], py[yk], v[e]);
        if (bias_in) v[e] = v[e] + bias_in[in];
        if (bias_out) v[e] = v[e] + bias_out[out];
        v[e] = apply_act(v[e], p.act, p.limit);
        if (++in == inner) {
          in = 0;
          if (++out == outer) { out = 0; ++b; }
        }
      }
    }
    if (i + 4 <= total) {
      __builtin_memcpy(p.out + i, v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (i + e < total) p.out[i + e] = v[e];
    }
  }
}

// The sum of a k split's parts, in the order of the parts, with the bias and the activation of the
// call: element i of batch b lies at b obs + i in every part and in the result (dense M x N).
__global__ __launch_bounds__(256) void f32_ksplit_reduce_kernel(F32GemmParams p, int parts, int64_t total) {
  const int64_t mn = (int64_t)p.M * p.N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    float v = p.part[i];
    for (int s = 1; s < parts; ++s) v = v + p.part[(int64_t)s * total + i];
    const int64_t j = i % mn;
    const int m = p.ocs == 1 ? (int)(j / p.N) : (int)(j % p.M);
    const int n = p.ocs == 1 ? (int)(j % p.N) : (int)(j / p.M);
    if (p.bias_row) v = v + p.bias_row[m];
    if (p.bias_col) v = v + p.bias_col[n];
    p.out[i] = apply_act(v, p.act, p.limit);
  }
}

// images of in_h x in_w copied into zero-filled images of ph x pw at (top, left)
__global__ __launch_bounds__(256) void f32_pad_nchw_kernel(const float *src, float *dst,
                                                           int64_t total, int in_h, int in_w, int ph,
                                                           int pw, int top, int left) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t img = i / ((int64_t)ph * pw);
    const int rem = (int)(i - img * ph * pw);
    const int y = rem / pw - top, x = rem % pw - left;
    dst[i] = ((unsigned)y < (unsigned)in_h && (unsigned)x < (unsigned)in_w)
                 ? src[(img * in_h + y) * in_w + x] : 0.f;
  }
}

struct F32GemvParams {
  const float *lhs, *rhs, *bias;
  float *out;
  int64_t lbs, rbs;
  int H, W;
  int act;        // applied to the finished sum as it is stored (FullyConnected's Activation)
  float limit;
};

// R rows against NB vectors: a row's 16-byte pieces (at any multiple of 4 bytes: a width need not be whole pieces) are
// dealt to `slices` wavefronts in turns, U pieces of every row in flight in a lane, each in a sum of its own; the lanes'
// sums are added pairwise, half of the values in half of the lanes at every step, and the slices' sums in LDS.
//
// Bound by reading the weights once where rows are many (16384 x 8192 81 us, 6.6 TB/s), by the chain of a wavefront's
// loads where they are few, and by the vectors' loads where those are many (NB per piece of weights, from L1 and L2),
// which four rows share.  Before (one wavefront a row, odd widths a float at a time, four vectors a pass) and now, us:
// 291 x 12869 18.4 and 6.2, 128 x 11904 9.5 and 4.1; 6 x 13230 x 294 19.5 and 7.7, 12 x 10232 x 503 50 and 10, 13 x 8975
// x 5888 225 and 74, 7 x 1825 x 7168 34 and 15.  (The block's wavefronts come
// as an argument: read from the launch, small calls took 0.15 - 0.3 us more.)
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));
template <int NB, int R, int U>
__device__ __forceinline__ void gemv_rows(const F32GemvParams &p, int batch, int slice_bits, int groups) {
  constexpr int N = R * NB <= 1 ? 1 : (R * NB <= 2 ? 2 : (R * NB <= 4 ? 4 : (R * NB <= 8 ? 8 : (R * NB <= 16 ? 16 :
                    (R * NB <= 32 ? 32 : 64)))));      // (values reduced together: a power of two)
  __shared__ float s_part[8][N];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int slices = 1 << slice_bits, slice = wave & (slices - 1);
  const int group = wave >> slice_bits;
  const int h0 = ((int)blockIdx.x * groups + group) * R;     // (rows past the last: read as the last, not stored)
  const int b0 = (int)blockIdx.y * NB;
  constexpr int PER = 64 / N;                                // lanes that end with the same value
  const int value = lane / PER, vi = value / NB, vj = value % NB;
  const float bias = p.bias ? p.bias[min(h0 + vi, p.H - 1)] : 0.f;
  const float *l = p.lhs + (int64_t)b0 * p.lbs;
  const float *lr[R], *r[NB];
#pragma unroll
  for (int i = 0; i < R; ++i) lr[i] = l + (int64_t)min(h0 + i, p.H - 1) * p.W;
#pragma unroll
  for (int j = 0; j < NB; ++j) r[j] = p.rhs + (int64_t)min(b0 + j, batch - 1) * p.rbs;
  const int pieces = p.W >> 2, turn = 64 * slices;
  float s[U][R * NB];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int i = 0; i < R * NB; ++i) s[u][i] = 0.f;
  auto dot4 = [](const f32x4 &a, const f32x4 &x) {
    return __builtin_fmaf(a.x, x.x, a.y * x.y) + __builtin_fmaf(a.z, x.z, a.w * x.w);
  };
  int c = 64 * slice;      // this wavefront's first piece of the turn
  for (; c + turn * (U - 1) + 64 <= pieces; c += turn * U) {
    f32x4 a[U][R];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < R; ++i)
        a[u][i] = __builtin_nontemporal_load((const f32x4_any *)(lr[i] + 4 * (int64_t)(c + turn * u + lane)));
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const f32x4 x = *(const f32x4_any *)(r[j] + 4 * (int64_t)(c + turn * u + lane));
#pragma unroll
        for (int i = 0; i < R; ++i) s[u][i * NB + j] += dot4(a[u][i], x);
      }
  }
  if (c < pieces) {        // the last turns: pieces past the row's end are read as its last one and count as zeros
    f32x4 a[U][R];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c + turn * u < pieces) {
#pragma unroll
        for (int i = 0; i < R; ++i)
          a[u][i] = __builtin_nontemporal_load((const f32x4_any *)(lr[i] + 4 * (int64_t)min(c + turn * u + lane, pieces - 1)));
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c + turn * u < pieces) {
        const bool in = c + turn * u + lane < pieces;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const f32x4 x = *(const f32x4_any *)(r[j] + 4 * (int64_t)min(c + turn * u + lane, pieces - 1));
#pragma unroll
          for (int i = 0; i < R; ++i) {
            const float d = dot4(a[u][i], x);
            s[u][i * NB + j] += in ? d : 0.f;
          }
        }
      }
  }
  if (slice == slices - 1 && lane < (p.W & 3)) {             // what is left of a width that is not whole pieces
    const int w = 4 * pieces + lane;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < R; ++i) s[U - 1][i * NB + j] += lr[i][w] * r[j][w];
  }
  float v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (i >= R * NB) v[i] = 0.f;
    else if constexpr (U == 4) v[i] = (s[0][i] + s[1][i]) + (s[2][i] + s[3][i]);
    else if constexpr (U == 2) v[i] = s[0][i] + s[1][i];
    else v[i] = s[0][i];
  }
  // (after the first log2(N) steps a lane holds the one value that its upper bits number)
#pragma unroll
  for (int step = 0; step < 6; ++step) {
    const int off = 32 >> step, left = N >> (step + 1);
    const bool upper = lane & off;
    if (left == 0) v[0] += __shfl_xor(v[0], off, 64);
#pragma unroll
    for (int i = 0; i < left; ++i) {
      const float mine = upper ? v[i + left] : v[i], theirs = upper ? v[i] : v[i + left];
      v[i] = mine + __shfl_xor(theirs, off, 64);
    }
  }
  float t = v[0];
  if (slices > 1) {
    if (lane % PER == 0) s_part[wave][value] = t;
    __syncthreads();
    if (slice != 0) return;
    t = s_part[wave][value] + s_part[wave + 1][value];
    if (slices == 4) t += s_part[wave + 2][value] + s_part[wave + 3][value];
    if (slices == 8) {
      t += s_part[wave + 2][value] + s_part[wave + 3][value];
      t += (s_part[wave + 4][value] + s_part[wave + 5][value]) + (s_part[wave + 6][value] + s_part[wave + 7][value]);
    }
  }
  if (lane % PER != 0 || value >= R * NB || h0 + vi >= p.H || b0 + vj >= batch) return;
  p.out[(int64_t)(b0 + vj) * p.H + h0 + vi] = apply_act(bias + t, p.act, p.limit);
}

template <int NB>
__global__ __launch_bounds__(512, 4) void f32_gemv_kernel(F32GemvParams p, int batch, int slice_bits, int groups) {
  gemv_rows<NB, 1, 4>(p, batch, slice_bits, groups);
}
template <int NB>
__global__ __launch_bounds__(512, 4) void f32_gemv_rows_kernel(F32GemvParams p, int batch, int slice_bits, int groups) {
  gemv_rows<NB, 4, 1>(p, batch, slice_bits, groups);
}

// One row a wavefront, float by float: coalesced 4-byte loads, which the address path takes at full width wherever a row
// begins, where 16-byte loads at odd addresses cost it twice.  For widths that are not whole pieces and rows for about
// a round of wavefronts (3323 x 2343 8.5 us by pieces, 6.9 here, 3712 x 1305 6.0 and 5.3, 8 x 119 x 1838 4.8 and 3.6).
// (A last turn of masked loads instead of the loads left over: 10 - 20 % slower.)
__global__ __launch_bounds__(256) void f32_gemv_floats_kernel(F32GemvParams p) {
  const int lane = threadIdx.x & 63;
  const int h = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (h >= p.H) return;
  const int b = blockIdx.y;
  const float *l = p.lhs + (int64_t)b * p.lbs + (int64_t)h * p.W;
  const float *r = p.rhs + (int64_t)b * p.rbs;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // (short chains: rounding as in the kernel by pieces)
  int w = lane;
  auto turn = [&](int at) __attribute__((always_inline)) {   // four loads of each operand in flight
    float a[4], x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) { a[u] = l[w + 64 * u]; x[u] = r[w + 64 * u]; }
#pragma unroll
    for (int u = 0; u < 4; ++u) s[at + u] = __builtin_fmaf(a[u], x[u], s[at + u]);
    w += 256;
  };
  while (w + 192 < p.W) {
    turn(0);
    if (w + 192 < p.W) turn(4);
  }
  for (; w < p.W; w += 64) s[7] = __builtin_fmaf(l[w], r[w], s[7]);
  float t = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
  if (lane == 0) p.out[(int64_t)b * p.H + h] = apply_act((p.bias ? p.bias[h] : 0.f) + t, p.act, p.limit);
}

}  // namespace

// Tiles of 32 x 32 fn, their depth in wk slices.
struct F32SlicesForm { int fn, wk; };
constexpr F32SlicesForm kF32Slices[mhv::F32_SLICES_FORMS] = {{1, 8}, {1, 4}, {2, 8}};
// Which form of the slices kernel a call takes whose 128 x 128 tiles are at most one per CU; -1: none, the tiles are
// faster.  Both times are estimated, in us: a k step takes a wavefront 0.75 (1.5 with two blocks), a CU's
// wavefronts together 0.14 - 0.17 each and 0.25 - 0.6 a tile beside them; a 128 x 128 tile 0.63 per 16 depths behind
// 5.3, in parts 12 and the parts' traffic, 3 more at depths in other than whole steps.  Measured, tiles then slices: 16 x 17 x
// 384 -> 320 pointwise 12.5 and 6.3, 34 x 35 x 112 -> 91 9.8 and 4.5, 1904 x 39 x 298 8.3 and 6.4, 653 x 1266 x 35 15.6 and 11.0,
// 512^3 15.7 and 7.3; against the rule 20 x 21 x 20 -> 160 at batch 20 8.0 and 9.5, 70 x 3456 x 679 21 and 30, 4 x 1024^3 50 and
// 107.  Of 1000 drawn calls in whole k steps 841 go here, in 0.60 of the tiles' time in the geometric mean, five of them more
// than 3 % slower; of 1000 others 886, 0.61 and twenty (196 x 2913 x 273 against transposed weights 35 us, in tiles 20, 883 x
// 2132 x 512 32 and 26); without the 3 us six, but 49 left to the tiles that are faster here, now one.
static int f32_slices_form(const mace_hip_ctx *ctx, int64_t batch, int64_t rows, int64_t cols, int64_t depth,
                           int64_t total, bool whole) {
  const double cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const int64_t nk = (depth + 15) / 16, tiles = batch * ((rows + 31) / 32) * ((cols + 31) / 32);
  const int parts = mh_f32_ksplit(ctx, batch, rows, cols, depth);
  const double old = parts > 1 ? (whole ? 12 : 15) + 0.63 * ((nk + parts - 1) / parts) + 8.0 * parts * total / 4e6
                               : (whole ? 5.3 : 8.3) + 0.63 * nk;
  const int form = tiles <= 400 ? 0 : 1, wk = kF32Slices[form].wk;
  // (a second tile on a few CUs counts from long depths on: 62 x 2112 x 4552, 286 tiles, 34.7 us, 24.9 by 128 x 128 tiles;
  // not where the parts of those could not be had)
  const bool held = parts <= 1 || mh_arena_can_hold(ctx, sizeof(float) * (size_t)parts * total + 256);
  const double share = nk > 64 && form == 0 && tiles > cus && held ? std::max(tiles / cus, 0.8 * ceil(tiles / cus)) : tiles / cus;
  const double one = 4.2 + std::max(0.75 * ((nk + wk - 1) / wk), share * (whole ? 0.25 + 0.14 * nk : 0.6 + 0.17 * nk));
  if (nk >= 24 && tiles > cus) {
    const int64_t wide = batch * ((rows + 31) / 32) * ((cols + 63) / 64);
    // (one workgroup a CU: rounds of them, with their starts and ends)
    const double rounds = ceil(wide / cus), two = 1.2 + rounds * (3 + 1.5 * ((nk + 7) / 8));
    if (two < one) return two < 0.95 * old ? 2 : -1;
  }
  // (more, in two slices: within 5 % of the tiles; at one or two k steps a third workgroup on a CU is 20 - 30 % more:
  // pointwise 12 x 13 x 17 -> 384 at batch 20, 1176 tiles, 11.4 us, 7.7 by tiles)
  return tiles <= (nk <= 2 ? 4 * cus : 1200) && one < 0.9 * old ? form : -1;
}

int mh_f32_gemm(mace_hip_ctx *ctx, const float *lhs, const float *rhs, int64_t batch,
                int64_t rows, int64_t cols, int64_t depth, int lhs_major, int rhs_major,
                int out_major, int lhs_batched, int rhs_batched, float *out,
                const F32Epilogue &ep) {
  MH_CHECK(ctx, batch >= 0 && rows >= 0 && cols >= 0 && depth >= 0, "negative dimension");
  MH_CHECK(ctx, (lhs_major | 1) == 1 && (rhs_major | 1) == 1 && (out_major | 1) == 1,
           "matrix major must be RowMajor (0) or ColMajor (1)");
  MH_CHECK(ctx, rows < (1ll << 31) && cols < (1ll << 31) && depth < (1ll << 31) && batch < 65536,
           "dimension too large");
  if (batch == 0 || rows == 0 || cols == 0) return MACE_HIP_SUCCESS;
  MH_CHECK(ctx, out && (depth == 0 || (lhs && rhs)), "null operand");
  F32GemmParams p{};
  p.lhs = lhs; p.rhs = rhs; p.out = out;
  // mace/ops/common/matrix.h:48-80: stride = cols (RowMajor) or rows (ColMajor)
  p.lrs = lhs_major == MACE_HIP_ROW_MAJOR ? depth : 1;
  p.lcs = lhs_major == MACE_HIP_ROW_MAJOR ? 1 : rows;
  p.rrs = rhs_major == MACE_HIP_ROW_MAJOR ? cols : 1;
  p.rcs = rhs_major == MACE_HIP_ROW_MAJOR ? 1 : depth;
  p.ors = out_major == MACE_HIP_ROW_MAJOR ? cols : 1;
  p.ocs = out_major == MACE_HIP_ROW_MAJOR ? 1 : rows;
  p.lbs = lhs_batched ? rows * depth : 0;
  p.rbs = rhs_batched ? depth * cols : 0;
  p.obs = rows * cols;
  p.M = (int)rows; p.N = (int)cols; p.K = (int)depth;
  p.bias_row = ep.bias_row; p.bias_col = ep.bias_col; p.act = ep.act; p.limit = ep.limit;
  const int64_t total = batch * rows * cols;
  if (depth <= 2) {
    dim3 grid((unsigned)std::min<int64_t>((total + 1023) / 1024, 65535));
    mh_plan_main(ctx, MACE_HIP_KF_F32_GEMM_FILL, 0, grid, dim3(256), 0);
    // (32-bit divisions where they do; the last stride past the end must not wrap either)
    if (total < (1ll << 31)) MH_KLAUNCH(ctx, f32_fill_kernel<uint32_t>, grid, dim3(256), 0, ctx->stream, p, (uint32_t)total);
    else MH_KLAUNCH(ctx, f32_fill_kernel<int64_t>, grid, dim3(256), 0, ctx->stream, p, total);
    MH_LAUNCH_CHECK(ctx);
    return MACE_HIP_SUCCESS;
  }
  // A shared left-hand matrix (a convolution's filter) against a batch: the columns of all batches
  // are one long row, so that tiles do not end at an image (7 x 7 pixels fill 49 of a tile's 128
  // columns: 1024 -> 1024 channels at batch 64 190 -> 55 us, the split above included).
  const int64_t images = batch;
  if (batch > 1 && !lhs_batched && rhs_batched && out_major == MACE_HIP_ROW_MAJOR &&
      rhs_major == MACE_HIP_ROW_MAJOR && batch * cols < (1ll << 31)) {
    p.flat = (int)cols;
    p.N = (int)(batch * cols);
    batch = 1;
  }
  // Up to 192 rows that leave the last 128-row tile at most half full: tiles of 64 rows (while there is at
  // least one for every CU; below, the eight-wavefront form with 128 rows).  A 64-row tile takes 1.2 to 1.4 times
  // half the time of a 128-row one, so a quarter of the work has to be padding: 64 x 256 x 70000 42.0 -> 29.7 us,
  // 192 x 512 x 40000 74.3 -> 66.5, but 320 x 256 x 20000 33.9 -> 38.0, 576 x 512 x 12000 54.8 -> 64.7.
  const int64_t cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const bool half = p.M <= TM + TM / 2 && (p.M - 1) % TM < TM / 2 &&
                    ((p.M + 63) / 64) * ((p.N + TN - 1) / TN) * batch > cus;
  const int tm = half ? TM / 2 : TM;
  p.tiles_m = (p.M + tm - 1) / tm;
  const int64_t tiles = (int64_t)p.tiles_m * ((p.N + TN - 1) / TN);
  MH_CHECK(ctx, tiles < (1ll << 31), "too many tiles");
  dim3 grid((unsigned)tiles, 1, (unsigned)batch), block(256), block2(512);
  const bool split = tiles * batch <= cus;   // at most one tile per CU
  const bool lk = lhs_major == MACE_HIP_ROW_MAJOR;   // depth contiguous
  const bool rk = rhs_major == MACE_HIP_COL_MAJOR;
  // Depths in whole k tiles, and rows along depth in aligned 16-byte pieces: no load is checked.  (An
  // operand that runs along m / n is read by 4-byte loads, so it may have any length and address.)
  const bool whole = depth % TK == 0 && (!lk || (uintptr_t)lhs % 16 == 0) && (!rk || (uintptr_t)rhs % 16 == 0);
  // The plan files calls whose operands are aligned 16-byte pieces in either direction under a family of
  // their own, which they had when those loads were 16 bytes wide as well.
  const bool vec = depth % TK == 0 && (lk || rows % 4 == 0) && (rk || cols % 4 == 0) &&
                   rows >= 4 && cols >= 4 && ((uintptr_t)lhs % 16 == 0) &&
                   ((uintptr_t)rhs % 16 == 0);
  if (split && !(ctx->kernel_mask & MH_MASK_NO_F32_SLICES)) {
    const int slices = f32_slices_form(ctx, batch, p.M, p.N, depth, total, whole);
    if (slices >= 0) {
      const F32SlicesForm &f = kF32Slices[slices];
      p.tiles_m = (p.M + 31) / 32;
      const int64_t small = (int64_t)p.tiles_m * ((p.N + 32 * f.fn - 1) / (32 * f.fn)), wt = 8 / f.wk;
      grid.x = (unsigned)((small + wt - 1) / wt);
      mh_plan_main(ctx, MACE_HIP_KF_F32_GEMM_SLICES, mhv::f32_slices(slices, lk, rk), grid, block2, 0);
      MH_PROF_BEGIN(ctx);
#define MH_F32_SLICES(L, R)                                                                                         \
  do {                                                                                                              \
    if (slices == 0) MH_KLAUNCH(ctx, (f32_gemm_slices_kernel<L, R, 1, 8>), grid, block2, 0, ctx->stream, p);        \
    else if (slices == 1) MH_KLAUNCH(ctx, (f32_gemm_slices_kernel<L, R, 1, 4>), grid, block2, 0, ctx->stream, p);   \
    else MH_KLAUNCH(ctx, (f32_gemm_slices_kernel<L, R, 2, 8>), grid, block2, 0, ctx->stream, p);                    \
  } while (0)
      if (lk && rk) MH_F32_SLICES(true, true);
      else if (lk) MH_F32_SLICES(true, false);
      else if (rk) MH_F32_SLICES(false, true);
      else MH_F32_SLICES(false, false);
#undef MH_F32_SLICES
      MH_PROF_END(ctx);
      MH_LAUNCH_CHECK(ctx);
      return MACE_HIP_SUCCESS;
    }
  }
  // More tiles than CUs, a right-hand matrix along its columns and rows whose parts fit in LDS: columns streamed past the
  // rows.  Tiles of 32 rows where a wavefront would have fewer than about two blocks of 32 rows x 32 columns (80 x 82 x 32
  // -> 70 at batch 6 8.0 us, in tiles of 64 11.1) and where those leave an eighth less padding; else of 64.  (Of one k step
  // the 128-row tiles are up to 10 % faster: 54 x 53 x 16 -> 129 at 10 9.0 us and 9.9.)
  if (!split && batch == 1 && !rk && out_major == MACE_HIP_ROW_MAJOR && !p.bias_col && depth > 16 && p.N >= 8ll * p.M &&
      images * depth * cols < (1ll << 30) && total < (1ll << 30) && !(ctx->kernel_mask & MH_MASK_NO_F32_PANEL)) {
    const int nks = (int)((depth + 15) / 16), blocks = (p.N + 31) / 32;
    auto lds_of = [&](int mi) { return (size_t)nks * 3 * mi * 1024 + 128 * mi; };
    const int64_t small = (p.M + 31) / 32, large = (p.M + 63) / 64;
    const bool narrow = p.M <= 32 || blocks * small <= 24 * cus || 23 * small <= 40 * large;
    // (Depths from 417 on leave room for 32 rows of more than that at a time: where loads are not checked only against
    // 128-row tiles that are a fifth padding.  14 x 14 x 512 -> 512 at batch 64 50 us in tiles, 55 - 66 here; 13440 columns,
    // 512 -> 258 46 and 33.)
    const bool deep = lds_of(2) > (size_t)ctx->lds_bytes;
    const int mi = narrow || deep ? 1 : 2;
    const size_t lds = lds_of(mi);
    // Depths that are not whole k steps cost every step here (loads are checked and cleared), the tiles only the last one: not
    // two tiles of 32 rows, each of which reads the columns, against one of 64 rows.  1 x 1 layers, tiles and here: 840 x 137 ->
    // 40 at batch 48 14.7 us and 20.8, 1640 x 201 -> 64 at 54 25.7 and 38.9.
    const bool twice = !whole && mi == 1 && p.M > 32 && p.M <= 64;
    // Nor deep ones, one workgroup a CU (384 x 829 x 31464 122 us and 216, 704 x 671 x 19600 128 and 212, 224 x 457 -> 576 at
    // batch 48 47 and 72), but for little more than a round of tiles a fifth of which is padding (148 x 418 x 12096 29.5 and
    // 24.1).  (Depths of 417 to 432, one step more than leaves room for 64 rows, come here as they did, though slower too: 111 x
    // 420 x 50176 43.5 us in tiles and 62.  A test names that plan.)
    const bool slow = !whole && deep && p.M > 32 && nks > 27 &&
                      !(6ll * p.M <= 5ll * tm * ((p.M + tm - 1) / tm) && 5 * tiles <= 6 * cus);
    if (lds <= (size_t)ctx->lds_bytes && !twice && !slow && (!deep || p.M <= 32 || !whole || 4 * TM * ((p.M + TM - 1) / TM) >= 5ll * p.M)) {
      p.tiles_m = (int)(mi == 1 ? small : large);
      // (k steps of loads on their way; a block's end is padded to a multiple of them)
      const int ahead = nks % 4 == 0 || nks >= 7 ? 4 : 2;
      auto launch = [&](auto kernel) -> int {
        MH_HIP(ctx, mh_allow_big_lds(ctx, (const void *)kernel, lds));
        const int64_t fit = cus * mh_blocks_per_cu(ctx, (const void *)kernel, 512, lds);
        const int groups = (int)std::max<int64_t>(1, std::min<int64_t>((blocks + 7) / 8, fit / p.tiles_m));
        grid.x = (unsigned)(groups * p.tiles_m);
        mh_plan_main(ctx, MACE_HIP_KF_F32_GEMM_PANEL, mhv::f32_panel(mi, ahead, !whole), grid, block2, (int)lds);
        MH_PROF_BEGIN(ctx);
        MH_KLAUNCH(ctx, kernel, grid, block2, lds, ctx->stream, p, groups, blocks);
        MH_PROF_END(ctx);
        MH_LAUNCH_CHECK(ctx);
        return MACE_HIP_SUCCESS;
      };
#define MH_F32_PANEL(MI, D) return whole ? launch(f32_gemm_panel_kernel<MI, D, false>) : launch(f32_gemm_panel_kernel<MI, D, true>)
      if (mi == 1 && ahead == 2) MH_F32_PANEL(1, 2);
      if (mi == 1) MH_F32_PANEL(1, 4);
      if (ahead == 2) MH_F32_PANEL(2, 2);
      MH_F32_PANEL(2, 4);
#undef MH_F32_PANEL
    }
  }
  // Few tiles and a long depth: the k tiles are dealt to several workgroups per tile, whose parts a
  // second launch adds up in a fixed order (see mh_f32_ksplit).
  ArenaScope scope(ctx);
  auto bytes_of = [&](int n) { return sizeof(float) * (size_t)n * total + 256; };
  int parts = mh_f32_ksplit(ctx, batch, rows, p.N, depth);
  // The long row has fewer tiles than the images have one by one, so it is split where they are not.
  // That needs scratch; where none can be had (in a capture, or beside other slices of the arena) the
  // images' own tiles decide, so that no call is refused for joining them.
  if (parts > 1 && p.flat && !mh_arena_can_hold(ctx, bytes_of(parts)))
    parts = mh_f32_ksplit(ctx, images, rows, cols, depth);
  if (parts > 1) {
    const size_t bytes = bytes_of(parts);
    // (scratch that does not fit while other slices of the arena are in use: no split)
    if (mh_arena_can_hold(ctx, bytes) || ctx->arena_used == 0) {
      MH_RETURN_IF_ERROR(mh_arena_reserve(ctx, bytes));
      p.part = (float *)mh_arena_take(ctx, bytes);
      if (!p.part) return mh_fail(ctx, MACE_HIP_RUNTIME_ERROR, "arena slice unavailable");
      const int64_t nk = (depth + TK - 1) / TK;
      p.kt_split = (int)((nk + parts - 1) / parts);
      p.part_stride = total;
      grid.y = (unsigned)((nk + p.kt_split - 1) / p.kt_split);
      mh_plan_aux(ctx, MACE_HIP_AUX_F32_KSPLIT);
    }
  }
  const int form = split ? mhv::F32_SPLIT : (half ? mhv::F32_64 : mhv::F32_128);
  if (vec) mh_plan_main(ctx, MACE_HIP_KF_F32_GEMM_VEC, mhv::f32_gemm_vec(form, lk, rk), grid,
                        split ? block2 : block, 0);
  else mh_plan_main(ctx, MACE_HIP_KF_F32_GEMM_GENERAL, mhv::f32_gemm_general(!whole, form, lk, rk), grid,
                    split ? block2 : block, 0);
  MH_PROF_BEGIN(ctx);
#define MH_F32(KERNEL, ...) MH_KLAUNCH(ctx, (KERNEL<__VA_ARGS__>), grid, split ? block2 : block, 0, ctx->stream, p)
#define MH_F32_LR(KERNEL, ...)                                                                  \
  do {                                                                                          \
    if (lk && rk) MH_F32(KERNEL, true, true, __VA_ARGS__);                                      \
    else if (lk) MH_F32(KERNEL, true, false, __VA_ARGS__);                                      \
    else if (rk) MH_F32(KERNEL, false, true, __VA_ARGS__);                                      \
    else MH_F32(KERNEL, false, false, __VA_ARGS__);                                             \
  } while (0)
  if (whole && split) MH_F32_LR(f32_gemm_vec_kernel, 2, 128);
  else if (whole && half) MH_F32_LR(f32_gemm_vec_kernel, 1, 64);
  else if (whole) MH_F32_LR(f32_gemm_vec_kernel, 1, 128);
  else if (split) MH_F32_LR(f32_gemm_kernel, 2, 128);
  else if (half) MH_F32_LR(f32_gemm_kernel, 1, 64);
  else MH_F32_LR(f32_gemm_kernel, 1, 128);
#undef MH_F32_LR
#undef MH_F32
  MH_PROF_END(ctx);
  if (p.kt_split) {
    p.N = (int)cols;   // (the parts and the result hold batch after batch, whatever the tiles were)
    const int64_t blocks = (total + 255) / 256;
    MH_KLAUNCH(ctx, f32_ksplit_reduce_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
               ctx->stream, p, (int)grid.y, total);
  }
  MH_LAUNCH_CHECK(ctx);
  return MACE_HIP_SUCCESS;
}

extern "C" {

int mace_hip_gemm_f32(mace_hip_ctx *ctx, const float *lhs, const float *rhs, int64_t batch,
                      int64_t rows, int64_t cols, int64_t depth, int lhs_major,
                      int rhs_major, int out_major, int lhs_batched, int rhs_batched,
                      float *out) {
  if (!ctx) return MACE_HIP_INVALID_ARGS;
  PlanScope plan_scope(ctx);
  F32Epilogue ep{nullptr, nullptr, MACE_HIP_ACT_NOOP, 0.f};
  return mh_f32_gemm(ctx, lhs, rhs, batch, rows, cols, depth, lhs_major, rhs_major, out_major,
                     lhs_batched, rhs_batched, out, ep);
}

int mace_hip_matmul_f32(mace_hip_ctx *ctx, const float *lhs, const float *rhs, const float *bias,
                        int64_t batch, int64_t lhs_rows, int64_t lhs_cols, int64_t rhs_rows,
                        int64_t rhs_cols, int transpose_lhs, int transpose_rhs, int lhs_batched,
                        int rhs_batched, float *out) {
  if (!ctx) return MACE_HIP_INVALID_ARGS;
  PlanScope plan_scope(ctx);
  // mace/ops/ref/gemm.cc:122-131, then mace/ops/matmul.cc:195-211: c[i * cols + w] += bias[w],
  // i.e. one binary32 addition to the finished sum, done here as the sum is stored
  const int64_t rows = transpose_lhs ? lhs_cols : lhs_rows;
  const int64_t depth = transpose_lhs ? lhs_rows : lhs_cols;
  const int64_t cols = transpose_rhs ? rhs_rows : rhs_cols;
  const int64_t depth2 = transpose_rhs ? rhs_cols : rhs_rows;
  MH_CHECK(ctx, depth == depth2,
           "Matrices that multiply have inconsistent depth dim: %lld vs. %lld",
           (long long)depth, (long long)depth2);
  F32Epilogue ep{nullptr, bias, MACE_HIP_ACT_NOOP, 0.f};
  return mh_f32_gemm(ctx, lhs, rhs, batch, rows, cols, depth,
                     transpose_lhs ? MACE_HIP_COL_MAJOR : MACE_HIP_ROW_MAJOR,
                     transpose_rhs ? MACE_HIP_COL_MAJOR : MACE_HIP_ROW_MAJOR, MACE_HIP_ROW_MAJOR,
                     lhs_batched, rhs_batched, out, ep);
}

int mace_hip_gemm_f32_transpose(mace_hip_ctx *ctx, const float *lhs, const float *rhs,
                                int64_t batch, int64_t lhs_rows, int64_t lhs_cols,
                                int64_t rhs_rows, int64_t rhs_cols, int transpose_lhs,
                                int transpose_rhs, int transpose_out, int lhs_batched,
                                int rhs_batched, float *out) {
  if (!ctx) return MACE_HIP_INVALID_ARGS;
  PlanScope plan_scope(ctx);
  // mace/ops/ref/gemm.cc:122-131
  const int64_t rows = transpose_lhs ? lhs_cols : lhs_rows;
  const int64_t depth = transpose_lhs ? lhs_rows : lhs_cols;
  const int64_t cols = transpose_rhs ? rhs_rows : rhs_cols;
  const int64_t depth2 = transpose_rhs ? rhs_cols : rhs_rows;
  MH_CHECK(ctx, depth == depth2,
           "Matrices that multiply have inconsistent depth dim: %lld vs. %lld",
           (long long)depth, (long long)depth2);
  return mace_hip_gemm_f32(ctx, lhs, rhs, batch, rows, cols, depth,
                           transpose_lhs ? MACE_HIP_COL_MAJOR : MACE_HIP_ROW_MAJOR,
                           transpose_rhs ? MACE_HIP_COL_MAJOR : MACE_HIP_ROW_MAJOR,
                           transpose_out ? MACE_HIP_COL_MAJOR : MACE_HIP_ROW_MAJOR,
                           lhs_batched, rhs_batched, out);
}

int mace_hip_gemv_f32(mace_hip_ctx *ctx, const float *lhs, const float *rhs,
                      const float *bias, int64_t batch, int64_t height, int64_t width,
                      int lhs_batched, int rhs_batched, float *out) {
  return mace_hip_gemv_f32_act(ctx, lhs, rhs, bias, batch, height, width, lhs_batched, rhs_batched,
                               MACE_HIP_ACT_NOOP, 0.f, out);
}

int mace_hip_gemv_f32_act(mace_hip_ctx *ctx, const float *lhs, const float *rhs,
                          const float *bias, int64_t batch, int64_t height, int64_t width,
                          int lhs_batched, int rhs_batched, int activation, float max_limit,
                          float *out) {
  if (!ctx) return MACE_HIP_INVALID_ARGS;
  PlanScope plan_scope(ctx);
  if (activation < MACE_HIP_ACT_NOOP || activation > MACE_HIP_ACT_RELUX)
    return mh_fail(ctx, MACE_HIP_UNSUPPORTED, "activation %d is not applied by this library", activation);
  MH_CHECK(ctx, batch >= 0 && height >= 0 && width >= 0, "negative dimension");
  MH_CHECK(ctx, height < (1ll << 31) && width < (1ll << 31) && batch <= 65535,
           "dimension too large");
  if (batch == 0 || height == 0) return MACE_HIP_SUCCESS;
  MH_CHECK(ctx, out && (width == 0 || (lhs && rhs)), "null operand");
  F32GemvParams p{lhs, rhs, bias, out, lhs_batched ? height * width : 0,
                  rhs_batched ? width : 0, (int)height, (int)width, activation, max_limit};
  // Weights shared by a batch: up to 16 vectors a pass with four rows a wavefront, four with one; more passes (which
  // find the weights in a cache) where the rows alone are too few wavefronts for the latency of their loads.  Four rows
  // share the vectors' loads from 512 rows on, fewer vectors than four from 2048 on; of one vector, short rows only
  // (14528 x 191 6.6 and 5.1 us, 9152 x 704 7.7 and 7.0; 10240 x 1600 12.1 and 12.9).  Measured, one pass and more: 16 x
  // 2048 x 2048 12.1 and 10.1, 11 x 1146 x 512 9.6 and 4.9; one row a wavefront and four: 8 x 1408 x 9728 25 and 20, 3 x
  // 1454 x 9904 16.1 and 20.1.
  static const int kVectors[mhv::F32_GEMV_VECTORS] = {1, 2, 3, 4, 6, 8, 12, 16};
  const int64_t vectors = !lhs_batched && rhs_batched ? batch : 1;
  const bool four = vectors >= 4 ? height >= 512 : (vectors > 1 ? height >= 2048 : height >= 8192 && width < 1024);
  // Slices of a row: a lane adds at most a quarter of its pieces of a row in one sum; more slices where rows are few.
  // The vectors of a pass: kVectors[form].
  int64_t passes = (vectors + (four ? 15 : 3)) / (four ? 16 : 4);
  int slices = 1;
  if (four) {
    while (slices < 4 && width > 256 * slices) slices *= 2;
    auto wavefronts = [&](int n) { return (height + 3) / 4 * n * passes; };
    while (wavefronts(width >= 4096 ? 8 : slices) < 2800 && (vectors + passes - 1) / passes > 4) ++passes;
    if (width >= 4096 && wavefronts(slices) < 2800) slices = 8;
  } else {
    while (slices < 8 && height * passes * slices < 1800 && width > 1024 * slices) slices *= 2;
  }
  int form = 0;
  // (three vectors as four with four rows: 3 x 4000 x 1000 6.0 us, 11.2 with loads that wait for one another)
  while (kVectors[form] < (vectors + passes - 1) / passes || (four && kVectors[form] == 3)) ++form;
  const int nb = kVectors[form];
  // Widths that are not whole aligned pieces: float by float where that is faster.  (Drawn widths, time against the kernels
  // by pieces: one vector a pass, 2400 to 6600 rows of 512 to 4096 floats, 44 MB at most, no more than two loads left over
  // behind turns of 256: 52 calls, 0.81 - 1.01, median 0.96; with more left over 0.84 - 1.16, with more rows to 1.25, with
  // 65 to 71 MB 1.09 - 1.11.  Four vectors a pass, too few rows for four a wavefront: 28 calls, 0.76 - 1.01, median 0.89;
  // three vectors 0.79 - 1.23.)
  const bool pieces = width % 4 == 0 && (uintptr_t)lhs % 16 == 0 && (uintptr_t)rhs % 16 == 0;
  const int64_t all_rows = batch * height;
  if (!pieces && width >= 512 &&
      (vectors == 1 ? all_rows >= 2400 && all_rows < 6600 && width < 4096 && all_rows * width < 11000000 && width % 256 <= 128
                    : !four && nb == 4 && all_rows < 6144 && width < 2700)) {
    const dim3 grid((unsigned)((height + 3) / 4), (unsigned)batch), block(256);
    mh_plan_main(ctx, MACE_HIP_KF_F32_GEMV_GENERAL, mhv::F32_GEMV_FLOATS, grid, block, 0);
    MH_PROF_BEGIN(ctx);
    MH_KLAUNCH(ctx, f32_gemv_floats_kernel, grid, block, 0, ctx->stream, p);
    MH_PROF_END(ctx);
    MH_LAUNCH_CHECK(ctx);
    return MACE_HIP_SUCCESS;
  }
  const int waves = slices > 4 ? slices : 4, bits = mhv::log2i(slices), groups = waves >> bits, rows = groups * (four ? 4 : 1);
  const dim3 grid((unsigned)((height + rows - 1) / rows), (unsigned)((batch + nb - 1) / nb)), block(64 * waves);
  if (four) mh_plan_main(ctx, MACE_HIP_KF_F32_GEMV_VEC, form - (nb > 3), grid, block, 0);
  else mh_plan_main(ctx, MACE_HIP_KF_F32_GEMV_GENERAL, form, grid, block, 0);
  MH_PROF_BEGIN(ctx);
  auto launch = [&](auto vectors) {
    constexpr int NB = decltype(vectors)::value;
    if constexpr (NB <= 4) {
      if (!four) {
        MH_KLAUNCH(ctx, f32_gemv_kernel<NB>, grid, block, 0, ctx->stream, p, (int)batch, bits, groups);
        return;
      }
    }
    if constexpr (NB != 3)
      MH_KLAUNCH(ctx, f32_gemv_rows_kernel<NB>, grid, block, 0, ctx->stream, p, (int)batch, bits, groups);
  };
  switch (nb) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    case 4: launch(std::integral_constant<int, 4>{}); break;
    case 6: launch(std::integral_constant<int, 6>{}); break;
    case 8: launch(std::integral_constant<int, 8>{}); break;
    case 12: launch(std::integral_constant<int, 12>{}); break;
    default: launch(std::integral_constant<int, 16>{}); break;
  }
  MH_PROF_END(ctx);
  MH_LAUNCH_CHECK(ctx);
  return MACE_HIP_SUCCESS;
}

int mace_hip_conv1x1_f32_nchw(mace_hip_ctx *ctx, const float *input, const float *filter,
                              const float *bias, int64_t n, int64_t cin, int64_t hw,
                              int64_t cout, int activation, float max_limit, float *out) {
  if (!ctx) return MACE_HIP_INVALID_ARGS;
  PlanScope plan_scope(ctx);
  MH_CHECK(ctx, activation >= MACE_HIP_ACT_NOOP && activation <= MACE_HIP_ACT_RELUX,
           "unsupported activation %d", activation);
  // mace/ops/arm/base/conv_2d_1x1.cc:66-68: Gemm(filter, input, batch, cout, cin, cin, hw,
  // no transposes, lhs_batched = false, rhs_batched = true); bias and activation follow
  // (mace/ops/conv_2d.cc:171-173) and are fused into the store here.
  F32Epilogue ep{bias, nullptr, activation, max_limit};
  return mh_f32_gemm(ctx, filter, input, n, cout, hw, cin, MACE_HIP_ROW_MAJOR,
                     MACE_HIP_ROW_MAJOR, MACE_HIP_ROW_MAJOR, 0, 1, out, ep);
}

int mace_hip_conv2d_f32_nchw(mace_hip_ctx *ctx, const float *input, const float *filter,
                             const float *bias, int64_t n, int64_t cin, int64_t in_h, int64_t in_w,
                             int64_t cout, int64_t k_h, int64_t k_w, int stride_h, int stride_w,
                             int dilation_h, int dilation_w, int pad_h, int pad_w, int activation,
                             float max_limit, float *out) {
  if (!ctx) return MACE_HIP_INVALID_ARGS;
  PlanScope plan_scope(ctx);
  MH_CHECK(ctx, n >= 0 && cin >= 0 && in_h >= 0 && in_w >= 0 && cout >= 0, "negative dimension");
  MH_CHECK(ctx, k_h >= 1 && k_w >= 1 && stride_h >= 1 && stride_w >= 1 && dilation_h >= 1 &&
                    dilation_w >= 1 && pad_h >= 0 && pad_w >= 0,
           "filter / stride / dilation < 1 or negative padding");
  // the case mace/ops/conv_2d.cc:101-105 hands to Conv2dK1x1; everything else stays with the
  // caller's general convolution
  if (k_h != 1 || k_w != 1 || stride_h != 1 || stride_w != 1 || dilation_h != 1 || dilation_w != 1)
    return mh_fail(ctx, MACE_HIP_UNSUPPORTED,
                   "only 1x1 filters at stride 1, dilation 1 run on the GPU");
  if (pad_h == 0 && pad_w == 0)
    return mace_hip_conv1x1_f32_nchw(ctx, input, filter, bias, n, cin, in_h * in_w, cout,
                                     activation, max_limit, out);
  // mace/ops/arm/base/conv_2d_1x1.cc:37-60: the input is copied into a zero-padded tensor
  // (pad / 2 rows above and columns to the left, the rest below and to the right) and the Gemm
  // runs over the padded image
  const int64_t ph = in_h + pad_h, pw = in_w + pad_w;
  const int64_t total = n * cin * ph * pw;
  MH_CHECK(ctx, total < (1ll << 40), "dimension too large");
  if (total == 0 || cout == 0) return MACE_HIP_SUCCESS;
  MH_CHECK(ctx, input && out, "null operand");
  // (the scratch of a split that only the joined images take is asked for, not insisted on)
  const size_t scratch = sizeof(float) * (size_t)total + 4096;
  const size_t joined = scratch + mh_f32_ksplit_bytes(ctx, n, cout, ph * pw, cin);
  MH_RETURN_IF_ERROR(mh_arena_reserve(ctx, mh_arena_can_hold(ctx, joined) ? joined
                                           : scratch + mh_f32_ksplit_bytes(ctx, n, cout, ph * pw, cin, false)));
  ArenaScope scope(ctx);
  float *padded = (float *)mh_arena_take(ctx, sizeof(float) * (size_t)total);
  if (!padded) return mh_fail(ctx, MACE_HIP_RUNTIME_ERROR, "arena slice unavailable");
  const int64_t blocks = (total + 255) / 256;
  mh_plan_aux(ctx, MACE_HIP_AUX_F32_PAD);
  MH_KLAUNCH(ctx, f32_pad_nchw_kernel, dim3((unsigned)(blocks < 65535 ? blocks : 65535)),
                     dim3(256), 0, ctx->stream, input, padded, total, (int)in_h, (int)in_w,
                     (int)ph, (int)pw, pad_h >> 1, pad_w >> 1);
  MH_LAUNCH_CHECK(ctx);
  return mace_hip_conv1x1_f32_nchw(ctx, padded, filter, bias, n, cin, ph * pw, cout, activation,
                                   max_limit, out);
}

}  // extern "C"
