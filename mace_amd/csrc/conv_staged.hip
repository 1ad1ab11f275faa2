// Quantized Conv2D (NHWC) in one launch: a workgroup stages the rows that its pixels reach in LDS, shifted, and walks the
// filter in pieces of 16 channels.  (mace/ops/conv_2d.cc:201-412: Im2col and the gemmlowp product it feeds; here no
// patch matrix and no copy of the input exists.)
#include <math.h>

#include <algorithm>

#include "common.h"
#include "q8_requant.h"
#include "q8_transfer.h"

namespace {

struct ConvStagedParams {
  const uint8_t *in, *filter;
  const int32_t *bias;
  uint8_t *out;
  int in_h, in_w, cin, cout, k_h, k_w, sh, sw, pt, pl, out_h, out_w;
  int depth, columns;
  int vh, cw;                   // rows of one image with its padding, pixels of such a row
  int pieces, taps, stages;     // 16-channel pieces of a pixel; taps of the filter; stages of 16 pieces of a patch
  int step_taps, step_pieces;   // 16 pieces on
  int tiles_x, tile_px;         // channel tiles; pixels of a tile
  int lanes_log2;               // staging: lanes per pixel
  int pitch;                    // bytes of a piece's plane
  int at_filter, at_offs, at_psum, at_cx;   // LDS, behind the planes
  uint32_t m_cw, m_vh, m_ow, m_oh, m_tiles, m_pieces, m_kw;   // magics of divisors (0: one)
  uint32_t in_last, filter_last;   // offset of the operands' last 16 bytes
  int32_t xcoef, ycoef, yadd;
  uint32_t zpf4;                // the input zero point ^ 0x80 in all four bytes
  RequantFixed rq;
  RequantMad rqm;               // of rq, where by_mad
  bool by_mad;
};

__host__ __device__ inline uint32_t staged_magic(uint32_t d) { return d <= 1 ? 0u : (uint32_t)((1ull << 32) / d + 1); }
// n / d for n d < 2^32
__device__ __forceinline__ int staged_div(int n, uint32_t magic) {
  return magic == 0 ? n : (int)__umulhi((uint32_t)n, magic);
}
// The low n of four bytes (n below 0: none, above 4: all)
__device__ __forceinline__ int staged_mask(int n) {
  return n >= 4 ? -1 : (n <= 0 ? 0 : (int)((1u << (8 * n)) - 1u));
}

// the sum over 2^lg neighbouring lanes (lg at most 4), in all of them
__device__ __forceinline__ int staged_lanes_sum(int v, int lg) {
  if (lg > 0) v += __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);    // lanes 1 0 3 2 of four
  if (lg > 1) v += __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);    // 2 3 0 1
  if (lg > 2) v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);   // eight lanes mirrored
  if (lg > 3) v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);   // sixteen
  return v;
}

constexpr int STAGED_KS = 8;       // k steps of a stage: 16 pieces of 16 bytes
constexpr int STAGED_PIXELS = 8;   // pixels that a thread stages at a time
__host__ __device__ constexpr int staged_filter_pitch(int fx) { return fx * 512 + 16; }

// A workgroup owns 32 FX output channels x up to 512 output pixels in the images' order.  It stages the rows that the
// pixels reach once, shifted to int8, as planes of 16 channels (padding as the zero point, any channel count: pieces are
// read unaligned and masked), with the sum of every pixel's bytes, and walks the filter in stages of 16 pieces (tap, 16
// channels): the pieces of the next stage are in registers while one is multiplied from LDS, masked, shifted and summed by
// channel on their way.  Where a piece of a patch lies behind its first pixel comes from a table in LDS, so that any filter
// and channel count take the same loop.  A pitch of planes and pieces that is 16 more than a multiple of 128 keeps the
// writes free of bank conflicts; reads are 512 bytes in a row.
//
// What bounds it: the serial chain of a tile, start (2.5 us), staging (2 - 2.5, a load's latency and its arithmetic), the
// k steps (28 x 28 x 128 -> 128 at batch 64: 3.8 at the MFMAs' rate, about 6 as they are) and the epilogue (1.5 - 2).
// Against the kernels that took these calls before, 3 x 3, us: 28 x 28 x 128 -> 128 at batch 64 18.9 (planes, two launches)
// -> 14.4, 14 x 14 x 256 -> 256 18.7 -> 15.5, 7 x 7 x 512 -> 512 24.0 -> 18.5, 56 x 56 x 64 -> 64 20.7 (resident-tile kernel,
// two launches) -> 18.4, 34 x 36 x 108 -> 28 18.8 -> 11.4, 28 x 28 x 128 -> 128 at 16 11.5 -> 9.0.  Of 3500 drawn layers 1300 go
// here, 1.17 times faster in the geometric mean.
//
// FX: blocks of 32 channels; WK: wavefronts that share a block of 64 pixels, each with its part of a stage's k steps;
// WHOLE: channels in whole pieces; TWO: of two blocks, 128 registers, so that two workgroups share a CU (56 x 56 x 64 -> 64
// 18.4 us, one a CU and fragments requested a k step ahead 22.0)
template <int FX, int WK, bool WHOLE, bool TWO>
__global__ __launch_bounds__(512, FX == 1 || TWO ? 4 : 2) void q8_conv_staged_kernel(ConvStagedParams p) {
  constexpr int KS = STAGED_KS, MINE = KS / WK, FP = staged_filter_pitch(FX);
  extern __shared__ __align__(16) uint8_t lds[];
  const v4i flip = {(int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080};
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r32 = lane & 31;
  const int wk = wave % WK, wy = wave / WK;
  // Workgroup w runs on XCD w % 8: every XCD gets a contiguous span of (pixel tile, channel tile).
  int wg = blockIdx.x;
  {
    const int per = (int)gridDim.x >> 3, more = (int)gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, more) + (wg >> 3);
  }
  const int group = staged_div(wg, p.m_tiles), x0 = (wg - group * p.tiles_x) * (32 * FX);
  const int px0 = group * p.tile_px, px1 = min(px0 + p.tile_px, p.columns) - 1;

  // ---- the filter: thread (channel of 32, piece of 16), the next stage's pieces on their way in registers
  const int fj = tid & 15, fc = tid >> 4;
  uint32_t frow[FX];
#pragma unroll
  for (int u = 0; u < FX; ++u) frow[u] = (uint32_t)min(x0 + u * 32 + fc, p.cout - 1) * (uint32_t)p.depth;
  int tap = staged_div(fj, p.m_pieces), pc = fj - tap * p.pieces;
  v4i fv[FX];
  int fleft, csum[FX];
  uint32_t fearly[FX];
#pragma unroll
  for (int u = 0; u < FX; ++u) csum[u] = 0;
  auto load_filter = [&]() __attribute__((always_inline)) {
    const bool in = tap < p.taps;                    // (past the patch: its first piece, counted as zeros)
    const uint32_t off = in ? (uint32_t)(tap * p.cin + pc * 16) : 0u;
    fleft = in ? p.cin - 16 * pc : 0;
#pragma unroll
    for (int u = 0; u < FX; ++u) {
      const uint32_t o = frow[u] + off;
      if constexpr (WHOLE) {
        __builtin_memcpy(&fv[u], p.filter + o, 16);
      } else {
        const uint32_t at = min(o, p.filter_last);
        fearly[u] = o - at;
        __builtin_memcpy(&fv[u], p.filter + at, 16);
      }
    }
    tap += p.step_taps;
    pc += p.step_pieces;
    if (pc >= p.pieces) { pc -= p.pieces; ++tap; }
  };
  auto store_filter = [&](int buf) __attribute__((always_inline)) {
    uint8_t *to = lds + p.at_filter + buf * (2 * KS * FP) + fj * FP + fc * 16;
#pragma unroll
    for (int u = 0; u < FX; ++u) {
      v4i w = fv[u];
      if constexpr (!WHOLE) {
        if (fearly[u] != 0) w = moved_down(w, fearly[u]);
      }
      w = w ^ flip;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (WHOLE) w[e] = fleft > 0 ? w[e] : 0;
        else w[e] &= staged_mask(fleft - 4 * e);
        csum[u] = __builtin_amdgcn_sdot4(w[e], 0x01010101, csum[u], false);
      }
      *(v4i *)(to + u * 512) = w;
    }
  };
  load_filter();
  int32_t fbias[FX];
#pragma unroll
  for (int u = 0; u < FX; ++u) fbias[u] = p.bias ? p.bias[min(x0 + u * 32 + fc, p.cout - 1)] : 0;

  // ---- the rows that the tile's pixels reach, padding and images included, as planes of 16 channels
  const int g0 = staged_div(px0, p.m_ow), g1 = staged_div(px1, p.m_ow);       // output rows
  const int img0 = staged_div(g0, p.m_oh), img1 = staged_div(g1, p.m_oh);
  const int row0 = (g0 - img0 * p.out_h) * p.sh, first = img0 * p.vh + row0;
  const int nrows = img1 * p.vh + (g1 - img1 * p.out_h) * p.sh + p.k_h - first;
  int32_t *const psum = (int32_t *)(lds + p.at_psum);
  {
    const int lg = p.lanes_log2, g = tid & ((1 << lg) - 1), slots = 512 >> lg, pixels = nrows * p.cw;
    for (int at0 = 0; at0 < pixels; at0 += slots * STAGED_PIXELS) {
      const int at = at0 + (tid >> lg);
      uint32_t base[STAGED_PIXELS];
      bool inside[STAGED_PIXELS];
      int sum[STAGED_PIXELS];
#pragma unroll
      for (int u = 0; u < STAGED_PIXELS; ++u) {
        const int px = min(at + u * slots, pixels - 1);
        const int r = staged_div(px, p.m_cw), col = px - r * p.cw;
        const int img = staged_div(first + r, p.m_vh), ih = first + r - img * p.vh - p.pt, iw = col - p.pl;
        inside[u] = (unsigned)ih < (unsigned)p.in_h && (unsigned)iw < (unsigned)p.in_w;
        base[u] = inside[u] ? (uint32_t)(((img * p.in_h + ih) * p.in_w + iw) * p.cin) : 0u;
        sum[u] = 0;
      }
      for (int c = g; c < p.pieces; c += 1 << lg) {
        v4i v[STAGED_PIXELS];
        const uint32_t ch = (uint32_t)(16 * c);
#pragma unroll
        for (int u = 0; u < STAGED_PIXELS; ++u)
          __builtin_memcpy(&v[u], p.in + (WHOLE ? base[u] + ch : min(base[u] + ch, p.in_last)), 16);
        __builtin_amdgcn_sched_barrier(0);
        v4i ones;
#pragma unroll
        for (int e = 0; e < 4; ++e) ones[e] = WHOLE ? 0x01010101 : 0x01010101 & staged_mask(p.cin - 16 * c - 4 * e);
#pragma unroll
        for (int u = 0; u < STAGED_PIXELS; ++u) {
          if constexpr (!WHOLE) {
            if (base[u] + ch > p.in_last) v[u] = moved_down(v[u], base[u] + ch - p.in_last);
          }
          v4i w = v[u] ^ flip;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            w[e] = inside[u] ? w[e] : (int)p.zpf4;
            sum[u] = __builtin_amdgcn_sdot4(w[e], ones[e], sum[u], false);
          }
          if (at + u * slots < pixels) *(v4i *)(lds + c * p.pitch + (at + u * slots) * 16) = w;
        }
      }
#pragma unroll
      for (int u = 0; u < STAGED_PIXELS; ++u) {
        const int s = staged_lanes_sum(sum[u], lg);
        if (g == 0 && at + u * slots < pixels) psum[at + u * slots] = s;
      }
    }
  }
  // where the pieces of a patch lie behind its first pixel: [stage][half][k step]
  for (int q = tid; q < p.stages * 2 * KS; q += 512) {
    const int t = staged_div(q, p.m_pieces), c = q - t * p.pieces, kh = staged_div(t, p.m_kw);
    const int in_stage = q & (2 * KS - 1);
    ((int32_t *)(lds + p.at_offs))[(q - in_stage) + (in_stage & 1) * KS + (in_stage >> 1)] =
        t < p.taps ? (kh * p.cw + t - kh * p.k_w) * 16 + c * p.pitch : 0;
  }
  // staged position of this lane's pixels
  int pos[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int px = min(px0 + (wy * 2 + j) * 32 + r32, px1);
    const int row = staged_div(px, p.m_ow), ow = px - row * p.out_w;
    const int img = staged_div(row, p.m_oh);
    pos[j] = ((img - img0) * p.vh + (row - img * p.out_h) * p.sh - row0) * p.cw + ow * p.sw;
  }
  v16i acc[FX][2];
#pragma unroll
  for (int i = 0; i < FX; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  // ---- a stage's pieces: multiplied from one buffer while the next stage's are stored in the other
  const bool live = px0 + wy * 64 <= px1;
  store_filter(0);
  if (p.stages > 1) load_filter();
  for (int st = 0; st < p.stages; ++st) {
    const int buf = st & 1;
    __syncthreads();                 // stage st is stored, stage st - 1 read
    // (of the two wavefronts on a SIMD one stores its pieces while the other multiplies)
    auto ahead = [&]() __attribute__((always_inline)) {
      if (st + 1 < p.stages) {
        store_filter(buf ^ 1);
        if (st + 2 < p.stages) load_filter();
      }
    };
    if (wave < 4) ahead();
    if (live) {
      const int32_t *offs = (const int32_t *)(lds + p.at_offs) + (st * 2 + h) * KS + wk * MINE;
      const uint8_t *f = lds + p.at_filter + buf * (2 * KS * FP) + (wk * MINE * 2 + h) * FP + r32 * 16;
      int off[MINE];
#pragma unroll
      for (int k = 0; k < MINE; ++k) off[k] = offs[k];
      v4i xf[2][FX], yf[2][2];
      auto fetch = [&](int set, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) yf[set][j] = *(const v4i *)(lds + pos[j] * 16 + off[k]);
#pragma unroll
        for (int i = 0; i < FX; ++i) xf[set][i] = *(const v4i *)(f + k * 2 * FP + i * 512);
      };
      fetch(0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < MINE; ++k) {
        if (k + 1 < MINE) fetch((k + 1) & 1, k + 1);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < FX; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xf[k & 1][i], yf[k & 1][j], acc[i][j], 0, 0, 0);
        if constexpr (FX == 2 && TWO) {
          __builtin_amdgcn_sched_barrier(0);
        } else {
          __builtin_amdgcn_sched_group_barrier(0x100, FX + 2, 0);   // the next fragments' reads
          __builtin_amdgcn_sched_group_barrier(0x008, 2 * FX, 0);   // MFMAs
        }
      }
    }
    if (wave >= 4) ahead();
  }

  // ---- corrections
  int32_t *const cx = (int32_t *)(lds + p.at_cx);
#pragma unroll
  for (int u = 0; u < FX; ++u) {
    const int s = staged_lanes_sum(csum[u], 4);
    if (fj == 0) cx[u * 32 + fc] = (int32_t)((uint32_t)p.xcoef * (uint32_t)s + (uint32_t)fbias[u]);
  }
  uint32_t cy[2];
  int sum[2] = {0, 0};
  if (p.k_w == 3) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      for (int kh = 0; kh < p.k_h; ++kh) {
        const int32_t *row = psum + pos[j] + kh * p.cw;
        sum[j] += row[0] + row[1] + row[2];
      }
  } else {   // (eight reads at a time: one behind the other they made 5 x 5 layers an eighth slower,
             // 96 x 94 x 16 -> 20 at batch 3 10.0 us, now 8.2, 16 x 14 x 24 -> 96 10.4 and 8.6)
    for (int kh = 0; kh < p.k_h; ++kh) {
      const int32_t *const r0 = psum + pos[0] + kh * p.cw, *const r1 = psum + pos[1] + kh * p.cw;
      int kw = 0;
      for (; kw + 4 <= p.k_w; kw += 4) {
        sum[0] += (r0[kw] + r0[kw + 1]) + (r0[kw + 2] + r0[kw + 3]);
        sum[1] += (r1[kw] + r1[kw + 1]) + (r1[kw + 2] + r1[kw + 3]);
      }
      for (; kw < p.k_w; ++kw) {
        sum[0] += r0[kw];
        sum[1] += r1[kw];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) cy[j] = (uint32_t)p.ycoef * (uint32_t)sum[j] + (uint32_t)p.yadd;
  __syncthreads();                   // the corrections are there, the last stage is read
  // ---- block by block of channels: the parts of the depth are added up, pixels j by wavefront j % WK of their group
  v4i *part = (v4i *)lds + wy * (2 * WK * 4 * 64);
#pragma unroll
  for (int i = 0; i < FX; ++i) {
    if constexpr (WK > 1) {
      if (i > 0) __syncthreads();    // the block before is read
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          part[((j * WK + wk) * 4 + q) * 64 + lane] =
              v4i{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int px = px0 + (wy * 2 + j) * 32 + r32;
      uint8_t *orow = p.out + (int64_t)px * p.cout + x0;
      if (px0 + (wy * 2 + j) * 32 > px1) continue;
      if constexpr (WK > 1) {
        if (j != wk) continue;
      }
      const int xb = i * 32;
      if (x0 + xb >= p.cout) continue;
      if constexpr (WK > 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v4i sum = {0, 0, 0, 0};
#pragma unroll
          for (int k = 0; k < WK; ++k) sum += part[((j * WK + k) * 4 + q) * 64 + lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] = sum[e];
        }
      }
      // register r: channel 8 (r / 4) + 4 h + r % 4 of the block, pixel lane % 32
      int32_t v[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v4i c = *(const v4i *)(cx + xb + 4 * h + 8 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[q * 4 + e] = (int32_t)((uint32_t)acc[i][j][q * 4 + e] + (uint32_t)c[e] + cy[j]);
      }
      uint32_t packed[4] = {0, 0, 0, 0};
      if (p.by_mad) {
        requant_16_by_mad(v, p.rqm, packed);
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) packed[r / 4] |= (uint32_t)mh_requant_fixed(v[r], p.rq) << (8 * (r % 4));
      }
      const v2u s02 = __builtin_amdgcn_permlane32_swap(packed[0], packed[2], false, false);
      const v2u s13 = __builtin_amdgcn_permlane32_swap(packed[1], packed[3], false, false);
      const v4i w = {(int)s02.x, (int)s02.y, (int)s13.x, (int)s13.y};
      const int xh = xb + 16 * h;
      if (px <= px1) {
        if (x0 + xh + 16 <= p.cout) {
          __builtin_memcpy(orow + xh, &w, 16);
        } else {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (x0 + xh + e < p.cout) orow[xh + e] = (uint8_t)(((uint32_t)w[e / 4] >> (8 * (e % 4))) & 0xff);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

struct StagedShape { int64_t n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, pt, pl, out_h, out_w; };
struct StagedPlan { int fx, wk; bool two; int64_t groups, lds; };
// LDS of a tile of `tile_px` pixels; sets the parameters that depend on it
int64_t staged_layout(const StagedShape &s, int fx, int64_t tile_px, ConvStagedParams *p, int *wk) {
  const int64_t blocks = (tile_px + 63) / 64;
  *wk = blocks > 4 ? 1 : (blocks > 2 ? 2 : (blocks > 1 ? 4 : 8));
  // rows that a tile's pixels reach: they lie in at most out_rows rows of at most images + 1 images
  const int64_t out_rows = (tile_px + s.out_w - 2) / s.out_w + 1, images = (out_rows + s.out_h - 2) / s.out_h;
  const bool whole = tile_px % s.out_w == 0;                                   // (tiles that begin with a row)
  const int64_t rows_out = whole ? tile_px / s.out_w : out_rows;
  const bool per_image = tile_px % (s.out_w * s.out_h) == 0;                   // (... with an image)
  const int64_t imgs = per_image ? tile_px / (s.out_w * s.out_h) - 1
                                 : (whole && (s.out_w * s.out_h) % tile_px == 0 ? 0 : images);
  const int64_t rows = (rows_out - 1) * s.sh + s.k_h + imgs * std::max<int64_t>(0, s.k_h - s.sh);
  const int64_t pixels = rows * p->cw;
  p->pitch = (int)mh_align_up((size_t)(pixels * 16), 128) + 16;
  const int64_t at_filter = (int64_t)mh_align_up((size_t)p->pitch * p->pieces, 16);
  const int64_t at_offs = at_filter + 2 * 2 * STAGED_KS * staged_filter_pitch(fx);
  const int64_t operands = at_offs + (int64_t)p->stages * 2 * STAGED_KS * 4;
  // (the parts' sums take the place of the operands)
  const int64_t at_psum = std::max<int64_t>(operands, *wk > 1 ? 8ll * 2 * 4096 : 0);
  const int64_t at_cx = at_psum + (int64_t)mh_align_up((size_t)(pixels * 4), 16);
  p->at_filter = (int)at_filter; p->at_offs = (int)at_offs; p->at_psum = (int)at_psum; p->at_cx = (int)at_cx;
  p->tile_px = (int)tile_px;
  return pixels < (1 << 20) ? at_cx + 32 * fx * 4 : INT64_MAX;
}
// what the kernel's 32-bit offsets and magics hold
bool staged_fits(const StagedShape &s) {
  const int64_t depth = s.k_h * s.k_w * s.cin, columns = s.n * s.out_h * s.out_w;
  const int64_t vh = (s.out_h - 1) * s.sh + s.k_h, cw = (s.out_w - 1) * s.sw + s.k_w;
  const int64_t in_bytes = s.n * s.in_h * s.in_w * s.cin, filter_bytes = s.cout * depth;
  if (s.cin < 1 || depth >= (1 << 18) || vh >= (1 << 30) || cw >= (1 << 14) || s.n * vh >= (1ll << 30) || s.cout >= (1 << 20))
    return false;
  return in_bytes >= 16 && filter_bytes >= 16 && in_bytes < (1ll << 31) - 64 && filter_bytes < (1ll << 31) - 64 &&
         (s.n == 1 || (s.n * vh * vh < (1ll << 32) && s.n * s.out_h * s.out_h < (1ll << 32))) &&
         columns * s.out_w < (1ll << 32) && columns < (1 << 30);
}
// The tile of a call on `cu` CUs with `lds_bytes` of LDS each, of fx blocks of channels; groups = 0: none fits.
StagedPlan staged_plan(const StagedShape &s, int fx, int64_t cu, int64_t lds_bytes, ConvStagedParams *p) {
  StagedPlan r{};
  const int64_t vh = (s.out_h - 1) * s.sh + s.k_h, cw = (s.out_w - 1) * s.sw + s.k_w, depth = s.k_h * s.k_w * s.cin;
  const int64_t columns = s.n * s.out_h * s.out_w;
  p->in_h = (int)s.in_h; p->in_w = (int)s.in_w; p->cin = (int)s.cin; p->cout = (int)s.cout;
  p->k_h = (int)s.k_h; p->k_w = (int)s.k_w; p->sh = (int)s.sh; p->sw = (int)s.sw; p->pt = (int)s.pt; p->pl = (int)s.pl;
  p->out_h = (int)s.out_h; p->out_w = (int)s.out_w;
  p->depth = (int)depth; p->columns = (int)columns; p->vh = (int)vh; p->cw = (int)cw;
  p->pieces = (int)((s.cin + 15) / 16); p->taps = (int)(s.k_h * s.k_w);
  p->stages = (int)(((int64_t)p->taps * p->pieces + 2 * STAGED_KS - 1) / (2 * STAGED_KS));
  p->step_taps = 2 * STAGED_KS / p->pieces; p->step_pieces = 2 * STAGED_KS % p->pieces;
  p->lanes_log2 = 0;
  while (p->lanes_log2 < 4 && (1 << p->lanes_log2) < p->pieces) ++p->lanes_log2;
  r.fx = fx;
  p->tiles_x = (int)((s.cout + 32 * r.fx - 1) / (32 * r.fx));
  // One round of workgroups where its tiles fit; else rounds of two workgroups per CU, whose phases overlap, and where
  // those do not fit of one.  Tiles of whole images or rows where that costs at most an eighth.
  const int64_t image = s.out_h * s.out_w, per = std::max<int64_t>(1, cu / p->tiles_x);
  auto try_tile = [&](int64_t groups, int64_t most) {
    int64_t tile = (columns + groups - 1) / groups;
    if (tile > 512) return false;
    for (const int64_t unit : {image, s.out_w}) {
      const int64_t up = (tile + unit - 1) / unit * unit;
      if (up <= 512 && up * 8 <= tile * 9) { tile = up; break; }
    }
    r.lds = staged_layout(s, r.fx, tile, p, &r.wk);
    if (r.lds > most) return false;
    r.groups = (columns + tile - 1) / tile;
    return true;
  };
  bool found = try_tile(std::min(columns, per), lds_bytes);
  for (int64_t rounds = 1; !found && rounds <= 64; ++rounds) {
    if (rounds * 2 * per > columns) break;
    found = try_tile(rounds * 2 * per, lds_bytes / 2) && r.wk == 1;
    if (!found) r.groups = 0;
    r.two = found;
  }
  for (int64_t rounds = 2; !found && rounds <= 64 && rounds * per <= columns; ++rounds) found = try_tile(rounds * per, lds_bytes);
  if (r.groups * p->tiles_x * p->tiles_x >= (1ll << 32)) r.groups = 0;   // (m_tiles)
  // (one image: every row is its own, whatever the divisor)
  p->m_cw = staged_magic((uint32_t)cw); p->m_vh = s.n > 1 ? staged_magic((uint32_t)vh) : 1;
  p->m_ow = staged_magic((uint32_t)s.out_w); p->m_oh = s.n > 1 ? staged_magic((uint32_t)s.out_h) : 1;
  p->m_tiles = staged_magic((uint32_t)p->tiles_x); p->m_pieces = staged_magic((uint32_t)p->pieces);
  p->m_kw = staged_magic((uint32_t)s.k_w);
  p->in_last = (uint32_t)(s.n * s.in_h * s.in_w * s.cin - 16); p->filter_last = (uint32_t)(s.cout * depth - 16);
  return r;
}
// Time that the staged kernel takes, in us: its start, for every tile of a CU the staging (a load's latency and the pieces'
// arithmetic, more of it for broken pieces), a stage's hand-over, the MFMAs of two wavefronts on a SIMD, the taps' sums
// where a filter row is not three, and the epilogue, and the bytes; of tiles that share a CU the second takes a part of the
// first, of others a little more.  Within 2.5 % in the middle half of 7000 drawn layers, -9 and +7 % in nine of ten.
// width: for the choice between widths of a tile alone, fitted to both of them on 500 layers.  (The other fit saw the width
// that this one chooses, and has two rounds of narrow tiles too low: 28 x 28 x 128 -> 128 at batch 64 by 32 channels.)
double staged_us(const StagedPlan &r, const ConvStagedParams &p, int64_t cu, int64_t lds_bytes, bool width) {
  const int slots = 512 >> p.lanes_log2, more = p.cin % 16 != 0 ? 1 : 0;
  const int64_t pixels = (p.pitch - 16) / 16, rounds = (r.groups * p.tiles_x + cu - 1) / cu;
  const double steps = (double)((pixels + slots * STAGED_PIXELS - 1) / (slots * STAGED_PIXELS)) *
                       ((p.pieces + (1 << p.lanes_log2) - 1) >> p.lanes_log2);
  const double mfma = p.stages * (STAGED_KS / r.wk) * r.fx * 2 * 2 * 32 / 2400.0;
  const bool share = (r.fx == 1 || r.two) && 2 * r.lds <= lds_bytes;
  if (width) {
    const double tile = 2.4 + steps * (0.78 + 0.49 * more) + p.stages * (0.2 + 0.19 * more) + 1.94 * mfma +
                        1.56 * (r.fx - 1) + (r.wk > 1 ? 0.22 : 0.0);
    return 2.8 + tile * (1 + (rounds - 1) * (share ? 0.7 : 1.15));
  }
  const double tile = 3.45 + steps * (1.29 + 0.17 * more) + p.stages * (0.228 + 0.083 * more) + 1.48 * mfma + 1.77 * (r.fx - 1) +
                      (r.wk > 1 ? 0.19 + 0.32 * (r.fx - 1) : 0.0) + (p.k_w == 3 ? 0.0 : 0.026 * p.taps);
  return 1.9 + tile * (1 + (rounds - 1) * (share ? 0.54 : 1.17)) + 0.206e-6 * p.columns * p.cout + 0.112e-6 * p.in_last;
}
// The better of the two widths of a tile, and its time.  (A tile of 64 channels costs 1.6 us more than one of 32.)
StagedPlan staged_best(const StagedShape &s, int64_t cu, int64_t lds_bytes, ConvStagedParams *p, double *us) {
  StagedPlan best = staged_plan(s, 1, cu, lds_bytes, p);
  if (s.cout > 32) {
    ConvStagedParams p2{};
    const StagedPlan two = staged_plan(s, 2, cu, lds_bytes, &p2);
    if (two.groups && (!best.groups || staged_us(two, p2, cu, lds_bytes, true) < staged_us(best, *p, cu, lds_bytes, true))) {
      best = two;
      *p = p2;
    }
  }
  *us = best.groups ? staged_us(best, *p, cu, lds_bytes, false) : HUGE_VAL;
  return best;
}
}  // namespace

// HUGE_VAL: not a call for it.
double mh_q8_conv_staged_us(const mace_hip_ctx *ctx, int64_t n, int64_t in_h, int64_t in_w, int64_t cin, int64_t cout,
                            int64_t k_h, int64_t k_w, int stride_h, int stride_w, int pad_top, int pad_left,
                            int64_t out_h, int64_t out_w, double *of_planes) {
  *of_planes = 0.94;
  if (ctx->kernel_mask & (MH_MASK_NO_CONV_STAGED | MH_MASK_NO_CONV_SHORT)) return HUGE_VAL;
  const StagedShape s{n, in_h, in_w, cin, cout, k_h, k_w, stride_h, stride_w, pad_top, pad_left, out_h, out_w};
  if (!staged_fits(s)) return HUGE_VAL;
  ConvStagedParams p{};
  double us;
  const int64_t cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const StagedPlan plan = staged_best(s, cu, ctx->lds_bytes, &p, &us);
  // (closer for tiles of 64 channels, whose estimate runs high, more so where wavefronts share the depth, and for few
  // workgroups: 56 x 56 x 128 -> 128 at batch 16 21.4 us on planes, 17.8 staged and 20.1 by the estimate)
  if (plan.fx == 2) *of_planes = plan.wk > 1 ? 1.05 : 0.98;
  else if (2 * plan.groups * p.tiles_x < cu) *of_planes = 0.98;
  return us;
}

// *taken = false: parameters outside the kernel's, which the general path takes or reports.
int mh_q8_conv_staged(mace_hip_ctx *ctx, const uint8_t *input, const uint8_t *filter, const int32_t *bias,
                      int64_t n, int64_t in_h, int64_t in_w, int64_t cin, int64_t cout, int64_t k_h,
                      int64_t k_w, int stride_h, int stride_w, int pad_top, int pad_left, int64_t out_h,
                      int64_t out_w, float input_scale, int32_t input_zp, float filter_scale, int32_t filter_zp,
                      float bias_scale, int32_t mult, int shift, int32_t out_zp, int clamp_min, int clamp_max,
                      uint8_t *out, bool *taken) {
  *taken = false;
  const StagedShape s{n, in_h, in_w, cin, cout, k_h, k_w, stride_h, stride_w, pad_top, pad_left, out_h, out_w};
  if (!staged_fits(s) || filter_zp < 0 || filter_zp > 255) return MACE_HIP_SUCCESS;
  if (shift < 0 || shift > 31 || clamp_min < 0 || clamp_max > 255 || clamp_min > clamp_max) return MACE_HIP_SUCCESS;
  ConvStagedParams p{};
  double us;
  const StagedPlan plan = staged_best(s, ctx->cu_count > 0 ? ctx->cu_count : 256, ctx->lds_bytes, &p, &us);
  if (us == HUGE_VAL) return MACE_HIP_SUCCESS;
  if (!mh_make_requant(mult, shift, out_zp, clamp_min, clamp_max, &p.rq)) return MACE_HIP_SUCCESS;
  p.by_mad = requant_by_mad(p.rq);
  if (p.by_mad) p.rqm = requant_mad(p.rq);
  *taken = true;
  if (mh_conv_bias_rescaled(bias, input_scale, filter_scale, bias_scale))   // (the only scratch)
    MH_RETURN_IF_ERROR(mh_arena_reserve(ctx, sizeof(int32_t) * cout + 4096));
  ArenaScope scope(ctx);
  MH_RETURN_IF_ERROR(mh_conv_bias(ctx, bias, cout, input_scale, filter_scale, bias_scale, &p.bias));
  p.in = input; p.filter = filter; p.out = out;
  const uint32_t zl = (uint32_t)filter_zp - 128u, zr = (uint32_t)input_zp - 128u;
  p.xcoef = (int32_t)(0u - zr); p.ycoef = (int32_t)(0u - zl); p.yadd = (int32_t)((uint32_t)p.depth * zl * zr);
  p.zpf4 = ((uint32_t)(input_zp & 0xff) * 0x01010101u) ^ 0x80808080u;
  const size_t lds = (size_t)plan.lds;
  const bool whole = cin % 16 == 0;
  auto launch = [&](auto kernel) -> int {
    MH_HIP(ctx, mh_allow_big_lds(ctx, (const void *)kernel, lds));
    dim3 grid((unsigned)(plan.groups * p.tiles_x)), block(512);
    mh_plan_main(ctx, MACE_HIP_KF_Q8_CONV_STAGED, mhv::conv_staged(plan.fx, plan.wk, whole, plan.fx == 2 && plan.two), grid, block, (int)lds);
    MH_PROF_BEGIN(ctx);
    MH_KLAUNCH(ctx, kernel, grid, block, lds, ctx->stream, p);
    MH_PROF_END(ctx);
    MH_LAUNCH_CHECK(ctx);
    return MACE_HIP_SUCCESS;
  };
#define MH_STAGED(FX, WK, TWO) return whole ? launch(q8_conv_staged_kernel<FX, WK, true, TWO>) : launch(q8_conv_staged_kernel<FX, WK, false, TWO>)
  switch (plan.wk * 2 + (plan.fx == 2 ? 1 : 0)) {
    case 2: MH_STAGED(1, 1, false);
    case 3: if (plan.two) MH_STAGED(2, 1, true); MH_STAGED(2, 1, false);
    case 4: MH_STAGED(1, 2, false);
    case 5: MH_STAGED(2, 2, false);
    case 8: MH_STAGED(1, 4, false);
    case 9: MH_STAGED(2, 4, false);
    case 16: MH_STAGED(1, 8, false);
    default: MH_STAGED(2, 8, false);
  }
#undef MH_STAGED
}
