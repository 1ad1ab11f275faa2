// Quantized Conv2D (NHWC) for any channel count, filter, stride and padding: the input copied once into padded
// planes that the multiplying kernel stages in LDS as they lie.  (mace/ops/conv_2d.cc:201-412: Im2col and the
// gemmlowp product it feeds; here no patch matrix exists.)
#include <math.h>

#include <algorithm>

#include "common.h"
#include "q8_requant.h"
#include "q8_transfer.h"

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));

struct ConvPlaneParams {
  const uint8_t *in, *filter;
  const int32_t *bias;
  uint8_t *planes, *packed;     // written by the first launch: padded input, filter in fragment order
  int32_t *psum, *cx;           // ... sums of its pixels' bytes, corrections by channel
  int32_t *wsums;               // a registered filter's sums by channel: kept with `packed`; else null
  bool kept;                    // ... both are there from an earlier call
  uint8_t *out;
  int n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, pt, pl, out_h, out_w;
  int depth, columns, tiles_x, tiles_p, channels;   // channels: cout in whole tiles
  int vh, cw, pixels;           // rows of one image with its padding, pixels of such a row, of all
  int pieces, slabs;            // planes of a slab (one or two), slabs
  int taps, run_len, spr, steps;   // taps and pieces of a filter row, its k steps, those of a slab
  int lanes_log2, pixel_blocks; // first launch: lanes per pixel, workgroups
  int plane_bytes;
  int stage_slabs, row_bytes;   // slabs of an LDS stage, bytes of a plane's rows in it
  int buffers;                  // 2: a stage is filled while the one before is multiplied
  bool keep;                    // all slabs in one stage: the filter stays in LDS from tile to tile
  int at_rows, filter_bytes, rows_bytes;   // LDS: rows behind the filter; bytes of a stage's
  int at_sums, psum_bytes;      // LDS: sums of pixels and channels, twice
  int at_part;                  // LDS: sums of the depth's parts
  int span, span_more;          // pixel tiles of a workgroup; so many take one more
  uint32_t m_cw, m_vh, m_ow, m_oh, m_tiles, m_pieces, m_slots, m_run, m_kh;   // magics of divisors (0: one)
  uint32_t in_last, filter_last;   // offset of the operands' last 16 bytes
  int32_t xcoef, ycoef, yadd;
  uint32_t zpf4;                // the input zero point ^ 0x80 in all four bytes
  RequantFixed rq;
  RequantMad rqm;               // of rq, where by_mad
  bool by_mad;
};

__host__ __device__ inline uint32_t plane_magic(uint32_t d) { return d <= 1 ? 0u : (uint32_t)((1ull << 32) / d + 1); }
// n / d for n d < 2^32
__device__ __forceinline__ int plane_div(int n, uint32_t magic) {
  return magic == 0 ? n : (int)__umulhi((uint32_t)n, magic);
}
// The low n of four bytes (n below 0: none, above 4: all)
__device__ __forceinline__ uint32_t low_bytes(int n) {
  return n >= 4 ? 0xffffffffu : (n <= 0 ? 0u : (1u << (8 * n)) - 1u);
}
// ---- first launch: planes and packed filter ------------------------------------------------------
//
// planes[16 channels][image, row, column][16]: the input shifted (x ^ 0x80), pixels of the padding as the
// zero point, bytes past the channels anything (the packed filter is zero there).  2^lanes_log2 lanes take a
// pixel, a thread four of them.  packed[block of 32 channels][slab][k step][half][channel][16]: MFMA fragments;
// a wavefront takes a channel.  Bound by memory and by its own start: 12.8 MB in and 13.8 out in 4 - 5 us at 56 x 56 x
// 64, batch 64; 16 lanes at most and four pixels a thread, so that a layer's few thousand workgroups' starts do not
// outlast the copy (one pixel a thread: four times the workgroups, 1 us more on 28 x 28 x 128).
constexpr int PACK_PIXELS = 4;
__global__ __launch_bounds__(256) void q8_conv_planes_pack_kernel(ConvPlaneParams p) {
  const v4i flip = {(int)0x80808080, (int)0x80808080, (int)0x80808080, (int)0x80808080};
  const int all = p.slabs * p.pieces;
  if ((int)blockIdx.x < p.pixel_blocks) {
    const int lg = p.lanes_log2, g = threadIdx.x & ((1 << lg) - 1), slots = 256 >> lg;
    const int px0 = (int)blockIdx.x * slots * PACK_PIXELS + (int)(threadIdx.x >> lg);
    uint32_t base[PACK_PIXELS];
    bool inside[PACK_PIXELS];
    int sum[PACK_PIXELS];
#pragma unroll
    for (int u = 0; u < PACK_PIXELS; ++u) {
      const int px = min(px0 + u * slots, p.pixels - 1);
      const int r = plane_div(px, p.m_cw), col = px - r * p.cw;
      const int img = plane_div(r, p.m_vh), ih = r - img * p.vh - p.pt, iw = col - p.pl;
      inside[u] = (unsigned)ih < (unsigned)p.in_h && (unsigned)iw < (unsigned)p.in_w;
      base[u] = inside[u] ? (uint32_t)(((img * p.in_h + ih) * p.in_w + iw) * p.cin) : 0u;
      sum[u] = 0;
    }
    for (int pc = g; pc < all; pc += 1 << lg) {
      v4i v[PACK_PIXELS];
      const uint32_t c = (uint32_t)min(16 * pc, p.cin - 1);
#pragma unroll
      for (int u = 0; u < PACK_PIXELS; ++u) __builtin_memcpy(&v[u], p.in + min(base[u] + c, p.in_last), 16);
      __builtin_amdgcn_sched_barrier(0);
      const int left = p.cin - 16 * pc;
      v4i ones;
#pragma unroll
      for (int e = 0; e < 4; ++e) ones[e] = 0x01010101 & (int)low_bytes(left - 4 * e);
      uint8_t *to = p.planes + (uint32_t)pc * (uint32_t)p.plane_bytes;
#pragma unroll
      for (int u = 0; u < PACK_PIXELS; ++u) {
        if (base[u] + c > p.in_last) v[u] = moved_down(v[u], base[u] + c - p.in_last);
        v4i w = v[u] ^ flip;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          w[e] = inside[u] ? w[e] : (int)p.zpf4;
          sum[u] = __builtin_amdgcn_sdot4(w[e], ones[e], sum[u], false);
        }
        const int px = px0 + u * slots;
        if (px < p.pixels) *(v4i *)(to + (uint32_t)px * 16u) = w;
      }
    }
    for (int m = 1 << lg >> 1; m > 0; m >>= 1) {
#pragma unroll
      for (int u = 0; u < PACK_PIXELS; ++u) sum[u] += __shfl_xor(sum[u], m, 64);
    }
#pragma unroll
    for (int u = 0; u < PACK_PIXELS; ++u)
      if (g == 0 && px0 + u * slots < p.pixels) p.psum[px0 + u * slots] = sum[u];
  } else if (p.kept) {
    const int x = ((int)blockIdx.x - p.pixel_blocks) * 256 + (int)threadIdx.x;
    if (x < p.channels)
      p.cx[x] = (int32_t)((uint32_t)p.xcoef * (uint32_t)p.wsums[x] + (uint32_t)(p.bias && x < p.cout ? p.bias[x] : 0));
  } else {
    const int lane = threadIdx.x & 63;
    const int x = ((int)blockIdx.x - p.pixel_blocks) * 4 + (int)(threadIdx.x >> 6);
    const int slots = p.slabs * p.steps * 2;
    if (x >= p.channels) return;
    const bool real = x < p.cout;
    const uint32_t row = (uint32_t)(real ? x : 0) * (uint32_t)p.depth;
    uint8_t *dst = p.packed + (uint32_t)(x >> 5) * (uint32_t)(p.slabs * p.steps * 1024) + (x & 31) * 16;
    int sum = 0;
    for (int q0 = lane; q0 < slots; q0 += 256) {
      v4i v[4];
      int left[4];
      uint32_t off[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = min(q0 + 64 * u, slots - 1);
        const int slab = plane_div(q, p.m_slots), in_slab = q - slab * 2 * p.steps;
        const int run = plane_div(in_slab, p.m_run), in_run = in_slab - run * 2 * p.spr;
        const int tap = plane_div(in_run, p.m_pieces), c = (slab * p.pieces + in_run - tap * p.pieces) * 16;
        left[u] = real && in_run < p.run_len ? p.cin - c : 0;
        off[u] = row + (uint32_t)(left[u] > 0 ? (run * p.taps + tap) * p.cin + c : 0);
        __builtin_memcpy(&v[u], p.filter + min(off[u], p.filter_last), 16);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = q0 + 64 * u;
        if (q < slots) {
          if (off[u] > p.filter_last) v[u] = moved_down(v[u], off[u] - p.filter_last);
          v4i w = v[u] ^ flip;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            w[e] &= (int)low_bytes(left[u] - 4 * e);
            sum = __builtin_amdgcn_sdot4(w[e], 0x01010101, sum, false);
          }
          *(v4i *)(dst + (q >> 1) * 1024 + (q & 1) * 512) = w;
        }
      }
    }
    for (int m = 32; m > 0; m >>= 1) sum += __shfl_xor(sum, m, 64);
    if (lane == 0) {
      if (p.wsums) p.wsums[x] = sum;
      p.cx[x] = (int32_t)((uint32_t)p.xcoef * (uint32_t)sum + (uint32_t)(p.bias && real ? p.bias[x] : 0));
    }
  }
}

// ---- second launch -----------------------------------------------------------------------------
// The kernel's arguments where the launch put them.  Each phase of the kernel reads the ones that it needs
// anew: kept in registers over the whole kernel they do not fit, and are spilled instead.
#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(4))) ConvPlaneParams *PlaneArgs;
__device__ __forceinline__ PlaneArgs plane_args(const ConvPlaneParams &) {
  PlaneArgs p = (PlaneArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}
#else
typedef const ConvPlaneParams *PlaneArgs;
__host__ __device__ inline PlaneArgs plane_args(const ConvPlaneParams &p) { return &p; }
#endif

//
// A workgroup owns a tile of output channels x output pixels in the images' order.  The rows that its pixels reach
// lie one behind the other in the planes, padding and images included, so a stage of `stage_slabs` slabs is one
// contiguous piece of every plane and of the packed filter, transferred into LDS as it lies: no address is
// checked and no byte is touched on the way.  A fragment is one conflict-free 16-byte LDS read per lane (16 bytes of
// neighbouring pixels, or of the filter in lane order), k steps walk the taps by adding to its address, and the
// pixels' byte sums, taken once per pixel, are added up over the window in the epilogue.
//
// What bounds it (3 x 3 at batch 64, us; this launch alone on planes still in the caches): 28 x 28 x 128 -> 128 about
// 13, 14 x 14 x 256 -> 256 13, 56 x 56 x 64 -> 64 16.6, of which the transfers account for 1, the MFMAs for less
// than 1 and the epilogue for 3.6 (ablations): the rest is instruction issue and the waits of each tile's serial
// chain (transfer, barrier, k steps, requantization), hidden by three to four wavefronts a SIMD.  From the first
// launch's planes, which the eight L2s have handed back at its end, add 3 - 4.  An earlier form that staged and
// shifted the input itself, one launch, needed 45 vector instructions per staged piece in every workgroup: 28 -
// 32 us on these layers, 30 on 80 x 80 x 25 -> 17 at batch 52 (23.4 now); two halves of a pixel side by side in LDS
// gave every fragment read a two-way bank conflict.
//
// SPR: k steps of a filter row, slabs of two planes (0: any number, any slab)
template <int FX, int FY, int WX, int WY, int WK, int SPR, int OCC>
__global__ __launch_bounds__(64 * WX * WY * WK, OCC) void q8_conv_planes_kernel(ConvPlaneParams params) {
  PlaneArgs p = plane_args(params);
  constexpr int NW = WX * WY * WK, XT = WX * FX * 32, TP = WY * FY * 32;
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r32 = lane & 31;
  const int wk = wave % WK, wy = wave / WK % WY, wx = wave / (WK * WY);
  const int line = p->cw * 16;

  // A workgroup keeps its channel tile and takes a span of pixel tiles; those with the same span lie side by
  // side, and workgroup w runs on XCD w % 8: every XCD gets a contiguous span of workgroups.
  int wg = blockIdx.x;
  {
    const int per = (int)gridDim.x >> 3, more = (int)gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, more) + (wg >> 3);
  }
  const int group = plane_div(wg, p->m_tiles), x0 = (wg - group * p->tiles_x) * XT;
  const int t0 = group * p->span + min(group, p->span_more), t1 = t0 + p->span + (group < p->span_more ? 1 : 0);

  // ---- transfers into LDS, 1 KiB each: the filter's k steps, the rows of every slab, with a tile's first stage
  // the sums
  const mh_rsrc rs_planes = dma_rsrc(p->planes), rs_packed = dma_rsrc(p->packed), rs_psum = dma_rsrc((const uint8_t *)p->psum),
                rs_cx = dma_rsrc((const uint8_t *)p->cx);
  struct Tile { int px0, px1, row0, img0, first, nrows; };
  auto tile_of = [&](int t) {
    const PlaneArgs p = plane_args(params);
    Tile g;
    g.px0 = t * TP;
    g.px1 = min(g.px0 + TP, p->columns) - 1;
    const int g0 = plane_div(g.px0, p->m_ow), g1 = plane_div(g.px1, p->m_ow);       // output rows
    g.img0 = plane_div(g0, p->m_oh);
    const int img1 = plane_div(g1, p->m_oh);
    g.row0 = (g0 - g.img0 * p->out_h) * p->sh;
    g.first = g.img0 * p->vh + g.row0;                                             // first row of the planes
    g.nrows = img1 * p->vh + (g1 - img1 * p->out_h) * p->sh + p->k_h - g.first;
    return g;
  };
  auto issue = [&](const Tile &g, int slab0, int buf, int parity, bool filter) {
    const PlaneArgs p = plane_args(params);
    const int slabs = min(p->stage_slabs, p->slabs - slab0);
    const int fu = slabs * p->steps;                       // transfers of a block of 32 channels
    const int ru = (g.nrows * line + 1023) >> 10;         // ... of a plane's rows
    if (filter) {
      uint8_t *to = lds + (p->keep ? 0 : buf) * p->filter_bytes;
      for (int i = 0; i < XT / 32; ++i) {
        const uint32_t src = (uint32_t)((((x0 >> 5) + i) * p->slabs + slab0) * p->steps) * 1024u;
        for (int u = wave; u < fu; u += NW)
          dma_16B(rs_packed, (uint32_t)lane * 16, src + (uint32_t)u * 1024u, to + (i * p->stage_slabs * p->steps + u) * 1024);
      }
    }
    uint8_t *rows = lds + p->at_rows + buf * p->rows_bytes;
    for (int s = 0; s < slabs * p->pieces; ++s) {
      const uint32_t src = (uint32_t)((slab0 * p->pieces + s) * p->plane_bytes) + (uint32_t)(g.first * line);
      for (int u = wave; u < ru; u += NW)
        dma_16B(rs_planes, (uint32_t)lane * 16, src + (uint32_t)u * 1024u, rows + s * p->row_bytes + u * 1024);
    }
    if (slab0 == 0) {
      uint8_t *sums = lds + p->at_sums + parity * (p->psum_bytes + 1024);
      const int pu = (g.nrows * p->cw * 4 + 1023) >> 10;
      for (int u = wave; u < pu; u += NW)
        dma_16B(rs_psum, (uint32_t)lane * 16, (uint32_t)(g.first * p->cw * 4) + (uint32_t)u * 1024u, sums + u * 1024);
      if (wave == NW - 1) dma_16B(rs_cx, (uint32_t)lane * 16, (uint32_t)(x0 * 4), sums + p->psum_bytes);
    }
  };

  int buf = 0, parity = 0;
  Tile next = tile_of(t0);
  if (p->buffers == 2) issue(next, 0, 0, 0, true);
  for (int t = t0; t < t1; ++t) {
    const Tile g = next;
    // staged position of this lane's pixels
    int pos[FY];
#pragma unroll
    for (int j = 0; j < FY; ++j) {
      const int px = min(g.px0 + (wy * FY + j) * 32 + r32, g.px1);
      const int row = plane_div(px, p->m_ow), ow = px - row * p->out_w;
      const int img = plane_div(row, p->m_oh);
      pos[j] = ((img - g.img0) * p->vh + (row - img * p->out_h) * p->sh - g.row0) * p->cw + ow * p->sw;
    }
    v16i acc[FX][FY];
#pragma unroll
    for (int i = 0; i < FX; ++i)
#pragma unroll
      for (int j = 0; j < FY; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

    for (int slab0 = 0; slab0 < p->slabs; slab0 += p->stage_slabs) {
      p = plane_args(params);
      const bool more = slab0 + p->stage_slabs < p->slabs;
      if (p->buffers == 1) {
        __syncthreads();               // the stage before is read
        issue(g, slab0, 0, parity, !p->keep || t == t0);
        if (!more && t + 1 < t1) next = tile_of(t + 1);
      }
      asm volatile("" ::: "memory");
      wait_vmcnt<0>();                 // this wavefront's transfers have landed
      __builtin_amdgcn_s_barrier();    // ... and everybody else's; the stage before is read
      asm volatile("" ::: "memory");
      if (p->buffers == 2) {
        if (more) {
          issue(g, slab0 + p->stage_slabs, buf ^ 1, parity, true);
        } else if (t + 1 < t1) {
          next = tile_of(t + 1);
          issue(next, 0, buf ^ 1, parity ^ 1, !p->keep);
        }
      }
      // ---- multiply: this wavefront's part of the stage's filter rows
      p = plane_args(params);
      const int total = min(p->stage_slabs, p->slabs - slab0) * p->k_h, spr = SPR ? SPR : p->spr;
      const int r0 = total * wk / WK, r1 = total * (wk + 1) / WK;
      const int block = p->stage_slabs * p->steps * 1024;
      const uint8_t *xsrc = lds + (p->keep ? 0 : buf) * p->filter_bytes + wx * FX * block + r0 * spr * 1024 + lane * 16;
      const int slab = plane_div(r0, p->m_kh);
      int kh = r0 - slab * p->k_h;
      const int slab_rows = p->pieces * p->row_bytes, along = p->pieces == 2 ? 16 : 32;   // (one plane: two taps a k step)
      const uint8_t *ysrc[FY];
      {
        const uint8_t *rows = lds + p->at_rows + buf * p->rows_bytes + slab * slab_rows + kh * line +
                              h * (p->pieces == 2 ? p->row_bytes : 16);
#pragma unroll
        for (int j = 0; j < FY; ++j) ysrc[j] = rows + pos[j] * 16;
      }
      const int next_row = line, next_slab = slab_rows - (p->k_h - 1) * line, k_h = p->k_h;
      auto advance = [&]() __attribute__((always_inline)) {
        const bool wrap = ++kh == k_h;
        kh = wrap ? 0 : kh;
        const int by = wrap ? next_slab : next_row;
#pragma unroll
        for (int j = 0; j < FY; ++j) ysrc[j] += by;
        xsrc += spr * 1024;
      };
      if constexpr (SPR > 0) {
        // the fragments of a filter row are requested while those of the row before are multiplied
        auto fetch = [&](v4i (&xf)[SPR][FX], v4i (&yf)[SPR][FY]) __attribute__((always_inline)) {
#pragma unroll
          for (int st = 0; st < SPR; ++st) {
#pragma unroll
            for (int j = 0; j < FY; ++j) yf[st][j] = *(const v4i *)(ysrc[j] + st * 16);
#pragma unroll
            for (int i = 0; i < FX; ++i) xf[st][i] = *(const v4i *)(xsrc + i * block + st * 1024);
          }
          advance();
        };
        auto multiply = [&](const v4i (&xf)[SPR][FX], const v4i (&yf)[SPR][FY]) __attribute__((always_inline)) {
#pragma unroll
          for (int st = 0; st < SPR; ++st)
#pragma unroll
            for (int j = 0; j < FY; ++j)
#pragma unroll
              for (int i = 0; i < FX; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xf[st][i], yf[st][j], acc[i][j], 0, 0, 0);
        };
        // (not where two sets do not leave room for four wavefronts on a SIMD: those hide the wait better)
        v4i xa[SPR][FX], ya[SPR][FY], xb[SPR][FX], yb[SPR][FY];
        int n = r1 - r0;
        if constexpr (FX * FY > 1) {
          for (; n > 0; --n) {
            fetch(xa, ya);
            multiply(xa, ya);
          }
        } else {
          if (n > 0) fetch(xa, ya);
          while (n > 0) {
            if (n > 1) fetch(xb, yb);
            multiply(xa, ya);
            if (n > 2) fetch(xa, ya);
            if (n > 1) multiply(xb, yb);
            n -= 2;
          }
        }
      } else {
        for (int r = r0; r < r1; ++r) {
          for (int st = 0; st < spr; ++st) {
            v4i xf[FX], yf[FY];
#pragma unroll
            for (int j = 0; j < FY; ++j) yf[j] = *(const v4i *)(ysrc[j] + st * along);
#pragma unroll
            for (int i = 0; i < FX; ++i) xf[i] = *(const v4i *)(xsrc + i * block + st * 1024);
#pragma unroll
            for (int j = 0; j < FY; ++j)
#pragma unroll
              for (int i = 0; i < FX; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xf[i], yf[j], acc[i][j], 0, 0, 0);
          }
          advance();
        }
      }
      if (p->buffers == 2) buf ^= 1;
    }

    // ---- corrections
    p = plane_args(params);
    const int32_t *psum = (const int32_t *)(lds + p->at_sums + parity * (p->psum_bytes + 1024));
    const int32_t *cx = psum + p->psum_bytes / 4;
    parity ^= 1;
    uint32_t cy[FY];
#pragma unroll
    for (int j = 0; j < FY; ++j) {
      int sum = 0;
      if (p->ycoef != 0)
        for (int kh = 0; kh < p->k_h; ++kh)
          for (int kw = 0; kw < p->k_w; ++kw) sum += psum[pos[j] + kh * p->cw + kw];
      cy[j] = (uint32_t)p->ycoef * (uint32_t)sum + (uint32_t)p->yadd;
    }
    // ---- the parts of the depth are added up: block b of the tile by wavefront b % WK of its group
    v4i *part = (v4i *)(lds + p->at_part) + (wave / WK) * (FX * FY * WK * 4 * 64);
    if constexpr (WK > 1) {
      __syncthreads();   // the last stage is read
      // [group][block][part][register group][lane] of 16 bytes
#pragma unroll
      for (int i = 0; i < FX; ++i)
#pragma unroll
        for (int j = 0; j < FY; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            part[(((i * FY + j) * WK + wk) * 4 + q) * 64 + lane] =
                v4i{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      __syncthreads();
    }
    const RequantFixed rq{p->rq.mult, p->rq.shift, p->rq.mask, p->rq.half, p->rq.blo, p->rq.bhi, p->rq.zp};
    const RequantMad rqm{p->rqm.c, p->rqm.mult, p->rqm.sh, p->rqm.lo, p->rqm.hi, p->rqm.no_sign, p->rqm.plus_x,
                         p->rqm.clamp, p->rqm.more};
    const bool by_mad = p->by_mad;
#pragma unroll
    for (int j = 0; j < FY; ++j) {
      const int px = g.px0 + (wy * FY + j) * 32 + r32;
      uint8_t *orow = p->out + (int64_t)px * p->cout + x0;
      if (g.px0 + (wy * FY + j) * 32 > g.px1) continue;
#pragma unroll
      for (int i = 0; i < FX; ++i) {
        if constexpr (WK > 1) {
          if ((i * FY + j) % WK != wk) continue;
        }
        const int xb = (wx * FX + i) * 32;
        if (x0 + xb >= p->cout) continue;
        if constexpr (WK > 1) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v4i sum = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < WK; ++k) sum += part[(((i * FY + j) * WK + k) * 4 + q) * 64 + lane];
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
        if (by_mad) {
          requant_16_by_mad(v, rqm, packed);
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) packed[r / 4] |= (uint32_t)mh_requant_fixed(v[r], rq) << (8 * (r % 4));
        }
        const v2u s02 = __builtin_amdgcn_permlane32_swap(packed[0], packed[2], false, false);
        const v2u s13 = __builtin_amdgcn_permlane32_swap(packed[1], packed[3], false, false);
        const v4i w = {(int)s02.x, (int)s02.y, (int)s13.x, (int)s13.y};
        const int xh = xb + 16 * h;
        if (px <= g.px1) {
          if (x0 + xh + 16 <= p->cout) {
            __builtin_memcpy(orow + xh, &w, 16);
          } else {
#pragma unroll
            for (int e = 0; e < 16; ++e)
              if (x0 + xh + e < p->cout) orow[xh + e] = (uint8_t)(((uint32_t)w[e / 4] >> (8 * (e % 4))) & 0xff);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// The tile forms: blocks of 32 channels and of 32 pixels of a wavefront, wavefronts along each and along the depth.
struct PlaneForm { int fx, fy, wx, wy, wk; };
constexpr PlaneForm kPlaneForms[mhv::PLANES_FORMS] = {{2, 1, 1, 8, 1}, {1, 2, 1, 4, 1}, {1, 1, 1, 4, 1}, {1, 1, 1, 1, 4}};
struct PlaneShape { int64_t n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, pt, pl, out_h, out_w; };
struct PlanePlan { int xt, tp, threads, pack_blocks; int64_t lds, scratch, packed_bytes, psum_bytes, cx_bytes, planes_bytes; bool fits; };
// Geometry, LDS and scratch of a form whose stages take up to `budget` bytes of LDS together.
PlanePlan plane_plan(const PlaneForm &f, const PlaneShape &s, int64_t budget, int buffers, ConvPlaneParams *p) {
  PlanePlan r{};
  r.xt = f.fx * f.wx * 32;
  r.tp = f.fy * f.wy * 32;
  r.threads = 64 * f.wx * f.wy * f.wk;
  const int64_t vh = (s.out_h - 1) * s.sh + s.k_h, cw = (s.out_w - 1) * s.sw + s.k_w, depth = s.k_h * s.k_w * s.cin;
  const int64_t columns = s.n * s.out_h * s.out_w, pixels = s.n * vh * cw;
  const int all = (int)((s.cin + 15) / 16);
  // A k step takes the same tap of two planes, or two taps of the only one there is.
  const int pieces = all == 1 ? 1 : 2, slabs = (all + pieces - 1) / pieces;
  p->n = (int)s.n; p->in_h = (int)s.in_h; p->in_w = (int)s.in_w; p->cin = (int)s.cin; p->cout = (int)s.cout;
  p->k_h = (int)s.k_h; p->k_w = (int)s.k_w; p->sh = (int)s.sh; p->sw = (int)s.sw; p->pt = (int)s.pt; p->pl = (int)s.pl;
  p->out_h = (int)s.out_h; p->out_w = (int)s.out_w;
  p->depth = (int)depth; p->columns = (int)columns;
  p->tiles_x = (int)((s.cout + r.xt - 1) / r.xt);
  p->tiles_p = (int)((columns + r.tp - 1) / r.tp);
  p->channels = p->tiles_x * r.xt;
  p->vh = (int)vh; p->cw = (int)cw; p->pixels = (int)pixels;
  p->pieces = pieces; p->slabs = slabs;
  p->taps = (int)s.k_w; p->run_len = p->taps * pieces; p->spr = (p->run_len + 1) / 2; p->steps = (int)s.k_h * p->spr;
  p->lanes_log2 = 0;
  while (p->lanes_log2 < 4 && (1 << p->lanes_log2) < all) ++p->lanes_log2;
  p->pixel_blocks = (int)(((pixels << p->lanes_log2) + 256 * PACK_PIXELS - 1) / (256 * PACK_PIXELS));
  r.pack_blocks = p->pixel_blocks + (p->channels + 3) / 4;
  const int64_t plane = (int64_t)mh_align_up((size_t)(pixels * 16), 1024);
  // rows that a tile's pixels reach: they lie in at most out_rows rows of at most images + 1 images
  const int64_t out_rows = (r.tp - 2) / s.out_w + 2, images = (out_rows - 1 + s.out_h - 1) / s.out_h;
  const int64_t rows = (out_rows - 1) * s.sh + s.k_h + images * std::max<int64_t>(0, s.k_h - s.sh);
  // (a run of an odd number of pieces reads half a k step on)
  const int64_t row_bytes = (int64_t)mh_align_up((size_t)(rows * cw * 16 + 16), 1024);
  const int64_t slab_filter = (int64_t)p->steps * r.xt * 32, slab_rows = pieces * row_bytes;
  const int64_t part = f.wk > 1 ? (int64_t)f.wx * f.wy * f.wk * f.fx * f.fy * 4096 : 0;
  const int64_t psum_lds = (int64_t)mh_align_up((size_t)(rows * cw * 4), 1024);
  const int64_t sums = 2 * (psum_lds + 1024);
  const int64_t room = budget - sums;
  p->keep = slabs * (slab_filter + buffers * slab_rows) <= room;
  int64_t stage = slabs;
  if (!p->keep) {
    stage = std::max<int64_t>(1, std::min<int64_t>(slabs, room / buffers / (slab_filter + slab_rows)));
    stage = (slabs + (slabs + stage - 1) / stage - 1) / ((slabs + stage - 1) / stage);   // stages of like length
  }
  const int64_t at_rows = (p->keep ? 1 : buffers) * stage * slab_filter, operands = at_rows + buffers * stage * slab_rows;
  // (the parts' sums take the place of the stage just read where it is the only one there)
  const int64_t at_part = p->keep || buffers == 2 ? operands : 0, at_sums = std::max<int64_t>(operands, at_part + part);
  r.lds = at_sums + sums;
  p->buffers = buffers;
  p->stage_slabs = (int)stage; p->row_bytes = (int)row_bytes;
  p->filter_bytes = (int)(stage * slab_filter); p->rows_bytes = (int)(stage * slab_rows);
  p->at_rows = (int)at_rows; p->at_part = (int)at_part; p->at_sums = (int)at_sums; p->psum_bytes = (int)psum_lds;
  p->plane_bytes = (int)plane;
  r.packed_bytes = (int64_t)p->channels * slabs * p->steps * 32;
  r.psum_bytes = (int64_t)mh_align_up((size_t)(pixels * 4 + 2048), 256);   // (transfers read whole KiB)
  r.cx_bytes = (int64_t)p->channels * 4 + 1024;
  r.planes_bytes = plane * slabs * pieces + 2048;
  r.scratch = r.planes_bytes + r.packed_bytes + r.psum_bytes + r.cx_bytes;
  r.fits = r.planes_bytes < (1ll << 31) && r.packed_bytes < (1ll << 31) && pixels * 4 < (1ll << 31) && r.lds < (1 << 30) &&
           4ll * slabs * p->steps * p->steps < (1ll << 32) &&
           (pixels << p->lanes_log2) < (1ll << 31);
  // (one image: every row is its own, whatever the divisor)
  p->m_cw = plane_magic((uint32_t)cw); p->m_vh = s.n > 1 ? plane_magic((uint32_t)vh) : 1;
  p->m_ow = plane_magic((uint32_t)s.out_w); p->m_oh = s.n > 1 ? plane_magic((uint32_t)s.out_h) : 1;
  p->m_tiles = plane_magic((uint32_t)p->tiles_x); p->m_pieces = plane_magic((uint32_t)pieces);
  p->m_slots = plane_magic((uint32_t)(2 * p->steps)); p->m_run = plane_magic((uint32_t)(2 * p->spr));
  p->m_kh = plane_magic((uint32_t)s.k_h);
  p->in_last = (uint32_t)(s.n * s.in_h * s.in_w * s.cin - 16); p->filter_last = (uint32_t)(s.cout * depth - 16);
  return r;
}
// what the kernels' 32-bit offsets and magics hold
bool plane_fits(const PlaneShape &s) {
  const int64_t depth = s.k_h * s.k_w * s.cin, columns = s.n * s.out_h * s.out_w;
  const int64_t vh = (s.out_h - 1) * s.sh + s.k_h, cw = (s.out_w - 1) * s.sw + s.k_w;
  const int64_t in_bytes = s.n * s.in_h * s.in_w * s.cin, filter_bytes = s.cout * depth;
  if (s.cin < 1 || depth >= (1 << 20) || vh >= (1 << 30) || cw >= (1 << 15) || s.n * vh >= (1ll << 30) || s.cout >= (1 << 20))
    return false;
  return in_bytes >= 16 && filter_bytes >= 16 && in_bytes < (1ll << 31) - 64 && filter_bytes < (1ll << 31) - 64 &&
         s.n * vh * cw * cw < (1ll << 32) &&
         (s.n == 1 || (s.n * vh * vh < (1ll << 32) && s.n * s.out_h * s.out_h < (1ll << 32))) && columns * s.out_w < (1ll << 32) && columns < (1 << 30);
}
}  // namespace

// Time that the one-launch GEMM kernel (q8_gemm_fused_small_kernel) would take, in us: a workgroup's depth, in
// pieces of 16, 4 or 1 bytes, and those of a CU's workgroups together, whose square sum it follows.  (Within 3 % in the
// median of 300 drawn 3 x 3 layers, 8 % in nine of ten; model and measured: 61 x 59 x 29 -> 80 at batch 12 39 and 34, 33 x
// 34 x 112 -> 214 at 22 31 and 32, 20 x 22 x 35 -> 38 at 3 16 and 15, 36 x 36 x 20 -> 112 at 1 5.8 and 6.1.)
double mh_q8_conv_small_us(const mace_hip_ctx *ctx, int64_t cout, int64_t columns, int64_t depth, int piece) {
  const double cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
  const double wgs = (double)((cout + 63) / 64) * (double)((columns + 63) / 64) / cu;
  if (piece == 16) return 4.6 + hypot(0.0076 * depth - 0.27, wgs * (0.0034 * depth + 0.45));
  if (piece == 4) return 2.0 + hypot(0.0137 * depth + 2.3, wgs * (0.002 * depth + 1.45));
  return 5.6 + hypot(0.0315 * depth - 0.25, wgs * (0.0124 * depth + 0.89));
}

// Time of the two launches, in us: their start, the bytes that the first moves, and what a CU's tiles cost each (the
// hand-over, the stages' bytes) and one after the other (k steps).  By tile form and by whether a filter row is three k
// steps; 32 x 256, which few calls take, as 64 x 256.  Within 5 % in the median of 1400 layers of all kinds, 13 % in nine
// of ten.
struct PlaneCost { double start, per_mb, per_tile, per_staged, per_step; };   // (staged: 100 KB)
static double planes_us(int form, const ConvPlaneParams &p, const PlaneShape &s, int64_t staged, int64_t span, int64_t at_once) {
  static const PlaneCost kThree[3] = {{6.8, 0.178, 1.76, 1.23, 0.111}, {7.8, 0.183, 0.565, 0.926, 0.060}, {8.3, 0.186, 0.313, 0.722, 0.038}};
  static const PlaneCost kAny[3] = {{9.3, 0.121, 1.40, 1.77, 0.096}, {9.0, 0.15, 0.09, 1.24, 0.072}, {9.2, 0.36, 0.02, 1.0, 0.033}};
  const PlaneCost &c = (p.spr == 3 && p.pieces == 2 ? kThree : kAny)[std::max(0, form - 1)];
  const double moved = (double)s.n * s.in_h * s.in_w * s.cin + (double)p.plane_bytes * p.slabs * p.pieces;
  return c.start + c.per_mb * moved / 1e6 + at_once * span * (c.per_tile + c.per_staged * staged / 1e5) +
         c.per_step * span * p.slabs * p.steps;
}

// *taken = false: not a call for it.  `other`: an estimate of the time, in us, that the call takes otherwise (HUGE_VAL
// where a patch matrix of several taps is written out: of 700 such layers none was faster than the planes).
//
// Two launches take 8.2 us at the least where a caller waits for none of them, one 4.  Against the kernels that
// took these calls before (3 x 3, us): an im2col of odd channel counts 34 x 36 x 108 -> 28 at batch 52 146 -> 17.5,
// 96 x 97 x 38 -> 21 at 7 65.6 -> 13.3, 7 x 9 x 797 -> 209 at 16 55.6 -> 17.8, 80 x 81 x 97 -> 35 of one image 24 -> 10;
// of whole pieces 27 x 29 x 224 -> 24 at 37 29.7 -> 15.4, 14 x 14 x 256 -> 256 at 64 27 -> 19, 7 x 7 x 512 -> 512 at 64
// 29 -> 24; a gathering GEMM on 128 channels 28 x 28 -> 128 at 64 21.3 -> 18.9.  A tile of 64 x 256 reads three fragments from LDS per two
// products, the gathering GEMM's 256 x 256 eight per sixteen, so layers that fill its rounds stay there, and so do
// strides that leave most of what the first launch copies unused: 56 x 56 x 512 -> 256 at stride 2, batch 64, 84 against
// 132 here, 28 x 28 x 1024 -> 1024 at stride 2, 64, 143 against 203, 28 x 28 x 256 -> 256 at 64 46 against 52, 56 x 56 x
// 128 -> 64 at stride 2, 64, 18.0 against 24.9; but 28 x 28 x 512 -> 256 at 32 49 against 43, 56 x 56 x 256 -> 256 at 8
// 30 against 25.  Of 712 gathered layers 104 lost more than 3 % here (the worst 71 %) before both times were estimated,
// 11 since (10 %).
int mh_q8_conv_planes(mace_hip_ctx *ctx, const uint8_t *input, const uint8_t *filter, const int32_t *bias,
                      int64_t n, int64_t in_h, int64_t in_w, int64_t cin, int64_t cout, int64_t k_h,
                      int64_t k_w, int stride_h, int stride_w, int pad_top, int pad_left, int64_t out_h,
                      int64_t out_w, float input_scale, int32_t input_zp, float filter_scale, int32_t filter_zp,
                      float bias_scale, int32_t mult, int shift, int32_t out_zp, int clamp_min, int clamp_max,
                      uint8_t *out, double other, bool *taken) {
  *taken = false;
  // (the two launches' start alone, before a tile's geometry is worked out: calls of 4 - 6 us notice a tenth)
  if (0.95 * other <= 7.5) return MACE_HIP_SUCCESS;
  const PlaneShape s{n, in_h, in_w, cin, cout, k_h, k_w, stride_h, stride_w, pad_top, pad_left, out_h, out_w};
  if (!plane_fits(s) || filter_zp < 0 || filter_zp > 255 || (ctx->kernel_mask & MH_MASK_NO_CONV_SHORT))
    return MACE_HIP_SUCCESS;
  if (shift < 0 || shift > 31 || clamp_min < 0 || clamp_max > 255 || clamp_min > clamp_max)
    return MACE_HIP_SUCCESS;   // (the general path reports these)
  const int64_t columns = n * out_h * out_w;
  ConvPlaneParams p{};
  if (!mh_make_requant(mult, shift, out_zp, clamp_min, clamp_max, &p.rq)) return MACE_HIP_SUCCESS;
  p.by_mad = requant_by_mad(p.rq);
  if (p.by_mad) p.rqm = requant_mad(p.rq);

  // The largest tiles that give most CUs one; with fewer, wavefronts share a tile's depth.  A tile a CU or less: all of
  // the LDS, the next stage on its way; else two workgroups a CU that wait in turn.  (3 x 3, us: 28 x 28 x 128 -> 128
  // at batch 64, 392 tiles of 64 x 256, 18.9, 784 of 64 x 128 20.2; 7 x 7 x 512 -> 512 at 64, 104 of 64 x 256 27, 400 of
  // 32 x 128 24.4; 80 x 80 x 25 -> 17 at 52, 1300 of 32 x 256 23.4, 2600 of 32 x 128 26; 27 x 29 x 224 -> 24 at 37, 61 of
  // 32 x 128 17, 243 of 32 x 32 in four parts 15.4.)
  const int64_t cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
  auto tiles = [&](int form) {
    const PlaneForm &f = kPlaneForms[form];
    return ((cout + 32 * f.fx * f.wx - 1) / (32 * f.fx * f.wx)) * ((columns + 32 * f.fy * f.wy - 1) / (32 * f.fy * f.wy));
  };
  int form = mhv::PLANES_32x32;
  if (cout > 32 && 8 * tiles(mhv::PLANES_64x256) >= 5 * cu) form = mhv::PLANES_64x256;
  else if (cout <= 32 && 2 * tiles(mhv::PLANES_32x256) >= 5 * cu) form = mhv::PLANES_32x256;
  else if (5 * tiles(mhv::PLANES_32x128) >= 2 * cu) form = mhv::PLANES_32x128;
  PlanePlan plan{};
  for (;; ++form) {   // (rows too wide for LDS beside a large tile's filter: smaller ones)
    const bool one = tiles(form) <= cu;
    plan = plane_plan(kPlaneForms[form], s, (one ? 156 : 78) * 1024, one ? 2 : 1, &p);
    if (plan.lds > ctx->lds_bytes) plan = plane_plan(kPlaneForms[form], s, 78 * 1024, 1, &p);
    if (plan.lds <= ctx->lds_bytes || form + 1 == mhv::PLANES_FORMS) break;
  }
  if (!plan.fits || plan.lds > ctx->lds_bytes || !mh_arena_can_hold(ctx, (size_t)plan.scratch + 8 * 256 + 4 * cout))
    return MACE_HIP_SUCCESS;
  const int64_t at_once = std::max<int64_t>(1, std::min<int64_t>(ctx->lds_bytes / std::max<int64_t>(1, plan.lds), 1024 / plan.threads));
  // (workgroups of a channel tile: as many as fit at once)
  const int64_t room = std::min<int64_t>(p.tiles_p, std::max<int64_t>(1, cu * at_once / p.tiles_x));
  const int64_t staged = (p.keep ? 0 : (int64_t)p.slabs * p.steps * plan.xt * 32) + (int64_t)p.slabs * p.pieces * p.row_bytes;
  // (packing the filter is 1 us a MB of it, which a registered one costs once: 7 x 7 x 512 -> 512 at batch 64 24.6 and 22.1)
  mh_weight *weight = mh_find_weight(ctx, filter, (size_t)(cout * p.depth));
  const double us = planes_us(form, p, s, staged, (p.tiles_p + room - 1) / room, (room * p.tiles_x + cu - 1) / cu);
  if (us - (weight ? 1e-6 * cout * p.depth : 0.0) >= 0.95 * other) return MACE_HIP_SUCCESS;
  *taken = true;

  MH_RETURN_IF_ERROR(mh_arena_reserve(ctx, (size_t)plan.scratch + 8 * 256 + sizeof(int32_t) * cout));
  ArenaScope scope(ctx);
  const int32_t *bias_used = nullptr;
  MH_RETURN_IF_ERROR(mh_conv_bias(ctx, bias, cout, input_scale, filter_scale, bias_scale, &bias_used));
  // A registered filter is packed and summed once, into memory of its own.  (Not where that cannot be had, nor in a
  // capture, which would fill it at a replay only: then as any other filter.)
  mh_weight_planes built{cin, cout, k_h, k_w, p.channels, nullptr, nullptr};
  auto give_back = [&]() {
    if (!ctx->plan_only) { (void)hipFree(built.packed); (void)hipFree(built.sums); }
    built.packed = nullptr;
  };
  if (weight) {
    for (const mh_weight_planes &c : weight->planes)
      if (c.cin == cin && c.cout == cout && c.k_h == k_h && c.k_w == k_w && c.channels >= p.channels) {
        p.kept = true;
        p.packed = c.packed;
        p.wsums = c.sums;
      }
    if (!p.kept && ctx->plan_only) {   // (addresses stand in for the two buffers)
      built.packed = (uint8_t *)(uintptr_t)0x300000000ull;
      built.sums = (int32_t *)(uintptr_t)0x300000000ull;
    } else if (!p.kept && !ctx->capturing) {
      if (hipMalloc((void **)&built.packed, (size_t)plan.packed_bytes) != hipSuccess ||
          hipMalloc((void **)&built.sums, (size_t)p.channels * 4) != hipSuccess) {
        (void)hipGetLastError();
        give_back();
      }
    }
    if (built.packed) {
      p.packed = built.packed;
      p.wsums = built.sums;
    }
  }
  if (p.kept) plan.pack_blocks = p.pixel_blocks + (p.channels + 255) / 256;
  if (!p.packed) p.packed = (uint8_t *)mh_arena_take(ctx, (size_t)plan.packed_bytes);
  p.psum = (int32_t *)mh_arena_take(ctx, (size_t)plan.psum_bytes);
  p.cx = (int32_t *)mh_arena_take(ctx, (size_t)plan.cx_bytes);
  p.planes = (uint8_t *)mh_arena_take(ctx, (size_t)plan.planes_bytes);
  if (!p.packed || !p.psum || !p.cx || !p.planes) {
    give_back();
    return mh_fail(ctx, MACE_HIP_RUNTIME_ERROR, "arena slice unavailable");
  }
  p.in = input; p.filter = filter; p.bias = bias_used; p.out = out;
  const uint32_t zl = (uint32_t)filter_zp - 128u, zr = (uint32_t)input_zp - 128u;
  p.xcoef = (int32_t)(0u - zr); p.ycoef = (int32_t)(0u - zl); p.yadd = (int32_t)((uint32_t)p.depth * zl * zr);
  p.zpf4 = ((uint32_t)(input_zp & 0xff) * 0x01010101u) ^ 0x80808080u;
  const size_t lds = (size_t)plan.lds;
  const bool three = p.spr == 3 && p.pieces == 2;
  auto launch = [&](auto kernel) -> int {
    MH_HIP(ctx, mh_allow_big_lds(ctx, (const void *)kernel, lds));
    const int64_t fit = cu * mh_blocks_per_cu(ctx, (const void *)kernel, plan.threads, lds);
    // workgroups of a channel tile: as many as fit at once
    const int64_t groups = std::min<int64_t>(p.tiles_p, std::max<int64_t>(1, fit / p.tiles_x));
    p.span = (int)(p.tiles_p / groups); p.span_more = (int)(p.tiles_p % groups);
    mh_plan_aux(ctx, MACE_HIP_AUX_CONV_PLANES | (p.kept ? MACE_HIP_AUX_WEIGHT_HIT : 0) | (built.packed ? MACE_HIP_AUX_WEIGHT_BUILD : 0));
    MH_KLAUNCH(ctx, q8_conv_planes_pack_kernel, dim3((unsigned)plan.pack_blocks), dim3(256), 0, ctx->stream, p);
    dim3 grid((unsigned)(groups * p.tiles_x)), block((unsigned)plan.threads);
    mh_plan_main(ctx, MACE_HIP_KF_Q8_CONV_PLANES, mhv::conv_planes(form, three), grid, block, (int)lds);
    MH_PROF_BEGIN(ctx);
    MH_KLAUNCH(ctx, kernel, grid, block, lds, ctx->stream, p);
    MH_PROF_END(ctx);
    MH_LAUNCH_CHECK(ctx);
    return MACE_HIP_SUCCESS;
  };
  int rc = MACE_HIP_SUCCESS;
#define MH_PLANES(...)                                                                 \
  rc = three ? launch(q8_conv_planes_kernel<__VA_ARGS__, 3, 4>) : launch(q8_conv_planes_kernel<__VA_ARGS__, 0, 4>)
  switch (form) {
    case mhv::PLANES_64x256: MH_PLANES(2, 1, 1, 8, 1); break;
    case mhv::PLANES_32x256: MH_PLANES(1, 2, 1, 4, 1); break;
    case mhv::PLANES_32x128: MH_PLANES(1, 1, 1, 4, 1); break;
    default: MH_PLANES(1, 1, 1, 1, 4); break;
  }
#undef MH_PLANES
  if (rc == MACE_HIP_SUCCESS && p.kept) ++ctx->weight_hits;
  if (rc == MACE_HIP_SUCCESS && built.packed) {
    weight->planes.push_back(built);
    ++ctx->weight_builds;
  } else if (built.packed) {
    give_back();
  }
  return rc;
}
