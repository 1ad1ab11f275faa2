// Runs the SOURCE of the uint8 GEMM kernels of mace_amd/csrc/q8_gemm.hip, of the convolution on padded planes and of
// some fp32 kernels on the CPU:
// kernel_emu_extract.py cuts their text out, this file supplies what the text needs from the GPU
// (thread and block indices, LDS, barriers, and the wavefront-wide instructions -- MFMA, lane
// shuffles, transfers into LDS, the transposing LDS read -- as collectives over the 64 host threads
// of a wavefront), and every case runs one launch with operands allocated at exactly their size.
// Built with AddressSanitizer: an access outside an operand aborts the run.  int32 results are
// compared with sums formed directly from the operands; uint8 launches must write every byte of
// the result (the requantization ends in GPU assembly and has no host form, so their values are not
// compared here; the GPU parity tests do that).
//
// What this covers is indexing and arithmetic of the source: row clamps, ragged tiles, depth
// tails, swizzles, store guards.  A transfer into LDS lands at once here, so the order of
// asynchronous transfers and reads is not covered, nor the compiler's GPU code, nor anything
// written in GPU assembly.
#include <algorithm>
#include <barrier>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <thread>
#include <type_traits>
#include <vector>
using std::max;
using std::min;

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline __attribute__((always_inline))
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define __shared__ static   // one workgroup runs at a time: a function's static is that workgroup's LDS

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
thread_local dim3 threadIdx, blockIdx;
dim3 gridDim, blockDim;

typedef int e4i __attribute__((ext_vector_type(4)));
typedef int e16i __attribute__((ext_vector_type(16)));
typedef unsigned e2u __attribute__((ext_vector_type(2)));
typedef unsigned uint4 __attribute__((ext_vector_type(4)));

struct Wave {
  std::barrier<> bar{64};
  e4i a[64], b[64];
  uint32_t w[64][2];
  uint64_t piece[64];
};
struct Block {
  std::barrier<> *bar = nullptr;   // of the launch's workgroup size
  Wave waves[8];
  alignas(16) uint8_t lds[160 * 1024];
};
static Block g_block;
static inline Wave &wave_of_thread() { return g_block.waves[threadIdx.x >> 6]; }
static inline int lane_of_thread() { return threadIdx.x & 63; }
uint8_t *emu_lds() { return g_block.lds; }
void __syncthreads() { g_block.bar->arrive_and_wait(); }
void emu_s_barrier() { g_block.bar->arrive_and_wait(); }

// ---- wavefront-wide instructions: every lane of the wavefront calls them together ---------------
int __shfl_xor(int v, int m, int = 64) {
  Wave &w = wave_of_thread();
  const int l = lane_of_thread();
  w.w[l][0] = (uint32_t)v;
  w.bar.arrive_and_wait();
  const int r = (int)w.w[l ^ m][0];
  w.bar.arrive_and_wait();
  return r;
}
// v_permlane32_swap: the upper half of the first register changes places with the lower half of
// the second; returns {first, second} afterwards
e2u emu_permlane32_swap(uint32_t a, uint32_t b, bool, bool) {
  Wave &w = wave_of_thread();
  const int l = lane_of_thread();
  w.w[l][0] = a;
  w.w[l][1] = b;
  w.bar.arrive_and_wait();
  e2u r;
  if (l < 32) { r.x = a; r.y = w.w[l + 32][0]; }
  else { r.x = w.w[l - 32][1]; r.y = b; }
  w.bar.arrive_and_wait();
  return r;
}
// v_mfma_i32_32x32x32_i8: lane l supplies row l % 32 of each operand, k bytes [16 (l / 32), +16);
// result register r of lane l is element (row 8 (r / 4) + 4 (l / 32) + r % 4 of the first operand,
// row l % 32 of the second)
e16i emu_mfma(e4i a, e4i b, e16i c, int, int, int) {
  Wave &w = wave_of_thread();
  const int l = lane_of_thread();
  w.a[l] = a;
  w.b[l] = b;
  w.bar.arrive_and_wait();
  const int y = l & 31;
  for (int r = 0; r < 16; ++r) {
    const int x = 8 * (r / 4) + 4 * (l / 32) + r % 4;
    int s = 0;
    for (int h = 0; h < 2; ++h) {
      const int8_t *pa = (const int8_t *)&w.a[x + 32 * h], *pb = (const int8_t *)&w.b[y + 32 * h];
      for (int k = 0; k < 16; ++k) s += (int)pa[k] * (int)pb[k];
    }
    c[r] += s;
  }
  w.bar.arrive_and_wait();
  return c;
}
// ds_read_b64_tr_b8: within 16 lanes the instruction takes 8 bytes at each lane's address and hands
// lane j < 8 byte j of the even lanes' pieces, lane 8 + j byte j of the odd lanes' pieces
typedef int v2i_t __attribute__((ext_vector_type(2)));
template <int OFF>
v2i_t lds_read_tr8(int lds_byte_address) {
  Wave &w = wave_of_thread();
  const int l = lane_of_thread();
  memcpy(&w.piece[l], g_block.lds + lds_byte_address + OFF, 8);
  w.bar.arrive_and_wait();
  const int g = l & ~15, j = l & 7, odd = (l >> 3) & 1;
  uint8_t out[8];
  for (int i = 0; i < 8; ++i) out[i] = (uint8_t)(w.piece[g + 2 * i + odd] >> (8 * j));
  w.bar.arrive_and_wait();
  v2i_t r;
  memcpy(&r, out, 8);
  return r;
}
inline void lds_wait_tr(e4i &, int) {}
inline void lds_written() { wave_of_thread().bar.arrive_and_wait(); }
inline int lds_address_of(const uint8_t *p) { return (int)(p - g_block.lds); }
// ---- per-lane instructions ------------------------------------------------------------------------
uint32_t emu_sad_u8(uint32_t a, uint32_t b, uint32_t c) {
  for (int i = 0; i < 4; ++i) c += (uint32_t)std::abs((int)((a >> (8 * i)) & 255) - (int)((b >> (8 * i)) & 255));
  return c;
}
int emu_sdot4(int a, int b, int c, bool) {
  for (int i = 0; i < 4; ++i) c += (int)(int8_t)(a >> (8 * i)) * (int)(int8_t)(b >> (8 * i));
  return c;
}
uint32_t emu_udot4(uint32_t a, uint32_t b, uint32_t c, bool) {
  for (int i = 0; i < 4; ++i) c += ((a >> (8 * i)) & 255) * ((b >> (8 * i)) & 255);
  return c;
}
uint32_t emu_perm(uint32_t hi, uint32_t lo, uint32_t sel) {
  const uint64_t both = ((uint64_t)hi << 32) | lo;
  uint32_t r = 0;
  for (int i = 0; i < 4; ++i) {
    const uint32_t s = (sel >> (8 * i)) & 255;
    r |= (s < 8 ? (uint32_t)((both >> (8 * s)) & 255) : 0u) << (8 * i);
  }
  return r;
}
// v_mov_dpp within sixteen lanes: a permutation of four, eight or sixteen lanes mirrored
int emu_update_dpp(int, int v, int ctrl, int, int, bool) {
  Wave &w = wave_of_thread();
  const int l = lane_of_thread();
  w.w[l][0] = (uint32_t)v;
  w.bar.arrive_and_wait();
  const int from = ctrl == 0x140 ? l ^ 15 : (ctrl == 0x141 ? l ^ 7 : (l & ~3) + ((ctrl >> (2 * (l & 3))) & 3));
  const int r = (int)w.w[from][0];
  w.bar.arrive_and_wait();
  return r;
}
uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
float __fmaf_rn(float a, float b, float c) { return fmaf(a, b, c); }
inline int emu_readfirstlane(int v) { return v; }
#define __builtin_amdgcn_mfma_i32_32x32x32_i8 emu_mfma
#define __builtin_amdgcn_permlane32_swap emu_permlane32_swap
#define __builtin_amdgcn_sad_u8 emu_sad_u8
#define __builtin_amdgcn_sdot4 emu_sdot4
#define __builtin_amdgcn_udot4 emu_udot4
#define __builtin_amdgcn_perm emu_perm
#define __builtin_amdgcn_update_dpp emu_update_dpp
#define __builtin_amdgcn_sched_group_barrier(...) ((void)0)
#define __builtin_amdgcn_readfirstlane emu_readfirstlane
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_s_barrier emu_s_barrier

// ---- what the kernels' text takes from common.h and from other parts of q8_gemm.hip --------------
struct RequantFixed {
  int32_t mult, shift, mask, half, blo, bhi, zp;
};
// a byte of the accumulator where the multiplier asks for one
inline int32_t mh_requant_fixed(int32_t acc, const RequantFixed &q) {
  return q.mult < 0 ? (acc >> (8 * (-1 - q.mult))) & 255 : 1;
}

#include "requant.inc"
namespace {
constexpr int XRES_SC_BYTES = 3072;
inline void transpose_16x16_bytes(v4i (&)[16]) {}   // (k-major X: not run here)
inline int atomicAdd(int *p, int v) { return __atomic_fetch_add(p, v, __ATOMIC_RELAXED); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
inline uint32_t emu_alignbyte(uint32_t hi, uint32_t lo, uint32_t by) {
  return (uint32_t)((((uint64_t)hi << 32) | lo) >> (8 * (by & 3)));
}
#define __builtin_amdgcn_alignbyte emu_alignbyte
inline uint32_t __umul24(uint32_t a, uint32_t b) { return (a & 0xffffff) * (b & 0xffffff); }
inline int __mul24(int a, int b) { return (int)((uint32_t)(a << 8 >> 8) * (uint32_t)(b << 8 >> 8)); }
namespace mhv { enum { PLANES_FORMS = 4 }; }
inline size_t mh_align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }
template <int N, bool LDS = false> inline void wait_vmcnt() {}
// global -> LDS transfer: lane l's 16 bytes land at lds_wave_base + 16 l
inline void dma_16B(const uint8_t *g, uint8_t *lds_wave_base) {
  memcpy(lds_wave_base + 16 * (threadIdx.x & 63), g, 16);
}
// ... addressed as base (the same for the wavefront) + lane offset + another offset
struct mh_rsrc { const uint8_t *base; };
inline mh_rsrc dma_rsrc(const uint8_t *base) { return mh_rsrc{base}; }
inline void dma_16B(mh_rsrc rs, uint32_t lane_off, uint32_t uniform_off, uint8_t *lds_wave_base) {
  memcpy(lds_wave_base + 16 * (threadIdx.x & 63), rs.base + lane_off + uniform_off, 16);
}
constexpr int SLAB = 64;
#include "pieces.inc"
#include "kernels.inc"
#include "conv_planes.inc"
#include "conv_staged.inc"
}  // namespace

// ---- what the fp32 kernels' text needs ---------------------------------------------------------------
namespace f32 {
typedef float v16f __attribute__((ext_vector_type(16)));
enum { MACE_HIP_ACT_NOOP, MACE_HIP_ACT_RELU, MACE_HIP_ACT_RELUX };
inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
inline float __shfl_xor(float v, int m, int n) { return __uint_as_float((uint32_t)::__shfl_xor((int)__float_as_uint(v), m, n)); }
int g_any;
inline int __syncthreads_or(int v) {
  __syncthreads();
  g_any = 0;
  __syncthreads();
  if (v) __atomic_store_n(&g_any, 1, __ATOMIC_RELAXED);
  __syncthreads();
  return g_any;
}
inline uint32_t emu_bf16(float f) {   // to nearest even
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 64;
  return (u + 0x7fff + ((u >> 16) & 1)) >> 16;
}
inline uint32_t emu_bf16_pair(float x, float y) { return emu_bf16(x) | (emu_bf16(y) << 16); }
// lane l supplies row l % 32 of each operand, depths [DEPTHS (l / 32), + DEPTHS); results as emu_mfma's
template <int DEPTHS>
inline v16f emu_mfma_f32(const float *a, const float *b, v16f c) {
  static float sa[8][64][8], sb[8][64][8];
  Wave &w = wave_of_thread();
  const int l = lane_of_thread(), wave = threadIdx.x >> 6;
  for (int k = 0; k < DEPTHS; ++k) { sa[wave][l][k] = a[k]; sb[wave][l][k] = b[k]; }
  w.bar.arrive_and_wait();
  for (int r = 0; r < 16; ++r) {
    const int x = 8 * (r / 4) + 4 * (l / 32) + r % 4;
    double s = c[r];
    for (int h = 0; h < 2; ++h)
      for (int k = 0; k < DEPTHS; ++k) s += (double)sa[wave][x + 32 * h][k] * sb[wave][(l & 31) + 32 * h][k];
    c[r] = (float)s;
  }
  w.bar.arrive_and_wait();
  return c;
}
template <typename V>
inline v16f emu_mfma_bf16(V a, V b, v16f c, int, int, int) {
  uint16_t ua[8], ub[8];
  memcpy(ua, &a, 16);
  memcpy(ub, &b, 16);
  float fa[8], fb[8];
  for (int k = 0; k < 8; ++k) { fa[k] = __uint_as_float((uint32_t)ua[k] << 16); fb[k] = __uint_as_float((uint32_t)ub[k] << 16); }
  return emu_mfma_f32<8>(fa, fb, c);
}
inline v16f emu_mfma_2f32(float a, float b, v16f c, int, int, int) { return emu_mfma_f32<1>(&a, &b, c); }
inline uint64_t emu_ballot(bool v) {
  Wave &w = wave_of_thread();
  w.w[lane_of_thread()][0] = v;
  w.bar.arrive_and_wait();
  uint64_t r = 0;
  for (int l = 0; l < 64; ++l) r |= (uint64_t)(w.w[l][0] != 0) << l;
  w.bar.arrive_and_wait();
  return r;
}
#define __builtin_amdgcn_ballot_w64 emu_ballot
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16 emu_mfma_bf16
#define __builtin_amdgcn_mfma_f32_32x32x2f32 emu_mfma_2f32
#include "f32.inc"
}  // namespace f32

// all workgroups of a grid, one after the other, on as many host threads as a workgroup has
static void run_grid(dim3 grid, const std::function<void()> &body, int threads = 256) {
  gridDim = grid;
  blockDim = dim3(threads);
  std::barrier<> bar(threads);
  g_block.bar = &bar;
  std::vector<std::thread> th;
  for (int t = 0; t < threads; ++t)
    th.emplace_back([&, t] {
      threadIdx = dim3(t, 0, 0);
      for (unsigned z = 0; z < grid.z; ++z)
        for (unsigned y = 0; y < grid.y; ++y)
          for (unsigned x = 0; x < grid.x; ++x) {
            blockIdx = dim3(x, y, z);
            body();
            g_block.bar->arrive_and_wait();
          }
    });
  for (auto &t : th) t.join();
}

static int g_failures = 0, g_cases = 0;
#define EXPECT(cond, ...)                                  \
  do {                                                     \
    if (!(cond)) {                                         \
      if (++g_failures <= 20) { printf("FAILED: " __VA_ARGS__); printf("\n"); } \
    }                                                      \
  } while (0)

static uint32_t g_seed = 12345;
static uint8_t rnd() { g_seed = g_seed * 1664525u + 1013904223u; return (uint8_t)(g_seed >> 24); }

// ---- one GEMM problem: OUT[y][x] = sum_k (X(x,k) - 128)(Y(y,k) - 128) + corrections --------------
// An operand is k-contiguous (row pitch ld >= k, the last row ending at its k-th byte: nothing
// readable behind it) or k-major ([k][n], n contiguous); X may be stored already shifted to int8.
struct Problem {
  int xn, yn, k;
  int64_t ldx, ldy;
  bool xt, yt, xf;
  int64_t xbytes, ybytes;
  uint8_t *X, *Y;
  int32_t *sumx, *sumy, *bias;
  GemmParams p{};
  int xat(int x, int c) const { return (int)((xt ? X[(int64_t)c * ldx + x] : X[(int64_t)x * ldx + c]) ^ (xf ? 0x80 : 0)) - 128; }
  int yat(int y, int c) const { return (int)(yt ? Y[(int64_t)c * ldy + y] : Y[(int64_t)y * ldy + c]) - 128; }
  Problem(int xn_, int yn_, int k_, int64_t ldx_, int64_t ldy_, bool xt_ = false, bool yt_ = false, bool xf_ = false)
      : xn(xn_), yn(yn_), k(k_), ldx(ldx_), ldy(ldy_), xt(xt_), yt(yt_), xf(xf_) {
    xbytes = xt ? (int64_t)(k - 1) * ldx + xn : (int64_t)(xn - 1) * ldx + k;
    ybytes = yt ? (int64_t)(k - 1) * ldy + yn : (int64_t)(yn - 1) * ldy + k;
    X = new uint8_t[xbytes];
    Y = new uint8_t[ybytes];
    for (int64_t i = 0; i < xbytes; ++i) X[i] = rnd();
    for (int64_t i = 0; i < ybytes; ++i) Y[i] = rnd();
    sumx = new int32_t[xn];
    sumy = new int32_t[yn];
    bias = new int32_t[xn];
    for (int x = 0; x < xn; ++x) {
      int s = 0;
      for (int c = 0; c < k; ++c) s += xat(x, c);
      sumx[x] = s;
      bias[x] = (int)rnd() * 37 - 4000;
    }
    for (int y = 0; y < yn; ++y) {
      int s = 0;
      for (int c = 0; c < k; ++c) s += yat(y, c);
      sumy[y] = s;
    }
    p.X = X; p.ldx = ldx; p.Y = Y; p.ldy = ldy;
    p.XN = xn; p.YN = yn; p.K = k;
    p.corrX = sumx; p.corrY = sumy;
    p.ldo = xn; p.obs = (int64_t)xn * yn;
    p.rq = RequantFixed{1 << 30, 8, 255, 127, -128, 127, 128};
    p.xcoef = -3; p.xadd = 11; p.xbias = bias;
    p.ycoef = 5; p.yadd = -7; p.ybias = nullptr;
  }
  ~Problem() {
    delete[] X; delete[] Y; delete[] sumx; delete[] sumy; delete[] bias;
  }
  int32_t expected(int x, int y) const {
    int64_t acc = 0;
    for (int c = 0; c < k; ++c) acc += xat(x, c) * yat(y, c);
    return (int32_t)((uint32_t)acc + (uint32_t)p.xcoef * (uint32_t)sumx[x] + (uint32_t)p.xadd + (uint32_t)bias[x] +
                     (uint32_t)p.ycoef * (uint32_t)sumy[y] + (uint32_t)p.yadd);
  }
  // runs `launch` once for an int32 and once for a uint8 result
  template <typename F32, typename F8>
  void check(const char *what, F32 launch32, F8 launch8) {
    ++g_cases;
    {
      int32_t *out = new int32_t[(int64_t)xn * yn];
      for (int64_t i = 0; i < (int64_t)xn * yn; ++i) out[i] = 0x5EEDBEEF;
      p.out = out;
      launch32(p);
      int64_t bad = 0;
      for (int y = 0; y < yn; ++y)
        for (int x = 0; x < xn; ++x) bad += out[(int64_t)y * xn + x] != expected(x, y);
      EXPECT(bad == 0, "%s XN %d YN %d K %d: %lld int32 results differ", what, xn, yn, k, (long long)bad);
      delete[] out;
    }
    {
      uint8_t *out = new uint8_t[(int64_t)xn * yn];
      memset(out, 0xEE, (int64_t)xn * yn);
      p.out = out;
      launch8(p);
      int64_t untouched = 0;
      for (int64_t i = 0; i < (int64_t)xn * yn; ++i) untouched += out[i] == 0xEE;
      EXPECT(untouched == 0, "%s XN %d YN %d K %d: %lld uint8 results not written", what, xn, yn, k,
             (long long)untouched);
      delete[] out;
    }
  }
};

// the ring kernel: slabs of KB bytes of k moved into LDS by transfers; X k-contiguous, k-major (XT)
// or repacked already shifted (XF); the panels' sums taken by the kernel or handed in
template <int WX, int WY, int FX, int FY, int STAGES, int KB, bool SUMY, bool XT = false, bool XF = false,
          bool SUMX = false>
static void ring_case(int xn, int yn, int k) {
  Problem pr(xn, yn, k, XT ? xn : k, k, XT, false, XF);
  constexpr int TX = WX * FX * 32, TY = WY * FY * 32;
  pr.p.tiles_x = (xn + TX - 1) / TX;
  pr.p.tiles_y = (yn + TY - 1) / TY;
  pr.p.sum_y = SUMY;
  const dim3 grid(pr.p.tiles_x * pr.p.tiles_y, 1, 1);
  char what[96];
  snprintf(what, sizeof what, "q8_gemm_dma_kernel<%d,%d,%d,%d,STAGES=%d,KB=%d,SUMY=%d,XT=%d,XF=%d,SUMX=%d>", WX, WY,
           FX, FY, STAGES, KB, (int)SUMY, (int)XT, (int)XF, (int)SUMX);
  pr.check(what,
           [&](GemmParams &p) {
             run_grid(grid, [&] { q8_gemm_dma_kernel<WX, WY, FX, FY, STAGES, int32_t, 1, SUMY, false, KB, XT, XF, SUMX>(p); },
                      WX * WY * 64);
           },
           [&](GemmParams &p) {
             run_grid(grid, [&] { q8_gemm_dma_kernel<WX, WY, FX, FY, STAGES, uint8_t, 1, SUMY, false, KB, XT, XF, SUMX>(p); },
                      WX * WY * 64);
           });
}

// the eight-wavefront kernel: either operand k-contiguous or k-major
template <bool XT, bool YT>
static void mid_case(int xn, int yn, int k) {
  Problem pr(xn, yn, k, XT ? xn : k, YT ? yn : k, XT, YT);
  pr.p.tiles_x = (xn + 127) / 128;
  pr.p.tiles_y = (yn + 127) / 128;
  pr.p.sum_y = true;
  const dim3 grid(pr.p.tiles_x * pr.p.tiles_y, 1, 1);
  char what[64];
  snprintf(what, sizeof what, "q8_gemm_mid_kernel<STAGES=4,XT=%d,YT=%d>", (int)XT, (int)YT);
  pr.check(what,
           [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_mid_kernel<int32_t, 4, XT, YT>(p); }, 512); },
           [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_mid_kernel<uint8_t, 4, XT, YT>(p); }, 512); });
}

// the eight-wavefront kernel on operands of any row length and depth
template <bool XT, bool YT>
static void loose_case(int xn, int yn, int k) {
  Problem pr(xn, yn, k, XT ? xn : k, YT ? yn : k, XT, YT);
  pr.p.tiles_x = (xn + 127) / 128;
  pr.p.tiles_y = (yn + 127) / 128;
  pr.p.sum_y = true;
  pr.p.K = (k + 127) / 128 * 128;
  pr.p.k_real = k;
  pr.p.x_left = pr.xbytes;
  pr.p.y_left = pr.ybytes;
  const dim3 grid(pr.p.tiles_x * pr.p.tiles_y, 1, 1);
  char what[64];
  snprintf(what, sizeof what, "q8_gemm_mid_kernel<STAGES=3,XT=%d,YT=%d,LOOSE>", (int)XT, (int)YT);
  pr.check(what,
           [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_mid_kernel<int32_t, 3, XT, YT, true>(p); }, 512); },
           [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_mid_kernel<uint8_t, 3, XT, YT, true>(p); }, 512); });
}

// the slices kernel: either operand k-contiguous or k-major, of any row length
template <bool XT, bool YT, int WK>
static void slices_case(int xn, int yn, int k) {
  Problem pr(xn, yn, k, XT ? xn : k, YT ? yn : k, XT, YT);
  pr.p.tiles_x = (xn + 31) / 32;
  pr.p.tiles_y = (yn + 31) / 32;
  pr.p.x_last = pr.X + pr.xbytes - 16;
  pr.p.y_last = pr.Y + pr.ybytes - 16;
  const int wt = 8 / WK;
  const dim3 grid((pr.p.tiles_x * pr.p.tiles_y + wt - 1) / wt, 1, 1);
  char what[64];
  snprintf(what, sizeof what, "q8_gemm_slices_kernel<XT=%d,YT=%d,WK=%d>", (int)XT, (int)YT, WK);
  pr.check(what,
           [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_slices_kernel<int32_t, XT, YT, WK>(p); }, 512); },
           [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_slices_kernel<uint8_t, XT, YT, WK>(p); }, 512); });
}

template <int WX, int WY, int FX, int FY>
static void tiled_case(int xn, int yn, int k, bool sum_y) {
  // rows padded to whole 16-byte pieces, as the callers of this kernel hand them over
  const int64_t ld = (k + 15) & ~15;
  Problem pr(xn, yn, (int)ld, ld, ld);
  constexpr int TX = WX * FX * 32, TY = WY * FY * 32;
  pr.p.tiles_x = (xn + TX - 1) / TX;
  pr.p.tiles_y = (yn + TY - 1) / TY;
  pr.p.sum_y = sum_y;
  const dim3 grid(pr.p.tiles_x * pr.p.tiles_y, 1, 1);
  char what[64];
  snprintf(what, sizeof what, "q8_gemm_kernel<%d,%d,%d,%d,SUMY=%d>", WX, WY, FX, FY, (int)sum_y);
  if (sum_y)
    pr.check(what,
             [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_kernel<WX, WY, FX, FY, int32_t, true>(p); }); },
             [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_kernel<WX, WY, FX, FY, uint8_t, true>(p); }); });
  else
    pr.check(what,
             [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_kernel<WX, WY, FX, FY, int32_t, false>(p); }); },
             [&](GemmParams &p) { run_grid(grid, [&] { q8_gemm_kernel<WX, WY, FX, FY, uint8_t, false>(p); }); });
}

// the resident-tile kernel on operands as they lie (row pitch = k); TAIL: k % 64 != 0
template <int FX, int FY, bool TAIL>
static void xres_case(int xn, int yn, int k, int wgs) {
  Problem pr(xn, yn, k, k, k);
  pr.p.sum_y = true;
  const dim3 grid(wgs, (xn + 32 * FX - 1) / (32 * FX), 1);
  char what[64];
  snprintf(what, sizeof what, "q8_gemm_xres_kernel<FX=%d,FY=%d,G=64,TAIL=%d> grid %d", FX, FY, (int)TAIL, wgs);
  pr.check(what,
           [&](GemmParams &p) {
             run_grid(grid, [&] { q8_gemm_xres_kernel<FX, FY, 64, int32_t, 2, false, false, TAIL>(p); });
           },
           [&](GemmParams &p) {
             run_grid(grid, [&] { q8_gemm_xres_kernel<FX, FY, 64, uint8_t, 2, false, false, TAIL>(p); });
           });
}

// ... on a batch of small products (per-batch operands): every (batch, tile) is computed exactly once
// whatever order the kernel walks them in
static void mid_batched_case(int batch, int xn, int yn, int k) {
  ++g_cases;
  std::vector<uint8_t> X((int64_t)batch * xn * k), Y((int64_t)batch * yn * k);
  for (auto &v : X) v = rnd();
  for (auto &v : Y) v = rnd();
  std::vector<int32_t> bias(xn), out((int64_t)batch * xn * yn, 0x5EEDBEEF);
  for (auto &v : bias) v = (int)rnd() * 37 - 4000;
  GemmParams p{};
  p.X = X.data(); p.ldx = k; p.xbs = (int64_t)xn * k;
  p.Y = Y.data(); p.ldy = k; p.ybs = (int64_t)yn * k;
  p.XN = xn; p.YN = yn; p.K = k;
  p.out = out.data(); p.ldo = xn; p.obs = (int64_t)xn * yn;
  p.xcoef = -3; p.xadd = 11; p.xbias = bias.data();
  p.ycoef = 5; p.yadd = -7;
  p.sum_y = true;
  p.tiles_x = (xn + 127) / 128;
  p.tiles_y = (yn + 127) / 128;
  run_grid(dim3(p.tiles_x * p.tiles_y, 1, batch), [&] { q8_gemm_mid_kernel<int32_t, 4, false, false>(p); }, 512);
  int64_t bad = 0;
  for (int b = 0; b < batch; ++b)
    for (int y = 0; y < yn; ++y)
      for (int x = 0; x < xn; ++x) {
        const uint8_t *xr = &X[((int64_t)b * xn + x) * k], *yr = &Y[((int64_t)b * yn + y) * k];
        int64_t acc = 0, sx = 0, sy = 0;
        for (int c = 0; c < k; ++c) {
          acc += ((int)xr[c] - 128) * ((int)yr[c] - 128);
          sx += (int)xr[c] - 128;
          sy += (int)yr[c] - 128;
        }
        const int32_t want = (int32_t)((uint32_t)acc + (uint32_t)p.xcoef * (uint32_t)sx + (uint32_t)p.xadd +
                                       (uint32_t)bias[x] + (uint32_t)p.ycoef * (uint32_t)sy + (uint32_t)p.yadd);
        bad += out[((int64_t)b * yn + y) * xn + x] != want;
      }
  EXPECT(bad == 0, "q8_gemm_mid_kernel batch %d XN %d YN %d K %d: %lld int32 results differ", batch, xn, yn, k,
         (long long)bad);
}

// The one-launch kernel: either operand k-contiguous ([n][k]) or k-major ([k][n]), rows of whole
// aligned 16-byte pieces or not (then read in 4-byte groups where everything is a multiple of 4,
// else byte by byte), or Y gathered from the NHWC input of a convolution.
struct Conv { int in_h, in_w, cin, k, stride, pad, out_h, out_w, zp; };
template <bool XT, bool YT>
static void small_case(int xn, int yn, int k, const Conv *cv = nullptr) {
  ++g_cases;
  const int64_t ldx = XT ? xn : k, ldy = cv ? 0 : (YT ? yn : k);
  const int64_t xbytes = XT ? (int64_t)k * xn : (int64_t)xn * k;
  const int64_t ybytes = cv ? (int64_t)(yn / (cv->out_h * cv->out_w)) * cv->in_h * cv->in_w * cv->cin
                            : (YT ? (int64_t)k * yn : (int64_t)yn * k);
  uint8_t *X = new uint8_t[xbytes], *Y = new uint8_t[ybytes];
  for (int64_t i = 0; i < xbytes; ++i) X[i] = rnd();
  for (int64_t i = 0; i < ybytes; ++i) Y[i] = rnd();
  auto xat = [&](int x, int c) { return (int)(XT ? X[(int64_t)c * xn + x] : X[(int64_t)x * k + c]) - 128; };
  auto yat = [&](int y, int c) {
    if (!cv) return (int)(YT ? Y[(int64_t)c * yn + y] : Y[(int64_t)y * k + c]) - 128;
    const int ow = y % cv->out_w, t = y / cv->out_w, oh = t % cv->out_h, img = t / cv->out_h;
    const int tap = c / cv->cin, ch = c % cv->cin, kh = tap / cv->k, kw = tap % cv->k;
    const int ih = oh * cv->stride - cv->pad + kh, iw = ow * cv->stride - cv->pad + kw;
    if (ih < 0 || ih >= cv->in_h || iw < 0 || iw >= cv->in_w) return cv->zp - 128;
    return (int)Y[(((int64_t)img * cv->in_h + ih) * cv->in_w + iw) * cv->cin + ch] - 128;
  };
  std::vector<int32_t> bias(xn), sumx(xn), sumy(yn);
  for (int x = 0; x < xn; ++x) {
    bias[x] = (int)rnd() * 91 - 9000;
    for (int c = 0; c < k; ++c) sumx[x] += xat(x, c);
  }
  for (int y = 0; y < yn; ++y)
    for (int c = 0; c < k; ++c) sumy[y] += yat(y, c);
  GemmParams p{};
  p.X = X; p.ldx = ldx; p.Y = Y; p.ldy = ldy;
  p.XN = xn; p.YN = yn; p.K = k;
  p.ldo = xn; p.obs = (int64_t)xn * yn;
  p.rq = RequantFixed{1 << 30, 8, 255, 127, -128, 127, 128};
  p.xcoef = -3; p.xadd = 11; p.xbias = bias.data();
  p.ycoef = 5; p.yadd = -7; p.ybias = nullptr;
  p.sum_y = true;
  p.tiles_x = (xn + 63) / 64;
  p.tiles_y = (yn + 63) / 64;
  // the host's rules (Q8Call::small_problem): whole aligned pieces, else 4-byte groups, else bytes
  auto vec = [&](bool t, int n) { return (t ? n : k) % 16 == 0; };
  auto dwords = [&](bool t, int n) { return (t ? n : k) % 4 == 0; };
  p.x_bytewise = !vec(XT, xn);
  p.x_dword = p.x_bytewise && dwords(XT, xn);
  if (cv) {
    p.conv = true;
    p.cv_in_h = cv->in_h; p.cv_in_w = cv->in_w; p.cv_cin = cv->cin; p.cv_kw = cv->k;
    p.cv_sh = p.cv_sw = cv->stride; p.cv_pt = p.cv_pl = cv->pad; p.cv_oh = cv->out_h; p.cv_ow = cv->out_w;
    p.cv_zp4 = (uint32_t)cv->zp * 0x01010101u;
    p.y_bytewise = cv->cin % 16 != 0;
    p.y_dword = p.y_bytewise && cv->cin % 4 == 0;
  } else {
    p.y_bytewise = !vec(YT, yn);
    p.y_dword = p.y_bytewise && dwords(YT, yn);
  }
  const bool bw = p.x_bytewise || p.y_bytewise;
  const dim3 grid(p.tiles_x * p.tiles_y, 1, 1);
  {
    std::vector<int32_t> out((int64_t)xn * yn, 0x5EEDBEEF);
    p.out = out.data();
    if (bw) run_grid(grid, [&] { q8_gemm_fused_small_kernel<int32_t, XT, YT, true>(p); });
    else run_grid(grid, [&] { q8_gemm_fused_small_kernel<int32_t, XT, YT, false>(p); });
    int64_t bad = 0;
    for (int y = 0; y < yn; ++y)
      for (int x = 0; x < xn; ++x) {
        int64_t acc = 0;
        for (int c = 0; c < k; ++c) acc += xat(x, c) * yat(y, c);
        const int32_t want = (int32_t)((uint32_t)acc + (uint32_t)p.xcoef * (uint32_t)sumx[x] + (uint32_t)p.xadd +
                                       (uint32_t)bias[x] + (uint32_t)p.ycoef * (uint32_t)sumy[y] + (uint32_t)p.yadd);
        bad += out[(int64_t)y * xn + x] != want;
      }
    EXPECT(bad == 0, "fused_small<XT=%d,YT=%d,BW=%d>%s XN %d YN %d K %d: %lld int32 results differ", (int)XT,
           (int)YT, (int)bw, cv ? " conv" : "", xn, yn, k, (long long)bad);
  }
  {
    std::vector<uint8_t> out((int64_t)xn * yn, 0xEE);
    p.out = out.data();
    if (bw) run_grid(grid, [&] { q8_gemm_fused_small_kernel<uint8_t, XT, YT, true>(p); });
    else run_grid(grid, [&] { q8_gemm_fused_small_kernel<uint8_t, XT, YT, false>(p); });
    int64_t untouched = 0;
    for (uint8_t v : out) untouched += v == 0xEE;
    EXPECT(untouched == 0, "fused_small<XT=%d,YT=%d,BW=%d> XN %d YN %d K %d: %lld uint8 results not written",
           (int)XT, (int)YT, (int)bw, xn, yn, k, (long long)untouched);
  }
  delete[] X;
  delete[] Y;
}
static void small_conv_case(int n, int hw, int cin, int cout, int k, int stride, int pad) {
  const int out = (hw + 2 * pad - k) / stride + 1;
  const Conv cv{hw, hw, cin, k, stride, pad, out, out, 77};
  small_case<false, false>(cout, n * out * out, k * k * cin, &cv);
}

// both operands of a call copied into padded panels by one launch: nb batches of n rows of k bytes
// next to nb batches of a k-major [k][nt] operand, with its row sums, as read or shifted
static void pack_case(int nb, int n, int nt, int k, bool flip) {
  ++g_cases;
  const int kp = (k + 63) & ~63;
  const int64_t rows = (int64_t)nb * n, cols = (int64_t)nb * nt;
  uint8_t *src = new uint8_t[rows * k], *dst = new uint8_t[rows * kp];
  uint8_t *tsrc = new uint8_t[cols * k], *tdst = new uint8_t[cols * kp];
  int32_t *sums = new int32_t[cols]();
  for (int64_t i = 0; i < rows * k; ++i) src[i] = rnd();
  for (int64_t i = 0; i < cols * k; ++i) tsrc[i] = rnd();
  memset(dst, 0xEE, rows * kp);
  memset(tdst, 0xEE, cols * kp);
  RepackJob a{}, b{};
  a.src = src; a.dst = dst; a.rows = rows; a.n = n; a.k = k; a.kp = kp;
  a.blocks = (rows * (kp / 16) + REPACK_PIECES - 1) / REPACK_PIECES;
  b.src = tsrc; b.dst = tdst; b.n = nt; b.k = k; b.kp = kp; b.sums = sums;
  b.flip = flip ? 0x80808080u : 0u;
  b.tiles_n = (nt + 127) / 128; b.tiles_k = (kp + 127) / 128;
  b.blocks = (int64_t)b.tiles_n * b.tiles_k * nb;
  // (a grid with more workgroups than there is work, in two rows)
  const dim3 grid((unsigned)((a.blocks + b.blocks) / 2 + 1), 2, 1);
  run_grid(grid, [&] { q8_repack_kernel(a, b); });
  int64_t bad = 0;
  for (int64_t r = 0; r < rows; ++r)
    for (int c = 0; c < kp; ++c) bad += dst[r * kp + c] != (c < k ? src[r * k + c] : 0x80);
  for (int64_t r = 0; r < cols; ++r) {
    int s = 0;
    for (int c = 0; c < kp; ++c) {
      const int v = c < k ? tsrc[(r / nt * k + c) * nt + r % nt] : 0x80;
      s += v - 128;
      bad += tdst[r * kp + c] != (uint8_t)(flip ? v ^ 0x80 : v);
    }
    bad += s != sums[r];
  }
  EXPECT(bad == 0, "repack nb %d n %d nt %d k %d: %lld bytes differ", nb, n, nt, k, (long long)bad);
  delete[] src;
  delete[] dst;
  delete[] tsrc;
  delete[] tdst;
  delete[] sums;
}

// the convolution on padded planes, both launches: geometry, LDS and scratch as the host code lays them out;
// every byte of the accumulators compared with sums formed directly from the operands
template <int FX, int FY, int WX, int WY, int WK, int SPR = 0>
static void planes_case(int n, int in_h, int in_w, int cin, int cout, int k_h, int k_w, int sh, int sw, int pt, int pl,
                        int out_h, int out_w, int budget, int buffers, int groups) {
  ++g_cases;
  const PlaneForm form{FX, FY, WX, WY, WK};
  const PlaneShape s{n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, pt, pl, out_h, out_w};
  EXPECT(plane_fits(s), "planes: the shape does not fit");
  const int64_t in_bytes = (int64_t)n * in_h * in_w * cin, depth = (int64_t)k_h * k_w * cin, columns = (int64_t)n * out_h * out_w;
  uint8_t *in = new uint8_t[in_bytes], *filter = new uint8_t[cout * depth];
  int32_t *bias = new int32_t[cout];
  for (int64_t i = 0; i < in_bytes; ++i) in[i] = rnd();
  for (int64_t i = 0; i < cout * depth; ++i) filter[i] = rnd();
  for (int i = 0; i < cout; ++i) bias[i] = (int)rnd() * 91 - 9000;
  const int zi = 77, zf = 140;
  std::vector<int32_t> want(columns * cout);
  for (int64_t px = 0; px < columns; ++px) {
    const int ow = px % out_w, oh = px / out_w % out_h, img = px / out_w / out_h;
    for (int c = 0; c < cout; ++c) {
      int64_t acc = bias[c];
      for (int kh = 0; kh < k_h; ++kh)
        for (int kw = 0; kw < k_w; ++kw) {
          const int ih = oh * sh - pt + kh, iw = ow * sw - pl + kw;
          if (ih < 0 || ih >= in_h || iw < 0 || iw >= in_w) continue;   // the zero point
          for (int ch = 0; ch < cin; ++ch)
            acc += ((int)in[(((int64_t)img * in_h + ih) * in_w + iw) * cin + ch] - zi) *
                   ((int)filter[c * depth + (kh * k_w + kw) * cin + ch] - zf);
        }
      want[px * cout + c] = (int32_t)acc;
    }
  }
  ConvPlaneParams p{};
  const PlanePlan plan = plane_plan(form, s, budget, buffers, &p);
  EXPECT(SPR == 0 || (SPR == p.spr && p.pieces == 2), "planes: %d k steps of a filter row", p.spr);
  p.in = in; p.filter = filter; p.bias = bias;
  p.xcoef = -(zi - 128); p.ycoef = -(zf - 128); p.yadd = (int)depth * (zi - 128) * (zf - 128);
  p.zpf4 = (uint32_t)(zi ^ 0x80) * 0x01010101u;
  p.planes = new uint8_t[plan.planes_bytes]; p.packed = new uint8_t[plan.packed_bytes];
  p.psum = (int32_t *)new uint8_t[plan.psum_bytes]; p.cx = (int32_t *)new uint8_t[plan.cx_bytes];
  memset(p.planes, 0xC3, plan.planes_bytes);
  p.span = p.tiles_p / groups; p.span_more = p.tiles_p % groups;
  const int wgs = groups * p.tiles_x;
  EXPECT(plan.fits && plan.lds <= (int64_t)sizeof(g_block.lds), "planes: %lld bytes of LDS", (long long)plan.lds);
  run_grid(dim3(plan.pack_blocks), [&] { q8_conv_planes_pack_kernel(p); });
  for (int byte = 0; byte < 4; ++byte) {
    p.rq = RequantFixed{-1 - byte, 0, 0, 0, 0, 255, 0};
    uint8_t *out = new uint8_t[columns * cout];
    memset(g_block.lds, 0xA5, sizeof(g_block.lds));
    p.out = out;
    run_grid(dim3(wgs), [&] { q8_conv_planes_kernel<FX, FY, WX, WY, WK, SPR, 1>(p); }, plan.threads);
    int64_t bad = 0;
    for (int64_t i = 0; i < columns * cout; ++i) bad += out[i] != (uint8_t)(want[i] >> (8 * byte));
    EXPECT(bad == 0, "planes<%d,%d,%d,%d,%d> n %d %dx%dx%d>%d k%dx%d s%dx%d stages of %d slabs, wgs %d: byte %d of %lld results differs",
           FX, FY, WX, WY, WK, n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, p.stage_slabs, wgs, byte, (long long)bad);
    for (int64_t i = plan.lds; i < (int64_t)sizeof(g_block.lds); ++i)
      if (g_block.lds[i] != 0xA5) { EXPECT(false, "planes: LDS byte %lld of %lld written", (long long)i, (long long)plan.lds); break; }
    delete[] out;
  }
  // a filter whose packed bytes and sums are kept: the first launch leaves the sums, a later one takes them
  p.wsums = new int32_t[p.channels];
  run_grid(dim3(plan.pack_blocks), [&] { q8_conv_planes_pack_kernel(p); });
  std::vector<int32_t> cx(p.cx, p.cx + p.channels);
  std::vector<uint8_t> packed(p.packed, p.packed + plan.packed_bytes);
  memset(p.cx, 0x5A, p.channels * 4);
  p.kept = true;
  run_grid(dim3(p.pixel_blocks + (p.channels + 255) / 256), [&] { q8_conv_planes_pack_kernel(p); });
  EXPECT(std::equal(cx.begin(), cx.end(), p.cx) && std::equal(packed.begin(), packed.end(), p.packed), "planes: a kept filter's corrections differ");
  delete[] p.wsums;
  delete[] in;
  delete[] filter;
  delete[] bias;
  delete[] p.planes;
  delete[] p.packed;
  delete[] (uint8_t *)p.psum;
  delete[] (uint8_t *)p.cx;
}

// ---- fp32: results against binary64, to the sum of the products' sizes times their number --------------
static float rnd_f32() { return ((int)rnd() * 256 + rnd() - 32768) / 8192.0f; }
static void check_f32(const char *what, const float *got, const std::vector<double> &want, const std::vector<double> &size, int k) {
  int64_t bad = 0;
  for (size_t i = 0; i < want.size(); ++i)
    bad += std::isfinite(want[i]) ? !(std::fabs(got[i] - want[i]) <= (k + 16) * std::ldexp(size[i], -24)) : std::isfinite(got[i]);
  EXPECT(bad == 0, "%s k %d: %lld of %zu results differ", what, k, (long long)bad, want.size());
}

// the fp32 slices kernel: operands along the depth (LK, RK) or along their rows and columns, images side by side
// (flat: columns of each), `inf`: one operand element that no sum can take
template <bool LK, bool RK, int FN, int WK>
static void f32_slices_case(int batch, int m, int n, int k, int flat = 0, bool inf = false) {
  ++g_cases;
  const int images = flat ? batch : 1, cols = flat ? flat * batch : n, gz = flat ? 1 : batch;
  const int per = flat ? flat : n;   // columns of a right-hand matrix in memory
  const int lb = flat ? 1 : batch;
  float *A = new float[(int64_t)lb * m * k], *B = new float[(int64_t)batch * k * per], *out = new float[(int64_t)batch * m * per];
  float *bias = new float[m];
  for (int64_t i = 0; i < (int64_t)lb * m * k; ++i) A[i] = rnd_f32();
  for (int64_t i = 0; i < (int64_t)batch * k * per; ++i) B[i] = rnd_f32();
  for (int i = 0; i < m; ++i) bias[i] = rnd_f32();
  if (inf) A[(int64_t)lb * m * k - 1] = INFINITY;
  std::vector<double> want((int64_t)batch * m * per), size(want.size());
  for (int b = 0; b < batch; ++b)
    for (int i = 0; i < m; ++i)
      for (int j = 0; j < per; ++j) {
        double s = bias[i], t = std::fabs(bias[i]);
        for (int c = 0; c < k; ++c) {
          const int64_t ao = (int64_t)(flat ? 0 : b) * m * k + (LK ? (int64_t)i * k + c : (int64_t)c * m + i);
          const int64_t bo = (int64_t)b * k * per + (RK ? (int64_t)j * k + c : (int64_t)c * per + j);
          s += (double)A[ao] * B[bo];
          t += std::fabs((double)A[ao] * B[bo]);
        }
        want[((int64_t)b * m + i) * per + j] = s;
        size[((int64_t)b * m + i) * per + j] = t;
      }
  f32::F32GemmParams p{};
  p.lhs = A; p.rhs = B; p.out = out;
  p.lrs = LK ? k : 1; p.lcs = LK ? 1 : m;
  p.rrs = RK ? 1 : per; p.rcs = RK ? k : 1;
  p.ors = per; p.ocs = 1;
  p.lbs = flat ? 0 : (int64_t)m * k; p.rbs = (int64_t)k * per; p.obs = (int64_t)m * per;
  p.M = m; p.N = cols; p.K = k; p.flat = images > 1 ? flat : 0; p.bias_row = bias;
  p.tiles_m = (m + 31) / 32;
  const int tiles = p.tiles_m * ((cols + 32 * FN - 1) / (32 * FN)), wt = 8 / WK;
  run_grid(dim3((tiles + wt - 1) / wt, 1, gz), [&] { f32::f32_gemm_slices_kernel<LK, RK, FN, WK>(p); }, 512);
  char what[96];
  snprintf(what, sizeof what, "f32_gemm_slices_kernel<%d,%d,%d,%d> batch %d m %d n %d", (int)LK, (int)RK, FN, WK, batch, m, n);
  check_f32(what, out, want, size, k);
  delete[] A; delete[] B; delete[] out; delete[] bias;
}

// A right-hand matrix of images side by side (flat: columns of each) or one: operands of exactly their size, `off` floats
// behind a multiple of 16 bytes, and what a sum of each result and of its products' sizes is
struct F32Problem {
  int m, n, k, flat, images, off;
  bool lk, rk;
  float *a0, *b0, *bias, *out;
  std::vector<double> want, size;
  f32::F32GemmParams p{};
  F32Problem(int images_, int m_, int n_, int k_, bool lk_, bool rk_, int off_, bool inf)
      : m(m_), n(n_), k(k_), flat(images_ > 1 ? n_ : 0), images(images_), off(off_), lk(lk_), rk(rk_) {
    const int64_t as = (int64_t)m * k, bs = (int64_t)images * k * n;
    a0 = new float[as + off]; b0 = new float[bs + off]; bias = new float[m]; out = new float[(int64_t)images * m * n];
    for (int64_t i = 0; i < as + off; ++i) a0[i] = rnd_f32();
    for (int64_t i = 0; i < bs + off; ++i) b0[i] = rnd_f32();
    for (int i = 0; i < m; ++i) bias[i] = rnd_f32();
    float *const a = a0 + off, *const b = b0 + off;
    if (inf) a[as - 1] = INFINITY;
    want.resize((int64_t)images * m * n);
    size.resize(want.size());
    for (int g = 0; g < images; ++g)
      for (int i = 0; i < m; ++i)
        for (int j = 0; j < n; ++j) {
          double s = bias[i], t = std::fabs(bias[i]);
          for (int c = 0; c < k; ++c) {
            const double v = (double)a[lk ? (int64_t)i * k + c : (int64_t)c * m + i] *
                             b[(int64_t)g * k * n + (rk ? (int64_t)j * k + c : (int64_t)c * n + j)];
            s += v;
            t += std::fabs(v);
          }
          want[((int64_t)g * m + i) * n + j] = s;
          size[((int64_t)g * m + i) * n + j] = t;
        }
    p.lhs = a; p.rhs = b; p.out = out;
    p.lrs = lk ? k : 1; p.lcs = lk ? 1 : m;
    p.rrs = rk ? 1 : n; p.rcs = rk ? k : 1;
    p.ors = n; p.ocs = 1;
    p.rbs = (int64_t)k * n; p.obs = (int64_t)m * n;
    p.M = m; p.N = images * n; p.K = k; p.flat = flat; p.bias_row = bias;
  }
  ~F32Problem() { delete[] a0; delete[] b0; delete[] bias; delete[] out; }
};

// the tile kernels: TMT x 128 tiles by four wavefronts (SPLIT = 1) or eight, loads checked (GUARD) or not; `parts` above 0:
// k tiles of 16 of a part of the depth, whose sums are added up here
template <bool LK, bool RK, int SPLIT, bool GUARD, int TMT>
static void f32_tile_case(int images, int m, int n, int k, int off = 0, int parts = 0, bool inf = false) {
  ++g_cases;
  F32Problem pr(images, m, n, k, LK, RK, off, inf);
  f32::F32GemmParams &p = pr.p;
  p.tiles_m = (m + TMT - 1) / TMT;
  const int ny = parts ? ((k + 15) / 16 + parts - 1) / parts : 1;
  const int64_t total = (int64_t)images * m * n;
  float *part = new float[parts ? ny * total : 1];
  if (parts) { p.part = part; p.kt_split = parts; p.part_stride = total; }
  run_grid(dim3(p.tiles_m * ((p.N + 127) / 128), ny), [&] {
    if constexpr (GUARD) f32::f32_gemm_kernel<LK, RK, SPLIT, TMT>(p);
    else f32::f32_gemm_vec_kernel<LK, RK, SPLIT, TMT>(p);
  }, 256 * SPLIT);
  if (parts)
    for (int64_t i = 0; i < total; ++i) {
      pr.out[i] = pr.bias[i / n % m];
      for (int q = 0; q < ny; ++q) pr.out[i] += part[q * total + i];
    }
  char what[112];
  snprintf(what, sizeof what, "f32_tile<%d,%d,SPLIT=%d,GUARD=%d,TM=%d> images %d m %d n %d off %d parts %d", (int)LK, (int)RK, SPLIT, (int)GUARD,
           TMT, images, m, n, off, parts);
  check_f32(what, pr.out, pr.want, pr.size, k);
  delete[] part;
}

// the panel kernel: 32 MI rows in LDS, D k steps of loads ahead, `groups` spans of columns
template <int MI, int D, bool GUARD>
static void f32_panel_case(int images, int m, int n, int k, int groups, bool lk = true, bool inf = false) {
  ++g_cases;
  F32Problem pr(images, m, n, k, lk, false, 0, inf);
  f32::F32GemmParams &p = pr.p;
  p.tiles_m = (m + 32 * MI - 1) / (32 * MI);
  const int64_t lds = (int64_t)((k + 15) / 16) * 3 * MI * 1024 + 128 * MI;
  memset(g_block.lds, 0xA5, sizeof(g_block.lds));
  run_grid(dim3(groups * p.tiles_m), [&] { f32::f32_gemm_panel_kernel<MI, D, GUARD>(p, groups, (p.N + 31) / 32); }, 512);
  char what[96];
  snprintf(what, sizeof what, "f32_gemm_panel_kernel<%d,%d,%d> images %d m %d n %d groups %d", MI, D, (int)GUARD, images, m, n, groups);
  check_f32(what, pr.out, pr.want, pr.size, k);
  for (int64_t i = lds; i < (int64_t)sizeof(g_block.lds); ++i)
    if (g_block.lds[i] != 0xA5) { EXPECT(false, "%s: LDS byte %lld of %lld written", what, (long long)i, (long long)lds); break; }
}

// the Gemv kernels: NB vectors a pass with one row a wavefront (R = 1) or four, rows in 2^bits slices; NB = 0: float by float
template <int NB, int R>
static void f32_gemv_case(int batch, int h, int w, bool lb, int bits) {
  ++g_cases;
  float *L = new float[(int64_t)(lb ? batch : 1) * h * w], *x = new float[(int64_t)batch * w], *bias = new float[h],
        *out = new float[(int64_t)batch * h];
  for (int64_t i = 0; i < (int64_t)(lb ? batch : 1) * h * w; ++i) L[i] = rnd_f32();
  for (int64_t i = 0; i < (int64_t)batch * w; ++i) x[i] = rnd_f32();
  for (int i = 0; i < h; ++i) bias[i] = rnd_f32();
  std::vector<double> want((int64_t)batch * h), size(want.size());
  for (int b = 0; b < batch; ++b)
    for (int i = 0; i < h; ++i) {
      double s = bias[i], t = std::fabs(bias[i]);
      for (int c = 0; c < w; ++c) {
        const double v = (double)L[((int64_t)(lb ? b : 0) * h + i) * w + c] * x[(int64_t)b * w + c];
        s += v;
        t += std::fabs(v);
      }
      want[(int64_t)b * h + i] = s;
      size[(int64_t)b * h + i] = t;
    }
  f32::F32GemvParams p{L, x, bias, out, lb ? (int64_t)h * w : 0, w, h, w, f32::MACE_HIP_ACT_NOOP, 0.f};
  char what[80];
  snprintf(what, sizeof what, "f32_gemv<NB=%d,R=%d> %d x %d x %d in %d", NB, R, batch, h, w, 1 << bits);
  if constexpr (NB == 0) {
    run_grid(dim3((h + 3) / 4, batch), [&] { f32::f32_gemv_floats_kernel(p); });
  } else {
    const int waves = (1 << bits) > 4 ? 1 << bits : 4, groups = waves >> bits, rows = groups * R;
    run_grid(dim3((h + rows - 1) / rows, (batch + NB - 1) / NB), [&] {
      if constexpr (R == 1) f32::f32_gemv_kernel<NB>(p, batch, bits, groups);
      else f32::f32_gemv_rows_kernel<NB>(p, batch, bits, groups);
    }, 64 * waves);
  }
  check_f32(what, out, want, size, w);
  delete[] L; delete[] x; delete[] bias; delete[] out;
}

template <int LPR>
static void sums_case(int n, int k) {
  ++g_cases;
  uint8_t *P = new uint8_t[(int64_t)n * k];
  int32_t *sums = new int32_t[n];
  for (int64_t i = 0; i < (int64_t)n * k; ++i) P[i] = rnd();
  const int rows_per_block = 4 * (64 / LPR);
  const dim3 grid((n + rows_per_block - 1) / rows_per_block, 1, 1);
  run_grid(grid, [&] { q8_panel_sums_kernel<LPR>(P, k, 0, n, k, sums, nullptr, 0); });
  int bad = 0;
  for (int r = 0; r < n; ++r) {
    int s = 0;
    for (int c = 0; c < k; ++c) s += (int)P[(int64_t)r * k + c] - 128;
    bad += s != sums[r];
  }
  EXPECT(bad == 0, "panel_sums<%d> n %d k %d: %d sums differ", LPR, n, k, bad);
  delete[] P;
  delete[] sums;
}

// the convolution on staged rows: the tile that the host code chooses on a device of `cu` CUs with `lds` bytes
// of LDS each, operands allocated at exactly their size, every byte of the accumulators compared
template <int FX, int WK, bool WHOLE, bool TWO = false>
static void staged_case(int n, int in_h, int in_w, int cin, int cout, int k_h, int k_w, int sh, int sw, int pt, int pl,
                        int out_h, int out_w, int cu, int lds = 160 * 1024) {
  ++g_cases;
  const StagedShape s{n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, pt, pl, out_h, out_w};
  EXPECT(staged_fits(s), "staged: the shape does not fit");
  const int64_t in_bytes = (int64_t)n * in_h * in_w * cin, depth = (int64_t)k_h * k_w * cin, columns = (int64_t)n * out_h * out_w;
  uint8_t *in = new uint8_t[in_bytes], *filter = new uint8_t[cout * depth];
  int32_t *bias = new int32_t[cout];
  for (int64_t i = 0; i < in_bytes; ++i) in[i] = rnd();
  for (int64_t i = 0; i < cout * depth; ++i) filter[i] = rnd();
  for (int i = 0; i < cout; ++i) bias[i] = (int)rnd() * 91 - 9000;
  const int zi = 77, zf = 140;
  ConvStagedParams p{};
  const StagedPlan plan = staged_plan(s, FX, cu, lds, &p);
  EXPECT(plan.groups > 0 && plan.lds <= lds && plan.fx == FX && plan.wk == WK && (TWO == (FX == 2 && plan.two)) && (cin % 16 == 0) == WHOLE,
         "staged: %lld tiles of %d pixels, FX %d WK %d, %lld bytes of LDS", (long long)plan.groups, p.tile_px, plan.fx, plan.wk,
         (long long)plan.lds);
  p.in = in; p.filter = filter; p.bias = bias;
  p.xcoef = -(zi - 128); p.ycoef = -(zf - 128); p.yadd = (int)depth * (zi - 128) * (zf - 128);
  p.zpf4 = (uint32_t)(zi ^ 0x80) * 0x01010101u;
  for (int byte = 0; byte < 3; byte += 2) {
    p.rq = RequantFixed{-1 - byte, 0, 0, 0, 0, 255, 0};
    uint8_t *out = new uint8_t[columns * cout];
    memset(g_block.lds, 0xA5, sizeof(g_block.lds));
    p.out = out;
    run_grid(dim3(plan.groups * p.tiles_x), [&] { q8_conv_staged_kernel<FX, WK, WHOLE, TWO>(p); }, 512);
    int64_t bad = 0;
    for (int64_t px = 0; px < columns; ++px) {
      const int ow = px % out_w, oh = px / out_w % out_h, img = px / out_w / out_h;
      for (int c = 0; c < cout; ++c) {
        int64_t acc = bias[c];
        for (int kh = 0; kh < k_h; ++kh)
          for (int kw = 0; kw < k_w; ++kw) {
            const int ih = oh * sh - pt + kh, iw = ow * sw - pl + kw;
            if (ih < 0 || ih >= in_h || iw < 0 || iw >= in_w) continue;   // the zero point
            for (int ch = 0; ch < cin; ++ch)
              acc += ((int)in[(((int64_t)img * in_h + ih) * in_w + iw) * cin + ch] - zi) *
                     ((int)filter[c * depth + (kh * k_w + kw) * cin + ch] - zf);
          }
        bad += out[px * cout + c] != (uint8_t)((int32_t)acc >> (8 * byte));
      }
    }
    EXPECT(bad == 0, "staged<%d,%d,%d> n %d %dx%dx%d>%d k%dx%d s%dx%d tiles of %d pixels: byte %d of %lld results differs", FX, WK,
           (int)WHOLE, n, in_h, in_w, cin, cout, k_h, k_w, sh, sw, p.tile_px, byte, (long long)bad);
    for (int64_t i = plan.lds; i < (int64_t)sizeof(g_block.lds); ++i)
      if (g_block.lds[i] != 0xA5) { EXPECT(false, "staged: LDS byte %lld of %lld written", (long long)i, (long long)plan.lds); break; }
    delete[] out;
  }
  delete[] in;
  delete[] filter;
  delete[] bias;
}

// PART (compile-time): 1 = everything but what follows, 2 = the ring and eight-wavefront kernels, 3 = the
// uint8 slices kernel and the convolution on padded planes, 4 = the fp32 kernels and the planes' tile of eight
// wavefronts, 5 = the convolution on staged rows and the fp32 panel kernel; the test builds and runs the parts side by side.
#ifndef PART
#define PART 0
#endif
int main() {
#if PART != 2 && PART != 3 && PART != 4 && PART != 5
  // the repacks of k-contiguous rows and of k-major operands: any row length
  for (int k : {1, 3, 15, 16, 17, 24, 63, 64, 65, 100, 127}) pack_case(1, 37, k, k, false);
  for (int k : {4, 8, 24, 40, 60, 64, 68, 120}) pack_case(1, 301, 130 + k, k, true);
  pack_case(3, 41, 157, 131, false);
  pack_case(2, 17, 7, 300, true);
  // row sums: rows of 16 .. 1024 bytes, row counts that leave part of a wavefront without a row
  sums_case<1>(70, 16);
  sums_case<2>(33, 32);
  sums_case<4>(144, 64);
  sums_case<8>(19, 128);
  sums_case<16>(40, 256);
  sums_case<64>(9, 1040);
  // the register-staged tiled kernel: every tile shape, whole slabs and depth tails, ragged tiles
  // in both directions, result rows of whole 16-byte pieces (the wide ragged stores) and not
  for (bool sum_y : {false, true}) {
    tiled_case<2, 2, 1, 1>(70, 130, 48, sum_y);
    tiled_case<2, 2, 1, 1>(64, 64, 64, sum_y);
    tiled_case<2, 2, 2, 2>(144, 300, 64, sum_y);
    tiled_case<2, 2, 2, 2>(131, 129, 176, sum_y);
    tiled_case<1, 4, 2, 2>(48, 600, 96, sum_y);
    tiled_case<1, 4, 2, 2>(37, 257, 16, sum_y);
    tiled_case<2, 2, 4, 4>(144, 520, 64, sum_y);
    tiled_case<2, 2, 4, 4>(300, 290, 16, sum_y);
  }
  // the one-launch kernel: both layouts of both operands; rows of whole pieces, of 4-byte groups, of
  // single bytes; ragged tiles; depths from one byte to several k tiles; gathered convolutions
  small_case<false, false>(128, 128, 256);
  small_case<false, false>(70, 130, 48);
  small_case<false, false>(33, 65, 100);
  small_case<false, false>(64, 17, 27);
  small_case<false, false>(5, 3, 1);
  small_case<false, false>(100, 90, 333);
  small_case<true, false>(128, 64, 128);
  small_case<true, false>(100, 70, 96);
  small_case<true, false>(37, 64, 50);
  small_case<false, true>(64, 112, 80);
  small_case<false, true>(48, 101, 64);
  small_case<true, true>(80, 48, 144);
  small_case<true, true>(31, 29, 67);
  small_conv_case(2, 9, 16, 24, 3, 1, 1);
  small_conv_case(1, 12, 8, 16, 3, 2, 1);
  small_conv_case(1, 10, 3, 32, 3, 2, 0);
  small_conv_case(2, 7, 5, 17, 2, 1, 1);
  small_conv_case(1, 8, 32, 64, 1, 1, 0);
  // the resident-tile kernel: 64- and 128-row tiles, 32- and 64-row blocks, more blocks than
  // wavefronts and fewer, whole groups, depth tails of whole pieces and of half a piece
  xres_case<2, 1, false>(48, 700, 64, 3);
  xres_case<2, 2, false>(64, 333, 128, 2);
  xres_case<4, 1, false>(144, 500, 192, 2);
  xres_case<4, 2, false>(200, 1000, 64, 5);
  xres_case<4, 2, true>(144, 600, 96, 2);
  xres_case<2, 1, true>(17, 900, 80, 4);
  xres_case<4, 2, true>(144, 777, 24, 3);
  xres_case<2, 2, true>(64, 290, 40, 1);
  xres_case<4, 1, true>(130, 515, 72, 2);
  xres_case<2, 1, true>(24, 4000, 120, 40);
  xres_case<4, 2, true>(128, 256, 328, 1);
#endif
#if PART != 1 && PART != 3 && PART != 4
  // the ring kernel in the tile shapes, ring depths and slab widths the dispatch uses; ragged tiles
  ring_case<2, 2, 4, 4, 2, 128, false>(300, 260, 384);
  ring_case<2, 2, 4, 4, 2, 128, true>(256, 257, 256);
  ring_case<2, 2, 4, 4, 2, 128, false, true>(304, 200, 384);           // X k-major, read in place
  ring_case<2, 2, 4, 4, 2, 128, true, true, false, true>(272, 300, 256);   // ... and summed in the kernel
  ring_case<2, 2, 4, 4, 2, 128, false, false, true>(260, 300, 384);    // X repacked already shifted
  ring_case<2, 4, 2, 1, 2, 128, true>(130, 140, 1024);
  ring_case<2, 2, 2, 2, 2, 128, false>(200, 129, 1024);
  ring_case<2, 2, 4, 4, 4, 64, true>(257, 300, 192);
  ring_case<1, 4, 2, 2, 4, 64, false>(48, 300, 256);
  ring_case<2, 2, 2, 2, 4, 64, true>(130, 200, 448);
  ring_case<2, 2, 1, 1, 4, 64, false>(70, 65, 192);
  ring_case<1, 4, 2, 2, 3, 64, true>(64, 513, 128);
  ring_case<2, 2, 2, 2, 3, 64, false>(129, 131, 128);
  // the eight-wavefront kernel: every layout of both operands, ragged tiles, the shortest depth
  mid_case<false, false>(200, 130, 512);
  mid_case<true, false>(144, 129, 640);
  mid_case<false, true>(129, 208, 512);
  mid_case<true, true>(272, 144, 512);
  mid_case<false, false>(128, 128, 128);
  // ... on rows that are not whole pieces: a slab and a byte, the fewest slabs, short k-major rows, tiles of a few columns
  loose_case<false, false>(130, 77, 257);
  loose_case<true, false>(133, 66, 391);
  loose_case<false, true>(65, 131, 263);
  loose_case<true, true>(67, 129, 300);
  loose_case<true, false>(7, 128, 640);
  mid_batched_case(8, 200, 128, 128);    // 16 workgroups: dealt to the XCDs in spans of (batch, tile)
  mid_batched_case(3, 129, 130, 128);    // a workgroup count that is not a multiple of 8
#endif
#if PART != 1 && PART != 2 && PART != 4
  // the slices kernel in every layout: depths below a step, ragged and whole, operands that end inside a piece, fewer
  // rows than a tile, rows shorter than a piece
  slices_case<false, false, 8>(70, 33, 333);
  slices_case<true, false, 8>(45, 64, 300);
  slices_case<false, true, 8>(64, 3, 259);
  slices_case<true, true, 8>(3, 5, 131);
  slices_case<true, true, 4>(129, 40, 64);
  slices_case<false, false, 4>(1, 77, 17);
  slices_case<true, false, 4>(100, 31, 96);
  slices_case<false, true, 4>(33, 97, 40);
  slices_case<true, true, 8>(1, 1, 700);
  // the convolution on planes: channel counts that are not whole pieces, one or two planes per slab, several
  // slabs in one stage and in several, tiles over rows and images, strides, padding on any side, spans of tiles
  planes_case<2, 2, 1, 4, 1, 3>(2, 9, 20, 20, 70, 3, 3, 1, 1, 1, 1, 9, 20, 150000, 2, 1);
  planes_case<2, 1, 1, 4, 1, 3>(3, 7, 7, 50, 33, 3, 3, 1, 1, 1, 1, 7, 7, 60000, 2, 2);
  planes_case<2, 1, 1, 4, 1>(3, 7, 7, 50, 33, 3, 3, 1, 1, 1, 1, 7, 7, 40000, 1, 1);
  planes_case<1, 1, 1, 2, 4, 3>(2, 7, 8, 70, 40, 3, 3, 2, 2, 0, 1, 4, 4, 60000, 1, 1);
  planes_case<1, 1, 1, 2, 4>(2, 9, 8, 70, 40, 3, 3, 2, 1, 0, 1, 5, 8, 150000, 2, 1);
  planes_case<2, 2, 2, 2, 1>(1, 13, 17, 3, 130, 3, 3, 2, 1, 1, 1, 7, 17, 80000, 2, 1);
  planes_case<1, 2, 1, 4, 1>(1, 300, 1, 37, 17, 1, 1, 1, 1, 0, 0, 300, 1, 80000, 1, 2);
  planes_case<1, 1, 1, 1, 4>(1, 6, 9, 64, 64, 5, 2, 1, 3, 4, 0, 10, 4, 50000, 2, 1);
  planes_case<1, 1, 1, 4, 1>(2, 5, 6, 48, 31, 3, 3, 1, 1, 1, 1, 5, 6, 80000, 1, 1);
  planes_case<1, 1, 1, 1, 4, 3>(1, 4, 9, 200, 40, 3, 3, 1, 1, 1, 1, 4, 9, 150000, 2, 1);
#endif
#if PART == 0 || PART == 4
  // the fp32 slices kernel in its three forms: depths of less than half a step, a step, a step and a bit, fewer steps than
  // slices and more; the planes' tile of eight wavefronts; Gemv widths of less than a piece, a piece and a rest, whole
  // and broken turns, rows that leave part of a wavefront's four, vectors that leave part of a pass
  f32_slices_case<true, true, 1, 8>(1, 33, 31, 3);
  f32_slices_case<true, false, 1, 8>(2, 1, 65, 15);
  f32_slices_case<false, true, 1, 8>(1, 70, 1, 17);
  f32_slices_case<false, false, 1, 8>(1, 40, 33, 200);
  f32_slices_case<true, true, 1, 8>(1, 32, 32, 16, 0, true);
  f32_slices_case<true, true, 1, 4>(1, 65, 33, 100);
  f32_slices_case<false, false, 1, 4>(3, 31, 34, 41);
  f32_slices_case<true, false, 1, 4>(3, 40, 0, 23, 49);
  f32_slices_case<true, true, 2, 8>(1, 33, 65, 129);
  f32_slices_case<true, false, 2, 8>(2, 64, 0, 50, 37);
  f32_slices_case<false, true, 2, 8>(1, 5, 63, 301, 0, true);
  // the tiles with checked loads in every layout and form: depths below a piece, a piece, a piece and a bit, a k tile and
  // a bit, several; operands at any address; parts that end inside a k tile and with less than a piece; an infinity
  f32_tile_case<true, true, 1, true, 128>(1, 130, 3, 3);
  f32_tile_case<true, false, 1, true, 128>(2, 3, 70, 7);
  f32_tile_case<false, true, 1, true, 128>(1, 33, 129, 8);
  f32_tile_case<false, false, 1, true, 128>(1, 129, 5, 9);
  f32_tile_case<true, true, 1, true, 64>(1, 65, 130, 15);
  f32_tile_case<true, false, 1, true, 64>(3, 7, 50, 49);
  f32_tile_case<false, true, 1, true, 64>(1, 64, 33, 7);
  f32_tile_case<false, false, 1, true, 64>(1, 5, 131, 65);
  f32_tile_case<true, true, 2, true, 128>(1, 40, 129, 63);
  f32_tile_case<true, false, 2, true, 128>(2, 131, 20, 5);
  f32_tile_case<false, true, 2, true, 128>(1, 3, 33, 41);
  f32_tile_case<false, false, 2, true, 128>(1, 35, 1, 100);
  f32_tile_case<true, true, 1, true, 128>(1, 9, 17, 48, 1);
  f32_tile_case<true, true, 1, true, 64>(1, 3, 2, 83, 3);
  f32_tile_case<true, true, 2, true, 128>(1, 9, 17, 96, 2);
  f32_tile_case<true, false, 2, true, 128>(1, 34, 40, 70, 0, 2);
  f32_tile_case<true, true, 2, true, 128>(1, 33, 41, 85, 1, 3);
  f32_tile_case<true, true, 1, true, 128>(1, 33, 34, 6, 0, 0, true);
  f32_tile_case<false, true, 2, true, 128>(1, 33, 34, 43, 0, 0, true);
  // ... and with loads that need no check
  f32_tile_case<true, true, 1, false, 128>(1, 130, 131, 48);
  f32_tile_case<true, false, 1, false, 64>(2, 33, 70, 16);
  f32_tile_case<false, true, 2, false, 128>(1, 40, 33, 48);
  f32_tile_case<false, false, 2, false, 128>(1, 7, 9, 64, 0, 2);
  f32_gemv_case<1, 1>(1, 5, 1, false, 0);
  f32_gemv_case<1, 1>(1, 7, 255, false, 0);
  f32_gemv_case<1, 1>(2, 3, 1027, true, 1);
  f32_gemv_case<1, 1>(1, 2, 4097, false, 3);
  f32_gemv_case<3, 1>(5, 6, 261, false, 2);
  f32_gemv_case<4, 1>(7, 3, 1030, false, 0);
  f32_gemv_case<1, 4>(1, 9, 3, false, 0);
  f32_gemv_case<2, 4>(2, 17, 259, false, 0);
  f32_gemv_case<4, 4>(6, 33, 516, false, 1);
  f32_gemv_case<6, 4>(6, 6, 77, false, 2);
  f32_gemv_case<16, 4>(17, 18, 2051, false, 3);
  f32_gemv_case<0, 1>(1, 6, 513, false, 0);
  f32_gemv_case<0, 1>(3, 3, 767, true, 0);
  f32_gemv_case<0, 1>(2, 5, 1090, false, 0);
  planes_case<2, 1, 1, 8, 1, 3>(2, 9, 20, 20, 70, 3, 3, 1, 1, 1, 1, 9, 20, 150000, 2, 1);
  planes_case<2, 1, 1, 8, 1, 3>(5, 7, 9, 50, 33, 3, 3, 1, 1, 1, 1, 7, 9, 60000, 1, 2);
#endif
#if PART == 0 || PART == 5
  // the convolution on staged rows: every tile form, whole and broken pieces, tiles over rows and images, tiles of
  // whole images, strides above and below the filter, padding on any side, patches that end inside a stage
  staged_case<2, 8, true>(1, 4, 9, 16, 40, 3, 3, 1, 1, 1, 1, 4, 9, 4);
  staged_case<1, 8, false>(2, 3, 4, 45, 31, 3, 3, 1, 1, 2, 2, 5, 6, 2);
  staged_case<2, 4, false>(2, 7, 7, 35, 33, 3, 3, 1, 1, 1, 1, 7, 7, 1);
  staged_case<1, 4, true>(1, 9, 8, 32, 5, 4, 2, 2, 1, 1, 1, 4, 18, 1);
  staged_case<2, 2, true>(1, 13, 14, 64, 36, 1, 1, 1, 1, 0, 0, 13, 14, 1);
  staged_case<1, 2, false>(1, 29, 9, 21, 20, 2, 3, 1, 2, 0, 1, 28, 5, 1);
  staged_case<2, 1, false>(1, 19, 15, 3, 34, 5, 5, 1, 1, 2, 2, 19, 15, 1);
  staged_case<2, 1, true, true>(1, 25, 22, 16, 34, 1, 1, 1, 1, 0, 0, 25, 22, 1);
  staged_case<1, 1, true>(6, 16, 20, 16, 9, 3, 3, 2, 2, 0, 0, 7, 9, 1);
  // the fp32 panel kernel in its forms: rows and columns that end inside a block, one row, images of other than whole
  // blocks, more wavefronts than blocks and blocks for a second turn, depths of a step and a bit, a step less one, whole
  // ones, padded to the steps ahead; rows along the depth or not; an infinity
  f32_panel_case<1, 2, true>(1, 1, 33, 17, 1);
  f32_panel_case<1, 2, false>(3, 31, 50, 32, 2);
  f32_panel_case<1, 4, true>(2, 33, 49, 33, 1, false);
  f32_panel_case<1, 4, false>(1, 32, 300, 64, 1);
  f32_panel_case<2, 2, true>(5, 65, 7, 31, 1);
  f32_panel_case<2, 2, false>(1, 64, 64, 48, 1, false);
  f32_panel_case<2, 4, true>(2, 40, 33, 113, 2);
  f32_panel_case<2, 4, false>(1, 5, 290, 80, 1);
  f32_panel_case<1, 2, true>(2, 30, 40, 21, 1, true, true);
  f32_panel_case<2, 4, true>(1, 70, 37, 59, 1, false, true);
#endif
  if (g_failures) {
    printf("kernel_emu: %d failures in %d cases\n", g_failures, g_cases);
    return 1;
  }
  printf("kernel_emu: ok (%d cases)\n", g_cases);
  return 0;
}
