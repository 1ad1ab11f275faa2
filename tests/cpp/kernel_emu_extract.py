"""Cuts the source text of a few GPU kernels out of the .hip files in mace_amd/csrc for kernel_emu.cpp, which
compiles them for the host (see there).  Usage: kernel_emu_extract.py <output directory>."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
CSRC = os.path.join(ROOT, "mace_amd", "csrc")

# (first line of the piece, first line of what follows it)
PIECES = [
    ("constexpr int BK = 64;", "// A piece that was loaded `early` bytes"),
    ("__device__ inline v4i bytes_from", "// Sum of the 16 bytes of a fragment as read"),
    ("__device__ inline int sum16_u8", "// Epilogue shared by the GEMM kernels"),
    ("template <int WX, int WY, int FX, int FY, typename OutT, bool SUMY, bool PRESTAGED = false>",
     "// ---- small problems: everything in one launch"),
    ("template <typename OutT, bool XT, bool YT, bool BW>\n__global__ __launch_bounds__(256, BW ? 5 : 1) void q8_gemm_fused_small_kernel",
     "// ---- the streaming GEMM kernel: global -> LDS"),
    ("template <int WX, int WY, int FX, int FY, int STAGES, typename OutT, int OCC = 1,",
     "// ---- few tiles, any layout, any depth"),
    ("template <typename OutT, bool XT, bool YT, int WK>\n__global__ __launch_bounds__(512, 4) void q8_gemm_slices_kernel",
     "// ---- one round of 128 x 128 tiles"),
    ("template <typename OutT, int STAGES, bool XT, bool YT = false, bool LOOSE = false>\n__global__ __launch_bounds__(512, 1) void q8_gemm_mid_kernel",
     "// ---- the kernel for an X panel that fits in LDS"),
    ("template <int FX, int FY, int G, typename OutT, int OCC, bool CONV = false, bool XT = false,",
     "// ---- the streaming kernel for a small X panel"),
    ("struct RepackJob {", "__global__ __launch_bounds__(256) void q8_zero_i32_kernel"),
    ("template <int LPR>\n__global__ __launch_bounds__(256) void q8_panel_sums_kernel",
     "int launch_panel_sums("),
]
# the fp32 tile, panel and slices kernels and the Gemv kernels
F32_PIECES = [
    ("constexpr int TM = 128, TN = 128, TK = 16;", "// ---- the tile kernels: binary32 products"),
    ("typedef float f4v __attribute__", "// ---- few tiles, or shallow ones: a wavefront per slice"),
    ("template <bool LK, bool RK, int FN, int WK>", "// Depths of at most two: 0"),
    ("struct F32GemvParams {", "}  // namespace\n\n// Tiles of 32 x 32 fn"),
]
# source lines that only make sense on the GPU, and what stands in for them on the host
PATCHES = [
    ("extern __shared__ __align__(16) uint8_t lds[];", "uint8_t *lds = emu_lds();"),
    ("__launch_bounds__(256, OCC)", ""),
    ("__launch_bounds__(WX *WY * 64, OCC)", ""),
    ("__launch_bounds__(512, 1)", ""),
    ('asm volatile("" ::: "memory");', ""),
    # 16-byte accesses at addresses that are multiples of 8 only: fine on the GPU, not for SSE
    ("v4i v = *(const v4i *)at;", "v4i v; memcpy(&v, at, 16);"),
    ("*(v4i *)(to + 16 * lane) = *(const v4i *)from;", "memcpy(to + 16 * lane, from, 16);"),
]


def main(out_dir):
    src = open(os.path.join(CSRC, "q8_gemm.hip")).read()
    parts = []
    for first, after in PIECES:
        if first not in src or after not in src[src.index(first):]:
            sys.exit("kernel_emu_extract: q8_gemm.hip no longer has the piece that starts with %r" % first)
        a = src.index(first)
        parts.append(src[a:src.index(after, a)])
    body = "\n".join(parts)
    for old, new in PATCHES:
        if old not in body:
            sys.exit("kernel_emu_extract: q8_gemm.hip no longer has the line %r" % old)
        body = body.replace(old, new)
    open(os.path.join(out_dir, "kernels.inc"), "w").write(body)
    transfer = open(os.path.join(CSRC, "q8_transfer.h")).read()
    open(os.path.join(out_dir, "pieces.inc"), "w").write(
        transfer[transfer.index("__device__ __forceinline__ v4i moved_down"):transfer.index("// s_waitcnt vmcnt(N) alone")])
    planes = open(os.path.join(CSRC, "conv_planes.hip")).read()
    planes = planes[planes.index("struct ConvPlaneParams {"):planes.index("}  // namespace\n\n// Time that the one-launch")]
    for old, new in (("extern __shared__ __align__(16) uint8_t lds[];", "uint8_t *lds = emu_lds();"),
                     ('asm volatile("" ::: "memory");', "")):
        if old not in planes:
            sys.exit("kernel_emu_extract: conv_planes.hip no longer has the line %r" % old)
        planes = planes.replace(old, new)
    open(os.path.join(out_dir, "conv_planes.inc"), "w").write(planes)
    staged = open(os.path.join(CSRC, "conv_staged.hip")).read()
    staged = staged[staged.index("struct ConvStagedParams {"):staged.index("// Time that the staged kernel takes, in us")]
    old = "extern __shared__ __align__(16) uint8_t lds[];"
    if old not in staged:
        sys.exit("kernel_emu_extract: conv_staged.hip no longer has the line %r" % old)
    open(os.path.join(out_dir, "conv_staged.inc"), "w").write(staged.replace(old, "uint8_t *lds = emu_lds();"))
    src = open(os.path.join(CSRC, "f32_gemm.hip")).read()
    parts = []
    for first, after in F32_PIECES:
        if first not in src or after not in src[src.index(first):]:
            sys.exit("kernel_emu_extract: f32_gemm.hip no longer has the piece that starts with %r" % first)
        parts.append(src[src.index(first):src.index(after, src.index(first))])
    body = "\n".join(parts)
    if body.count("  return 0;\n#endif\n}") != 1:
        sys.exit("kernel_emu_extract: f32_gemm.hip no longer has the host's bf16_pair")
    body = body.replace("  return 0;\n#endif\n}", "  return emu_bf16_pair(x, y);\n#endif\n}")
    for old, new in (('asm("" : "+v"(t), "+s"(first));', ""),
                     ("extern __shared__ __align__(16) u4v panel[];", "u4v *const panel = (u4v *)emu_lds();")):
        if old not in body:
            sys.exit("kernel_emu_extract: f32_gemm.hip no longer has the line %r" % old)
        body = body.replace(old, new)
    open(os.path.join(out_dir, "f32.inc"), "w").write(body)
    rq = open(os.path.join(CSRC, "q8_requant.h")).read().replace('#include "common.h"', "")
    rq = rq.replace("#pragma once", "")
    open(os.path.join(out_dir, "requant.inc"), "w").write(rq)


if __name__ == "__main__":
    main(sys.argv[1])
