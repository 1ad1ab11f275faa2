"""The shapes that other tests run with kernels switched off, by the dispatch that a caller gets: whatever kernel takes them,
the results are the oracle's.  (Which one it is the plan tests hold.)"""
import json
import os

import numpy as np
import pytest

from mace_amd import lib as mh
from oracle import mace_oracle as orc
import test_gpu_conv2d_q8 as conv
import test_gpu_kernel_coverage as coverage
import test_gpu_q8_gemm as gemm

pytestmark = pytest.mark.gpu
R, Cm = mh.ROW_MAJOR, mh.COL_MAJOR
LATER = mh.MASK_NO_CONV_STAGED | mh.MASK_NO_F32_PANEL | mh.MASK_NO_Q8_LOOSE

with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "kernel_recipes.json")) as _f:
    RECIPES = [r for r in json.load(_f) if r["call"].get("mask", 0) & LATER]


@pytest.fixture(scope="module")
def ctx():
    c = mh.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,cout,cin,in_h,in_w,k_h,k_w,pad,st", [c[:9] for c in conv.PLANES_CASES])
def test_convolutions_of_the_padded_planes(ctx, n, cout, cin, in_h, in_w, k_h, k_w, pad, st):
    rng = np.random.default_rng(cout * 7 + cin + k_h * 3 + k_w + in_w + 1)
    x = rng.integers(0, 256, (n, in_h, in_w, cin), dtype=np.uint8)
    f = rng.integers(0, 256, (cout, k_h, k_w, cin), dtype=np.uint8)
    bias = rng.integers(-2 ** 15, 2 ** 15, cout).astype(np.int32)
    z_in, z_f = int(rng.integers(110, 147)), int(rng.integers(110, 147))
    s_in, s_f = np.float32(0.02), np.float32(0.01)
    s_out = np.float32(max(6.0, 3 * 74.0 * 74.0 * np.sqrt(k_h * k_w * cin) * float(s_in * s_f)) / 255.0)
    _, _, ph, pw = orc.calc_padding_and_output_size(in_h, in_w, k_h, k_w, st, pad)
    for (bb, s_b, so, z_o, lo, hi) in ((bias, np.float32(s_in * s_f), s_out, 0, 0, 255),
                                       (bias, np.float32(2.5 * float(s_in * s_f)), s_out, 100, 100, 230),
                                       (None, np.float32(0), s_out, 128, 0, 255)):
        args = (x, f, bb, n, in_h, in_w, cin, cout, k_h, k_w, st, (ph, pw), s_in, z_in, s_f, z_f, s_b, so, z_o, lo, hi)
        want = orc.conv2d_q8_nhwc(*args, nthreads=16)
        np.testing.assert_array_equal(conv.conv_host(ctx, *args), want)


@pytest.mark.parametrize("recipe", RECIPES, ids=["%d-%s" % (i, r["kernel"]) for i, r in enumerate(RECIPES)])
def test_recipes_without_the_later_masks(ctx, recipe):
    call = recipe["call"]
    rng = np.random.default_rng(recipe["family"] * 1000 + recipe["variant"] + 1)
    ctx.call("mace_hip_ctx_set_kernel_mask", call["mask"] & ~LATER)
    try:
        coverage.RUN[call["kind"]](ctx, call, rng)
    finally:
        ctx.call("mace_hip_ctx_set_kernel_mask", 0)


@pytest.mark.parametrize("mask", [0, mh.MASK_NO_SMALL])
@pytest.mark.parametrize("batch,rows,depth,cols,lb,rb", gemm.REPACK_SHAPES + [(1, 80, 2048, 100, True, True)])
@pytest.mark.parametrize("lo,ro,oo", [(R, R, R), (R, Cm, R), (Cm, R, R), (Cm, Cm, Cm), (R, R, Cm)])
def test_products_that_are_repacked(ctx, mask, batch, rows, depth, cols, lb, rb, lo, ro, oo):
    ctx.call("mace_hip_ctx_set_kernel_mask", mask)
    try:
        gemm.check_gemm(ctx, batch, rows, depth, cols, lb, rb, lo, ro, oo)
    finally:
        ctx.call("mace_hip_ctx_set_kernel_mask", 0)


@pytest.mark.parametrize("batch,rows,depth,cols,lb,rb,lo,ro,oo", [c[:9] for c in gemm.MID_SHAPES])
def test_products_of_one_round_of_tiles(ctx, batch, rows, depth, cols, lb, rb, lo, ro, oo):
    gemm.check_gemm(ctx, batch, rows, depth, cols, lb, rb, lo, ro, oo)


@pytest.mark.parametrize("n,h,w,cin,cout", [(8, 34, 36, 108, 28), (64, 14, 14, 256, 256), (1, 18, 18, 160, 160), (24, 40, 41, 13, 70),
                                            (1, 13, 12, 255, 232)])
def test_convolutions_with_a_registered_filter(ctx, n, h, w, cin, cout):
    import torch
    rng = np.random.default_rng(n + cin + 1)
    f = rng.integers(0, 256, (cout, 3, 3, cin), dtype=np.uint8)
    fd = torch.from_numpy(f).cuda()
    out = torch.empty(n * h * w * cout, dtype=torch.uint8, device="cuda")
    ctx.call("mace_hip_weight_register", fd.data_ptr(), fd.numel())
    try:
        for zp in (90, 128, 200):
            x = rng.integers(0, 256, (n, h, w, cin), dtype=np.uint8)
            bias = rng.integers(-2 ** 15, 2 ** 15, cout).astype(np.int32)
            xd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(bias).cuda()
            out.fill_(0xA5)
            torch.cuda.synchronize()
            ctx.call("mace_hip_conv2d_q8_nhwc", xd.data_ptr(), fd.data_ptr(), bd.data_ptr(), n, h, w, cin, cout, 3, 3, 1, 1, 2, 2,
                     0.02, zp, 0.01, 121, float(np.float32(0.02 * 0.01)), 2.0, 10, 0, 255, out.data_ptr())
            ctx.sync()
            want = orc.conv2d_q8_nhwc(x, f, bias, n, h, w, cin, cout, 3, 3, (1, 1), (2, 2), 0.02, zp, 0.01, 121,
                                      np.float32(0.02 * 0.01), 2.0, 10, nthreads=16)
            np.testing.assert_array_equal(out.cpu().numpy().reshape(want.shape), want)
    finally:
        ctx.call("mace_hip_weight_unregister", fd.data_ptr())
