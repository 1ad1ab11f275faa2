"""The fp32 GEMM kernels at the edges of their forms: k tiles of 16 and 32 with half a tile at the end,
guarded depths, 64- and 128-row tiles, columns of a batch run as one long row, parts of the depth; and
operands that the split into bf16 parts cannot represent, which a tile is computed again for; and operands
so small that unscaled parts would be subnormal.

Bound: six MFMAs per 16 depths, each rounding the running sum twice (2^-24 of at most sum |a||b|), eight
products at a time aligned to the largest of them (8 2^-24), left-out products 2^-24 and the split's
own last bit: (0.75 K + 16) 2^-24 sum |a||b|, element by element."""
import numpy as np
import pytest

from mace_amd import lib as mh
from gpu_util import Dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[mh.MASK_NO_F32_SLICES, 0], ids=["tiles", "any"])
def ctx(request):
    """the tile kernels alone, and with the slices kernel for the calls that it takes"""
    c = mh.Context(0)
    c.lib.mace_hip_ctx_set_kernel_mask(c.handle, request.param)
    yield c
    c.close()


def run(ctx, a, b, lb=True, rb=True, ta=False, tb=False, bias=None):
    """a [batch, m, k], b [batch, k, n], bias [n] -> result and the sums of |a||b|, binary64 on the CPU"""
    batch = max(a.shape[0], b.shape[0])
    m, k, n = a.shape[1], a.shape[2], b.shape[2]
    d = Dev()
    pa = d.put(a.transpose(0, 2, 1) if ta else a)
    pb = d.put(b.transpose(0, 2, 1) if tb else b)
    pbias = None if bias is None else d.put(bias)
    t, po = d.empty(batch * m * n, np.float32)
    d.sync()
    ctx.call("mace_hip_matmul_f32", pa, pb, pbias, batch, *((k, m) if ta else (m, k)), *((n, k) if tb else (k, n)),
             int(ta), int(tb), int(lb), int(rb), po)
    ctx.sync()
    with np.errstate(all="ignore"):
        want = np.matmul(a.astype(np.float64), b.astype(np.float64))
        size = np.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64))
        if bias is not None:
            want, size = want + bias, size + np.abs(bias)
    return t.cpu().numpy().reshape(batch, m, n), want, size


def close(got, want, size, k):
    assert np.all(np.abs(got - want) <= (0.75 * k + 16) * 2.0 ** -24 * size)


@pytest.mark.parametrize("m,k,n", [(128, 16, 128), (64, 48, 129), (130, 80, 49), (65, 33, 127), (1, 7, 1), (200, 100, 260)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_tile_edges(ctx, m, k, n, ta, tb):
    rng = np.random.default_rng(m + k + n)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((1, m, k), (1, k, n)))
    close(*run(ctx, a, b, False, False, ta, tb), k)


@pytest.mark.parametrize("batch,m,k,n", [(3, 70, 64, 49), (200, 48, 32, 196), (5, 128, 96, 1), (90, 160, 40, 400)])
def test_shared_left_matrix_over_a_batch(ctx, batch, m, k, n):
    rng = np.random.default_rng(batch)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((1, m, k), (batch, k, n)))
    close(*run(ctx, a, b, lb=False), k)


@pytest.mark.parametrize("batch,m,k,n", [(3, 70, 64, 49), (40, 48, 33, 100), (300, 130, 64, 132)])
def test_shared_left_matrix_with_a_bias_per_column(ctx, batch, m, k, n):
    """every batch's columns take the same n biases"""
    rng = np.random.default_rng(n)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((1, m, k), (batch, k, n)))
    close(*run(ctx, a, b, lb=False, bias=rng.standard_normal(n).astype(np.float32)), k)


def test_few_tiles_and_a_long_depth(ctx):
    rng = np.random.default_rng(9)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((1, 100, 2064), (4, 2064, 30)))
    close(*run(ctx, a, b, lb=False), 2064)


# (at most one tile per CU; more: 128-row tiles, 64-row tiles with idle loader threads; depths that are not
# whole k tiles)
OUTSIDE = [(140, 64, 133), (40, 50, 300), (2304, 32, 2200), (2304, 33, 2200), (190, 48, 16401), (190, 19, 16401)]


@pytest.mark.parametrize("m,k,n", OUTSIDE)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_operands_outside_the_split(ctx, m, k, n, ta, tb):
    rng = np.random.default_rng(k)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((1, m, k), (1, k, n)))
    form = dict(lb=False, rb=False, ta=ta, tb=tb)
    close(*run(ctx, a * np.float32(2.0 ** -120), b * np.float32(2.0 ** 120), **form), k)   # scaled past bf16's range
    tiny = a.copy()
    tiny[0, 3] *= np.float32(2.0 ** -140)                  # a row of subnormal numbers
    close(*run(ctx, tiny, b * np.float32(2.0 ** 90), **form), k)
    huge = a.copy()
    huge[0, 5] = 0
    huge[0, 5, 1] = np.finfo(np.float32).max               # hi would round to infinity
    close(*run(ctx, huge, np.clip(b, -0.9, 0.9), **form), k)
    inf = a.copy()
    inf[0, 7, 2] = np.inf
    inf[0, 8, 0] = np.nan
    inf[0, m - 1, 1] = -np.inf
    bb = b.copy()
    bb[0, 2] = 1.0                                         # exact in bf16: its smaller parts are zeros
    got, want, _ = run(ctx, inf, bb, **form)
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(got), kind(want))
    keep = np.isfinite(want).all(axis=2)[0]
    close(got[:, keep], want[:, keep], np.matmul(np.abs(a[:, keep]).astype(np.float64), np.abs(bb)), k)
    got, want, size = run(ctx, np.zeros_like(a), b, **form)
    assert not got.any()


@pytest.mark.parametrize("batch,m,k,n", [(40, 48, 33, 100), (300, 130, 64, 132)])
def test_images_outside_the_split(ctx, batch, m, k, n):
    """tiles that straddle images are computed again as well"""
    rng = np.random.default_rng(batch)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((1, m, k), (batch, k, n)))
    b[:, 1, ::37] = 1e38
    close(*run(ctx, np.clip(a, -0.9, 0.9), b, lb=False), k)


# Relative 2-norm error: a part that the matrix instruction took for zero would show as 2^-18 = 4e-6
# (lo) or 2^-9 (mid); binary32 sums of these depths measure 1e-7 to 2e-7.
@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -105, 2.0 ** -110, 2.0 ** -118, 2.0 ** -126])
@pytest.mark.parametrize("m,k,n", [(140, 64, 133), (2304, 33, 2200)])
def test_small_operands_keep_all_their_parts(ctx, scale, m, k, n):
    rng = np.random.default_rng(k)
    a = (rng.standard_normal((1, m, k)) * scale).astype(np.float32)
    b = (rng.standard_normal((1, k, n)) * 2.0 ** 80).astype(np.float32)
    got, want, _ = run(ctx, a, b, False, False)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


def test_small_operands_go_at_full_speed(ctx):
    """the tails of a softmax (down to 1e-45 here) once took seven times as long"""
    rng = np.random.default_rng(3)
    x = rng.standard_normal((4, 1024, 1024)) * 25
    soft = np.exp(x - x.max(axis=2, keepdims=True))
    soft = (soft / soft.sum(axis=2, keepdims=True)).astype(np.float32)
    assert ((soft > 0) & (soft < 2.0 ** -112)).any(axis=2).mean() > 0.01
    b = rng.standard_normal((4, 1024, 1024)).astype(np.float32)
    times = []
    for a in (x.astype(np.float32), soft):
        d = Dev()
        pa, pb = d.put(a), d.put(b)
        _, po = d.empty(4 * 1024 * 1024, np.float32)
        d.sync()
        ctx.profile(True)
        for _ in range(20):
            ctx.call("mace_hip_gemm_f32", pa, pb, 4, 1024, 1024, 1024, 0, 0, 0, 1, 1, po)
        times.append(min(ctx.kernel_ms_list()))
        ctx.profile(False)
    assert times[1] < 2 * times[0], times


def test_joined_images_captured_without_scratch():
    """32 images of 7 x 7: joined they are few enough tiles to split the depth, one by one they are not.
    A context without scratch records the call unsplit; one that had to split before still refuses."""
    import ctypes as C
    n, cin, hw, cout = 32, 1024, 49, 1024
    rng = np.random.default_rng(1)
    x = rng.standard_normal((n, cin, hw)).astype(np.float32)
    f = (rng.standard_normal((cout, cin)) / 32).astype(np.float32)
    c = mh.Context(0)
    c.lib.mace_hip_ctx_set_kernel_mask(c.handle, mh.MASK_NO_F32_SLICES)
    try:
        d = Dev()
        px, pf = d.put(x), d.put(f)
        t, po = d.empty(n * cout * hw, np.float32)
        d.sync()
        args = (px, pf, None, n, cin, hw, cout, mh.ACT_RELU, 0.0, po)
        g = C.c_void_p()
        c.call("mace_hip_graph_capture_begin")
        status = c.status("mace_hip_conv1x1_f32_nchw", *args)
        plan = c.last_plan()
        refused = c.status("mace_hip_gemm_f32", px, pf, 1, 512, 512, 512, 0, 0, 0, 1, 1, po)
        c.call("mace_hip_graph_capture_end", C.byref(g))
        assert status == mh.SUCCESS and plan.launches == 1 and refused == mh.INVALID_ARGS
        want = np.maximum(np.matmul(f.astype(np.float64), x.astype(np.float64)), 0)
        size = np.matmul(np.abs(f).astype(np.float64), np.abs(x).astype(np.float64))
        for _ in range(3):
            t.zero_()
            d.sync()
            c.call("mace_hip_graph_launch", g)
            c.sync()
            close(t.cpu().numpy().reshape(want.shape), want, size, cin)
            t.zero_()
            d.sync()
            c.call("mace_hip_conv1x1_f32_nchw", *args)      # outside the capture: split, with scratch
            assert c.last_plan().aux & mh.AUX_F32_KSPLIT
            c.sync()
            close(t.cpu().numpy().reshape(want.shape), want, size, cin)
        c.call("mace_hip_graph_destroy", g)
    finally:
        c.close()


def test_long_depth_recorded_without_scratch():
    """62 x 2112 x 4552: tiles in parts of the depth where the parts can be had, else the slices kernel"""
    import ctypes as C
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((62, 2112)).astype(np.float32), rng.standard_normal((2112, 4552)).astype(np.float32)
    want = np.matmul(a.astype(np.float64), b.astype(np.float64))
    size = np.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64))
    c = mh.Context(0)
    try:
        d = Dev()
        pa, pb = d.put(a), d.put(b)
        t, po = d.empty(want.size, np.float32)
        d.sync()
        args = (pa, pb, 1, 62, 4552, 2112, 0, 0, 0, 1, 1, po)
        g = C.c_void_p()
        c.call("mace_hip_graph_capture_begin")
        status, kernel = c.status("mace_hip_gemm_f32", *args), c.last_plan().kernel
        c.call("mace_hip_graph_capture_end", C.byref(g))
        assert status == mh.SUCCESS and "slices" in kernel
        for _ in range(3):
            for run_it in (lambda: c.call("mace_hip_graph_launch", g), lambda: c.call("mace_hip_gemm_f32", *args)):
                t.zero_()
                d.sync()
                run_it()
                c.sync()
                close(t.cpu().numpy().reshape(want.shape), want, size, 2112)
            assert "slices" not in c.last_plan().kernel
        c.call("mace_hip_graph_destroy", g)
    finally:
        c.close()


@pytest.mark.parametrize("lm,rm,om", [(0, 0, 0), (0, 1, 1), (1, 0, 1), (1, 1, 0)])
@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("batch,m,n,lb", [(1, 300, 257, 1), (3, 70, 129, 1), (70, 1, 1001, 0), (3, 1001, 1, 1), (5, 1, 1, 1), (2, 64, 128, 1)])
def test_one_or_two_products_per_output(ctx, batch, m, n, lb, k, lm, rm, om):
    """as binary32 multiply-adds round them: one product once, two products twice"""
    rng = np.random.default_rng(m + n)

    def some(*shape):
        return (rng.standard_normal(shape) * 2.0 ** rng.integers(-60, 60, shape)).astype(np.float32)
    a, b = some(batch if lb else 1, m, k), some(batch, k, n)
    d = Dev()
    pa = d.put(a.transpose(0, 2, 1) if lm else a)
    pb = d.put(b.transpose(0, 2, 1) if rm else b)
    t, po = d.empty(batch * m * n, np.float32)
    d.sync()
    ctx.call("mace_hip_gemm_f32", pa, pb, batch, m, n, k, lm, rm, om, lb, 1, po)
    ctx.sync()
    got = t.cpu().numpy()
    got = got.reshape(batch, n, m).transpose(0, 2, 1) if om else got.reshape(batch, m, n)
    first = a[:, :, :1] * b[:, :1]
    if k == 1:
        assert np.array_equal(got, first)
    else:      # (binary64 holds the second product exactly; its sum with the first is rounded twice)
        want = first.astype(np.float64) + a[:, :, 1:].astype(np.float64) * b[:, 1:]
        assert np.all(np.abs(got - want) <= 0.5001 * np.spacing(np.abs(want).astype(np.float32)))


def test_one_product_per_output_with_bias_and_activation(ctx):
    rng = np.random.default_rng(2)
    x, f, bias = (rng.standard_normal(s).astype(np.float32) for s in ((3, 1, 50), (40, 1), (40,)))
    d = Dev()
    px, pf, pb = d.put(x), d.put(f), d.put(bias)
    t, po = d.empty(3 * 40 * 50, np.float32)
    d.sync()
    ctx.call("mace_hip_conv1x1_f32_nchw", px, pf, pb, 3, 1, 50, 40, mh.ACT_RELUX, 1.5, po)
    ctx.sync()
    want = np.clip(f[None] * x + bias[None, :, None], 0, np.float32(1.5))
    assert np.array_equal(t.cpu().numpy().reshape(3, 40, 50), want)


# tiles of 32 columns in 8 and 4 slices and of 64 in 8; depths of less than a step, whole steps, a step and a bit, and
# more steps than slices; rows and columns that leave part of a tile, one of either
SLICES_CASES = [("FN=1,WK=8", 1, 100, 70, 5), ("FN=1,WK=8", 2, 33, 31, 16), ("FN=1,WK=8", 1, 1, 300, 200),
                ("FN=1,WK=8", 3, 64, 95, 401), ("FN=1,WK=8", 1, 257, 1, 1003), ("FN=1,WK=4", 1, 1000, 550, 24),
                ("FN=1,WK=4", 5, 130, 1000, 40),
                ("FN=2,WK=8", 1, 500, 620, 777), ("FN=2,WK=8", 2, 384, 637, 900)]


@pytest.mark.parametrize("form,batch,m,n,k", SLICES_CASES)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_slices_of_the_depth(form, batch, m, n, k, ta, tb):
    """against binary64, and no further from it in the 2-norm than the tile kernels"""
    rng = np.random.default_rng(m + n + k)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((batch, m, k), (batch, k, n)))
    bias = rng.standard_normal(n).astype(np.float32)
    c = mh.Context(0)
    try:
        got, want, size = run(c, a, b, ta=ta, tb=tb, bias=bias)
        assert form in c.last_plan().kernel and c.last_plan().launches == 1, c.last_plan()
        close(got, want, size, k)
        c.lib.mace_hip_ctx_set_kernel_mask(c.handle, mh.MASK_NO_F32_SLICES)
        tiles = run(c, a, b, ta=ta, tb=tb, bias=bias)[0]
        assert "slices" not in c.last_plan().kernel
        off, before = (np.linalg.norm(x - want) / np.linalg.norm(want) for x in (got, tiles))
        assert off <= before, (off, before)
        c.lib.mace_hip_ctx_set_kernel_mask(c.handle, 0)
        # sums that are not finite: the tile again by the binary32 instruction, the others as they were
        a[0, m // 2, k // 2] = np.inf
        b[-1, k // 3, n // 2] = np.nan
        bad, want, size = run(c, a, b, ta=ta, tb=tb, bias=bias)
        with np.errstate(all="ignore"):
            lost = ~np.isfinite(want)
        assert np.array_equal(np.isnan(bad), np.isnan(want)) and np.array_equal(np.isposinf(bad), np.isposinf(want))
        assert np.array_equal(np.isneginf(bad), np.isneginf(want))
        with np.errstate(all="ignore"):
            assert np.all((np.abs(bad - want) <= (0.75 * k + 16) * 2.0 ** -24 * size) | lost)
    finally:
        c.close()


def test_slices_over_images_with_bias_and_activation():
    """pointwise layers: columns of all images side by side, bias per row, ReLUX"""
    rng = np.random.default_rng(4)
    c = mh.Context(0)
    try:
        for (n, cin, hw, cout) in ((1, 384, 272, 320), (5, 23, 64 * 66, 28), (16, 26, 49, 228), (3, 300, 7, 33)):
            x = rng.standard_normal((n, cin, hw)).astype(np.float32)
            f = (rng.standard_normal((cout, cin)) / np.sqrt(cin)).astype(np.float32)
            bias = rng.standard_normal(cout).astype(np.float32)
            d = Dev()
            px, pf, pb = d.put(x), d.put(f), d.put(bias)
            t, po = d.empty(n * cout * hw, np.float32)
            d.sync()
            c.call("mace_hip_conv1x1_f32_nchw", px, pf, pb, n, cin, hw, cout, mh.ACT_RELUX, 1.25, po)
            c.sync()
            assert "slices" in c.last_plan().kernel, c.last_plan()
            raw = np.matmul(f.astype(np.float64), x.astype(np.float64)) + bias[None, :, None]
            size = np.matmul(np.abs(f).astype(np.float64), np.abs(x).astype(np.float64)) + np.abs(bias)[None, :, None]
            close(t.cpu().numpy().reshape(raw.shape), np.clip(raw, 0, 1.25), size, cin)
    finally:
        c.close()


# tiles of 32 and 64 rows, two and four k steps ahead; rows, columns and depths that end inside a tile, a block, a step
PANEL_CASES = [("MI=1,D=2,GUARD=false", 37, 32, 30, 900), ("MI=1,D=4,GUARD=true", 37, 53, 30, 901), ("MI=2,D=2,GUARD=true", 33, 21, 64, 3001),
               ("MI=2,D=4,GUARD=false", 64, 128, 120, 800), ("MI=2,D=4,GUARD=true", 60, 211, 61, 1999), ("MI=1,D=4,GUARD=true", 24, 403, 129, 1500),
               ("MI=1,D=2,GUARD=true", 1, 17, 5, 33001), ("MI=1,D=2,GUARD=false", 700, 96, 90, 49)]


@pytest.mark.parametrize("form,images,k,m,n", PANEL_CASES)
def test_columns_streamed_past_rows_in_lds(form, images, k, m, n):
    """the same bits as the tile kernel's, the result alone written, against binary64; images that are not finite"""
    rng = np.random.default_rng(m + n + k)
    x, f, bias = (rng.standard_normal(s).astype(np.float32) for s in ((images, k, n), (m, k), (m,)))
    c = mh.Context(0)
    try:
        d = Dev()
        pf, pb = d.put(f), d.put(bias)

        def conv(x, act, mask):
            px = d.put(x)
            t, po = d.empty(images * m * n + 32, np.float32)
            t.fill_(-7.0)
            d.sync()
            c.lib.mace_hip_ctx_set_kernel_mask(c.handle, mask)
            c.call("mace_hip_conv1x1_f32_nchw", px, pf, pb, images, k, n, m, act, 3.0, po.value + 64)
            c.sync()
            got = t.cpu().numpy()
            assert (got[:16] == -7.0).all() and (got[16 + images * m * n:] == -7.0).all()
            return got[16:16 + images * m * n].reshape(images, m, n)
        for act in (mh.ACT_NOOP, mh.ACT_RELUX):
            got = conv(x, act, 0)
            assert c.last_plan().kernel == "f32_gemm_panel_kernel<%s>" % form, c.last_plan()
            tiles = conv(x, act, mh.MASK_NO_F32_PANEL)
            assert "panel" not in c.last_plan().kernel and "slices" not in c.last_plan().kernel
            assert np.array_equal(got, tiles)
        got = conv(x, mh.ACT_NOOP, 0)
        want = np.matmul(f.astype(np.float64), x.astype(np.float64)) + bias[:, None].astype(np.float64)
        size = np.matmul(np.abs(f).astype(np.float64), np.abs(x).astype(np.float64)) + np.abs(bias)[:, None]
        close(got, want, size, k)
        x[0, k // 2, n // 3] = np.inf
        x[-1, k // 3, n // 2] = np.nan
        x[images // 2, :, n - 1] = 1e36           # (beyond the split)
        got = conv(x, mh.ACT_NOOP, 0)
        want = np.matmul(f.astype(np.float64), x.astype(np.float64)) + bias[:, None].astype(np.float64)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        fin = np.isfinite(want)
        size = np.matmul(np.abs(f).astype(np.float64), np.abs(np.where(np.isfinite(x), x, 0)).astype(np.float64)) + np.abs(bias)[:, None]
        close(got[fin], want[fin], size[fin], k)
    finally:
        c.close()


# more tiles than CUs, of 128 and of 64 rows, and few tiles by eight wavefronts
GUARDED_TILES = [("SPLIT=1>", 2301, 2301), ("SPLIT=1,TM=64>", 190, 16401), ("SPLIT=2>", 300, 200)]


@pytest.mark.parametrize("form,m,n", GUARDED_TILES)
@pytest.mark.parametrize("k,off", [(3, 0), (7, 0), (8, 0), (9, 0), (15, 0), (49, 0), (63, 0), (65, 0), (1001, 0), (48, 1), (64, 3)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_tiles_of_guarded_depths(form, m, n, k, off, ta, tb):
    """Depths that are not whole k tiles, and operands that are not 16-byte pieces, in every layout: against binary64, the
    result alone written, and the same bits as the kernels without a check give for the depth filled up with zeros; then with
    an infinity, a NaN and numbers beyond the split in a few rows."""
    if off and ta and not tb:
        pytest.skip("no operand along the depth: any address is whole")
    rng = np.random.default_rng(m + 8 * k + off)
    a, b, bias = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (n,)))
    c = mh.Context(0)
    try:
        c.lib.mace_hip_ctx_set_kernel_mask(c.handle, mh.MASK_NO_F32_SLICES | mh.MASK_NO_F32_PANEL)
        d = Dev()
        pbias = d.put(bias)

        def matmul(a, b, off):
            kk = a.shape[1]
            l, r = (d.put(np.concatenate([np.zeros(off, np.float32), x.reshape(-1)]))
                    for x in (np.ascontiguousarray(a.T if ta else a), np.ascontiguousarray(b.T if tb else b)))
            t, po = d.empty(m * n + 32, np.float32)
            t.fill_(-7.0)
            d.sync()
            c.call("mace_hip_matmul_f32", l.value + 4 * off, r.value + 4 * off, pbias, 1, *((kk, m) if ta else (m, kk)),
                   *((n, kk) if tb else (kk, n)), int(ta), int(tb), 1, 1, po.value + 64)
            c.sync()
            got = t.cpu().numpy()
            assert (got[:16] == -7.0).all() and (got[16 + m * n:] == -7.0).all()
            return got[16:16 + m * n].reshape(m, n), c.last_plan().kernel
        got, kernel = matmul(a, b, off)
        assert kernel.startswith("f32_gemm_kernel<") and kernel.endswith(form), kernel
        size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64) + np.abs(bias)
        close(got, a.astype(np.float64) @ b.astype(np.float64) + bias, size, k)
        more = -k % 16
        filled, kernel = matmul(np.pad(a, ((0, 0), (0, more))), np.pad(b, ((0, more), (0, 0))), 0)
        assert kernel.startswith("f32_gemm_vec_kernel<") and kernel.endswith(form), kernel
        assert np.array_equal(got, filled)
        if k > 65:
            return
        a[m // 2, k - 1], a[m // 3, 0], a[m - 1] = np.inf, np.nan, 1e36
        got, _ = matmul(a, b, off)
        want = a.astype(np.float64) @ b.astype(np.float64) + bias
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        fin = np.isfinite(want)
        size = np.abs(np.where(np.isfinite(a), a, 0)).astype(np.float64) @ np.abs(b).astype(np.float64) + np.abs(bias)
        close(got[fin], want[fin], size[fin], k)
    finally:
        c.close()
