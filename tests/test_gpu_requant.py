"""The uint8 output pipeline as the GEMM kernels evaluate it -- one 64-bit multiply-add per output, its
sign term and its clamp -- at the edges of that form, and just outside it, where the plain arithmetic
takes over.  The accumulators are read back through the int32 entry point and
put through the oracle's pipeline: equal bytes are required."""
import numpy as np
import pytest

from mace_amd import lib as mh
from oracle import mace_oracle as orc
from gpu_util import Dev

pytestmark = pytest.mark.gpu
M, K, N = 64, 64, 80      # 80 columns: whole tiles and a ragged one

CASES = [  # multiplier, right shift, zero point, clamp
    (2 ** 30, 1, 0, 0, 255), (2 ** 31 - 1, 1, 0, 0, 255),        # smallest shift, no sign term (zero point 0)
    (2 ** 30, 1, 128, 0, 255), (2 ** 31 - 1, 7, 128, 0, 255),    # sign term
    (2 ** 30 + 1, 9, 131, 131, 255), (1649267328, 9, 17, 17, 201), (1518500250, 12, 255, 3, 254),   # clamps
    (1518500250, 12, -300, 0, 255), (1518500250, 12, 700, 0, 255),   # offsets outside the byte
    (1, 4, 10, 0, 255), (3, 1, 250, 0, 255),                     # multipliers far below 2^30
    (2 ** 31 - 1, 22, 255, 0, 255), (2 ** 31 - 1, 23, 128, 0, 255),  # the largest shift with any byte offset; past it
    (2 ** 31 - 1, 30, 1, 0, 255), (2 ** 31 - 1, 30, 77, 77, 77), (2 ** 31 - 1, 31, 5, 0, 255),
    (2 ** 30, 0, 128, 0, 255), (2 ** 31 - 1, 0, 3, 0, 255),      # no shift
    (2 ** 29 + 5, 0, 17, 17, 201), (2 ** 30 + 9, 0, 255, 3, 254), (2 ** 31 - 1, 0, 700, 0, 255), (1, 0, 10, 0, 255),
    (-5, 3, 10, 0, 255), (-2 ** 31, 3, 10, 0, 255), (2 ** 30, 4, 40000, 0, 255),   # the plain arithmetic
]


@pytest.fixture(scope="module")
def ctx():
    c = mh.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("mult,shift,zp,lo,hi", CASES)
def test_output_pipeline(ctx, mult, shift, zp, lo, hi):
    rng = np.random.default_rng(shift * 1000 + zp)
    d = Dev()
    a = d.put(rng.integers(0, 256, (M, K), dtype=np.uint8))
    b = d.put(rng.integers(0, 256, (K, N), dtype=np.uint8))
    # biases that put the sums where the output moves (2^(shift + 8) or so either side of zero), at
    # zero, and at the ends of int32
    span = min(2 ** (shift + 8 + (31 - max(abs(mult), 1).bit_length())), 2 ** 30)
    bias = rng.integers(-span, span + 1, M).astype(np.int32)
    bias[:4] = 0
    bias[4:6] = 2 ** 31 - 1 - 2 ** 23, -2 ** 31 + 2 ** 23
    t32, p32 = d.empty(M * N, np.int32)
    t8, p8 = d.empty(M * N, np.uint8)
    pb = d.put(bias)
    d.sync()
    ctx.call("mace_hip_gemm_q8_i32", a, 0, b, 0, p32, 0, 1, M, K, N, 1, 1, -120, -131)
    ctx.call("mace_hip_gemm_q8_u8", a, 0, b, 0, p8, 0, 1, M, K, N, 1, 1, -120, -131, pb, mult, shift, zp, lo, hi)
    ctx.sync()
    acc = t32.cpu().numpy().reshape(M, N) + bias[:, None]
    want = np.array([orc.requant_fixed_u8(v, mult, shift, zp, lo, hi) for v in acc.reshape(-1)], np.uint8)
    assert np.array_equal(t8.cpu().numpy()[:M * N], want)


# layers of the kernels that have no other requantization: strips of few and of many channels, streaming
CONVS = [((64, 7, 8, 16, 1, 2, 0), "q8_conv_short_kernel"), ((64, 7, 32, 64, 3, 2, 2), "q8_conv_rows_kernel"),
         ((32, 56, 32, 64, 1, 1, 0), "q8_gemm_stream_kernel")]
# in_scale * filter_scale / out_scale, its right shift, output zero point, whether the form holds it
FORMS = [(0.7, 0, 0, True), (0.9999, 0, 131, True), (0.3, 1, 255, True), (0.005, 7, 128, True), (1.5e-7, 22, 200, True),
         (9e-8, 23, 255, True), (4e-10, 31, 0, True), (4.5e-8, 24, 200, False), (4e-10, 31, 128, False)]


@pytest.mark.parametrize("conv,kernel", CONVS)
@pytest.mark.parametrize("real,s,ozp,held", FORMS)
def test_convolutions_at_any_multiplier(ctx, conv, kernel, real, s, ozp, held):
    n, hw, cin, cout, k, st, pad = conv
    rng = np.random.default_rng(ozp + cin)
    near = 3 if real > 0.1 else 128      # bytes this close to the zero points: sums of a few hundred
    x = rng.integers(128 - near, 128 + near, (n, hw, hw, cin), dtype=np.uint8)
    f = rng.integers(128 - near, 128 + near, (cout, k, k, cin), dtype=np.uint8)
    span = int(min(300 / real, 2 ** 31 - 2 ** 24))
    bias = rng.integers(-span, span, cout).astype(np.int32)
    s_in, s_f = 0.02, 0.01
    s_out = s_in * s_f / real
    mult, shift = mh.get_output_multiplier_and_shift(s_in, s_f, s_out)
    assert mult >= 2 ** 30 and shift == s
    want = orc.conv2d_q8_nhwc(x, f, bias, n, hw, hw, cin, cout, k, k, (st, st), (pad, pad), s_in, 130, s_f, 126,
                              s_in * s_f, s_out, ozp, nthreads=16).reshape(-1)
    d = Dev()
    dx, df, db = d.put(x), d.put(f), d.put(bias)
    t, po = d.empty(want.size, np.uint8)
    d.sync()
    ctx.call("mace_hip_conv2d_q8_nhwc", dx, df, db, n, hw, hw, cin, cout, k, k, st, st, pad, pad, s_in, 130, s_f,
             126, s_in * s_f, s_out, ozp, 0, 255, po)
    plan = ctx.last_plan()
    ctx.sync()
    assert plan.kernel.startswith(kernel + "<") == held, plan
    assert len(np.unique(want)) >= (4 if real > 1e-9 else 2)   # (bias alone decides where the multiplier is small)
    np.testing.assert_array_equal(t.cpu().numpy()[:want.size], want)
