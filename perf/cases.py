"""What this library's users run, as timed cases: quantized MatMul, FullyConnected and Conv2D,
Quantize / Dequantize around them, and the fp32 MatMul and 1x1 convolution, from one image to large
batches, called through the C ABI (mace_amd.lib binds it) on tensors that are resident on the GPU.

A case's "kind" picks the op:

  matmul_q8      mace_hip_gemm_q8_u8 / _i32: [m x k] . [k x n], batched, either operand transposed
  fc_q8          mace_hip_gemv_q8_u8: weight [h x w] against `batch` vectors, int32 bias
  conv_q8        mace_hip_conv2d_q8_nhwc on each of the layers, SAME padding, int32 bias, ReLU6 range
  chain_q8       each of the layers as a float net runs it: Quantize, Conv2D, Dequantize
  matmul_f32     mace_hip_matmul_f32, batched, with a bias per column
  fc_f32         mace_hip_gemv_f32_act: weight [h x w] against `batch` vectors, bias, ReLU
  pointwise_f32  mace_hip_conv2d_f32_nchw with a 1x1 filter on each of the layers, bias, ReLU6

"layers" is a text: "HxWxCIN>COUTkKsS" for every layer (K x K filter, stride S), separated by spaces.
Layers are independent calls on inputs of their own: what lies between them in a net (depthwise
convolutions, poolings) is not part of this library.
"""
import ctypes as C
import functools
import math

import torch

from mace_amd import lib as mh

# MobileNetV1's pointwise layers at 224 x 224
POINTWISE = "112x112x32>64k1s1 56x56x128>128k1s1 28x28x256>256k1s1 14x14x512>512k1s1 7x7x1024>1024k1s1"
# MobileNetV1's first layer and the 3 x 3 layers of a residual net
SPATIAL = "224x224x3>32k3s2 56x56x64>64k3s1 28x28x128>128k3s1 14x14x256>256k3s1 7x7x512>512k3s1"

_ctx = None


def context():
    """The one context (a stream and its scratch arena) that a program keeps."""
    global _ctx
    if _ctx is None:
        _ctx = mh.Context(0)
    return _ctx


def listed():
    return [
        # one small quantized MatMul: a single op of a small net, launch latency
        dict(name="q8_matmul_128x256x128", kind="matmul_q8", batch=1, m=128, k=256, n=128, ta=False, tb=False,
             i32=False),
        # FullyConnected of one request, and of eight at once: the weights' bytes
        dict(name="q8_fc_4096x4096_b1", kind="fc_q8", batch=1, h=4096, w=4096),
        dict(name="q8_fc_4096x4096_b8", kind="fc_q8", batch=8, h=4096, w=4096),
        # the convolutions of one image, as an interactive program runs them
        dict(name="q8_conv_b1", kind="conv_q8", n=1, layers=POINTWISE + " " + SPATIAL),
        # pointwise and 3 x 3 layers of a serving batch
        dict(name="q8_pointwise_b64", kind="conv_q8", n=64, layers=POINTWISE),
        dict(name="q8_conv3x3_b64", kind="conv_q8", n=64, layers=SPATIAL),
        # float in, float out around quantized layers, at a middling batch
        dict(name="q8_chain_b16", kind="chain_q8", n=16, layers=POINTWISE),
        # a batched MatMul of odd sizes with the raw int32 result, right-hand matrix row-major
        dict(name="q8_matmul_ragged_i32", kind="matmul_q8", batch=4, m=1001, k=1500, n=777, ta=False, tb=False,
             i32=True),
        # square MatMuls: a common middle size and the largest
        dict(name="q8_matmul_2048", kind="matmul_q8", batch=1, m=2048, k=2048, n=2048, ta=False, tb=False, i32=False),
        dict(name="q8_matmul_8192", kind="matmul_q8", batch=1, m=8192, k=8192, n=8192, ta=False, tb=False, i32=False),
        # fp32: a batched MatMul against transposed weights, and the pointwise layers of a float net
        dict(name="f32_matmul_4x1024", kind="matmul_f32", batch=4, m=1024, k=1024, n=1024, ta=False, tb=True),
        dict(name="f32_pointwise_b64", kind="pointwise_f32", n=64, layers=POINTWISE),
    ]


# a drawn case's work stays below these (the largest listed case takes about half a millisecond)
MOST_OPS_Q8, MOST_OPS_CONV, MOST_OPS_F32, MOST_BYTES = 3e11, 3e10, 8e9, 2.5e8


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, uniform over its logarithm; every other one rounded to a
    multiple of the largest power of two (up to 64) that is at most a quarter of it, the rest as
    they come: odd ones among them."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < 0.5:
        unit = 1
        while unit < 64 and unit * 8 <= v:
            unit *= 2
        v = unit * round(v / unit)
    return max(lo, min(hi, int(round(v))))


def _draw_layers(rng, n, kinds):
    """One to three layers: few channels on large images to many channels on small ones."""
    out = []
    for _ in range(rng.randint(1, 3)):
        side = _log_int(rng, 7, 112)
        wide = max(7, min(112, side + rng.randint(-2, 2)))
        kernel, stride = rng.choice(kinds)
        cin = 3 if kernel == 3 and rng.random() < 0.2 else _log_int(rng, 16, max(17, min(1024, 8192 // side)))
        cout = _log_int(rng, 16, max(17, min(1024, 8192 // side)))
        out.append("%dx%dx%d>%dk%ds%d" % (side, wide, cin, cout, kernel, stride))
    return " ".join(out)


def draw(rng):
    while True:
        kind = rng.choice(["matmul_q8", "matmul_q8", "matmul_q8", "fc_q8", "conv_q8", "conv_q8", "conv_q8", "chain_q8",
                           "matmul_f32", "fc_f32", "pointwise_f32"])
        if kind in ("matmul_q8", "matmul_f32"):
            batch = rng.choice([1, 1, 1, _log_int(rng, 2, 32)])
            case = dict(kind=kind, batch=batch, m=_log_int(rng, 32, 8192), k=_log_int(rng, 32, 8192),
                        n=_log_int(rng, 32, 8192), ta=rng.random() < 0.25, tb=rng.random() < 0.5)
            if kind == "matmul_q8":
                case["i32"] = rng.random() < 0.3
        elif kind in ("fc_q8", "fc_f32"):
            case = dict(kind=kind, batch=rng.choice([1, 1, _log_int(rng, 2, 16)]), h=_log_int(rng, 64, 16384),
                        w=_log_int(rng, 64, 16384))
        else:
            n = rng.choice([1, _log_int(rng, 2, 64)])
            kinds = [(1, 1)] if kind == "pointwise_f32" else [(1, 1), (1, 1), (3, 1), (3, 1), (3, 2)]
            case = dict(kind=kind, n=n, layers=_draw_layers(rng, n, kinds))
        w = work(case)
        most = {"matmul_q8": MOST_OPS_Q8, "conv_q8": MOST_OPS_CONV, "chain_q8": MOST_OPS_CONV}.get(kind, MOST_OPS_F32)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= most:
            return case


def _layers(case):
    """(in_h, in_w, cin, cout, kernel, stride, out_h, out_w, pad_h, pad_w) of every layer, SAME padding."""
    for text in case["layers"].split():
        size, rest = text.split(">")
        h, w, cin = (int(v) for v in size.split("x"))
        cout, rest = rest.split("k")
        k, s = (int(v) for v in rest.split("s"))
        oh, ow = (h + s - 1) // s, (w + s - 1) // s
        yield (h, w, cin, int(cout), k, s, oh, ow, max((oh - 1) * s + k - h, 0), max((ow - 1) * s + k - w, 0))


def work(case):
    """Operations (a multiply and an add are two), and bytes: each input read, each output written, once."""
    kind = case["kind"]
    if kind in ("matmul_q8", "matmul_f32"):
        b, m, k, n = (case[v] for v in ("batch", "m", "k", "n"))
        if kind == "matmul_q8":
            nbytes = b * (m * k + k * n + m * n * (4 if case["i32"] else 1))
        else:
            nbytes = 4 * (b * (m * k + k * n + m * n) + n)
        return {"bytes": nbytes, "flops": 2 * b * m * k * n}
    if kind in ("fc_q8", "fc_f32"):
        b, h, w = case["batch"], case["h"], case["w"]
        size = 1 if kind == "fc_q8" else 4
        return {"bytes": size * (h * w + b * w + b * h) + 4 * h, "flops": 2 * b * h * w}
    nbytes = flops = 0
    for h, w, cin, cout, k, s, oh, ow, _, _ in _layers(case):
        n = case["n"]
        flops += 2 * n * oh * ow * cout * k * k * cin
        elements = n * (h * w * cin + oh * ow * cout)
        if kind == "pointwise_f32":
            nbytes += 4 * (elements + cout * cin + cout)
        else:
            # the chain's float input and output instead of bytes
            nbytes += (4 if kind == "chain_q8" else 1) * elements + cout * k * k * cin + 4 * cout
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Quantized results are whole numbers that follow from the inputs alone.  fp32: the order of the
    sums is free; against the same products summed in binary64 the 2-norm error measures about 4e-7
    at depth 1024."""
    if case["kind"].endswith("_f32"):
        return {"rel": 2e-6}
    if case["kind"] == "chain_q8":
        return {"rel": 1e-6}      # the same whole numbers, times the output scale
    return "exact"


class State:
    """Tensors of a case (kept alive), the bound calls of one pass, and the pass's outputs."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.keep, self.calls, self.outputs = [], [], []

    def _kept(self, t):
        self.keep.append(t)
        return t

    def u8(self, *shape):
        return self._kept(torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=self.gen))

    def i32(self, *shape):
        return self._kept(torch.randint(-2 ** 15, 2 ** 15, shape, dtype=torch.int32, device="cuda", generator=self.gen))

    def f32(self, *shape, scale=1.0):
        return self._kept(torch.randn(shape, dtype=torch.float32, device="cuda", generator=self.gen) * scale)

    def zero_point(self):
        """Near the middle of the byte range, where an asymmetric range of both signs puts it."""
        return int(torch.randint(116, 141, (1,), device="cuda", generator=self.gen))

    def out(self, dtype, *shape, result=True):
        t = self._kept(torch.empty(shape, dtype=dtype, device="cuda"))
        if result:
            self.outputs.append(t)
        return t

    def bind(self, name, *args):
        """The C function with its arguments converted once, as compiled code would have them."""
        ctx = context()
        fn = getattr(ctx.lib, name)
        conv = []
        for ctype, a in zip(fn.argtypes[1:], args):
            if isinstance(a, torch.Tensor):
                a = a.data_ptr()
            conv.append(ctype(a))
        assert len(conv) == len(args) == len(fn.argtypes) - 1, name
        self.calls.append(functools.partial(fn, ctx.handle, *conv))


def _out_scale(k, s_in, s_f, relu6):
    """An output scale that spreads the results over the byte range: uniform bytes make sums with a
    deviation of about 74 * 74 * sqrt(k) units."""
    span = 3 * 74.0 * 74.0 * math.sqrt(k) * s_in * s_f
    return max(6.0, span) / 255.0 if relu6 else 2 * span / 255.0


def prepare(case, seed):
    st = State(seed)
    kind = case["kind"]
    if kind == "matmul_q8":
        b, m, k, n = (case[v] for v in ("batch", "m", "k", "n"))
        lhs, rhs = st.u8(b, m, k), st.u8(b, k, n)       # a transposed operand is the same bytes, read the other way
        order = [b, m, k, n, int(b > 1), int(b > 1), -st.zero_point(), -st.zero_point()]
        if case["i32"]:
            out = st.out(torch.int32, b, m, n)
            st.bind("mace_hip_gemm_q8_i32", lhs, int(case["ta"]), rhs, int(case["tb"]), out, 0, *order)
        else:
            out = st.out(torch.uint8, b, m, n)
            mult, shift = mh.get_output_multiplier_and_shift(0.02, 0.015, _out_scale(k, 0.02, 0.015, False))
            st.bind("mace_hip_gemm_q8_u8", lhs, int(case["ta"]), rhs, int(case["tb"]), out, 0, *order, None, mult,
                    shift, 128, 0, 255)
    elif kind == "fc_q8":
        b, h, w = case["batch"], case["h"], case["w"]
        st.bind("mace_hip_gemv_q8_u8", st.u8(h, w), st.u8(b, w), st.i32(h), b, h, w, 0, 1, st.zero_point(),
                st.zero_point(), 0.01, 0.02, _out_scale(w, 0.01, 0.02, False), 128, mh.REQUANT_NEON,
                st.out(torch.uint8, b, h))
    elif kind in ("conv_q8", "chain_q8"):
        n = case["n"]
        for h, w, cin, cout, k, s, oh, ow, pad_h, pad_w in _layers(case):
            filt, bias, s_in, s_f = st.u8(cout, k, k, cin), st.i32(cout), 0.02, 0.01
            z_in, z_f, s_out = st.zero_point(), st.zero_point(), _out_scale(k * k * cin, 0.02, 0.01, True)
            if kind == "conv_q8":
                x, y = st.u8(n, h, w, cin), st.out(torch.uint8, n, oh, ow, cout)
            else:
                xf = st.f32(n, h, w, cin, scale=0.8)
                x = st.out(torch.uint8, n, h, w, cin, result=False)
                y = st.out(torch.uint8, n, oh, ow, cout, result=False)
                st.bind("mace_hip_quantize_tensor_u8", xf, xf.numel(), s_in, z_in, x)
            st.bind("mace_hip_conv2d_q8_nhwc", x, filt, bias, n, h, w, cin, cout, k, k, s, s, pad_h, pad_w, s_in, z_in,
                    s_f, z_f, s_in * s_f, s_out, 0, 0, 255, y)
            if kind == "chain_q8":
                yf = st.out(torch.float32, n, oh, ow, cout)
                st.bind("mace_hip_dequantize_tensor_u8", y, y.numel(), s_out, 0, yf)
    elif kind == "matmul_f32":
        b, m, k, n = (case[v] for v in ("batch", "m", "k", "n"))
        lhs = st.f32(b, k, m) if case["ta"] else st.f32(b, m, k)
        rhs = st.f32(b, n, k) if case["tb"] else st.f32(b, k, n)
        bias, out = st.f32(n), st.out(torch.float32, b, m, n)
        st.bind("mace_hip_matmul_f32", lhs, rhs, bias, b, *lhs.shape[1:], *rhs.shape[1:], int(case["ta"]),
                int(case["tb"]), int(b > 1), int(b > 1), out)
    elif kind == "fc_f32":
        b, h, w = case["batch"], case["h"], case["w"]
        st.bind("mace_hip_gemv_f32_act", st.f32(h, w, scale=w ** -0.5), st.f32(b, w), st.f32(h), b, h, w, 0, 1,
                mh.ACT_RELU, 0.0, st.out(torch.float32, b, h))
    else:
        n = case["n"]
        for h, w, cin, cout, k, s, oh, ow, _, _ in _layers(case):
            x, filt, bias = st.f32(n, cin, h, w), st.f32(cout, cin, scale=cin ** -0.5), st.f32(cout)
            st.bind("mace_hip_conv2d_f32_nchw", x, filt, bias, n, cin, h, w, cout, 1, 1, 1, 1, 1, 1, 0, 0,
                    mh.ACT_RELUX, 6.0, st.out(torch.float32, n, cout, h, w))
    return st


def run(state):
    for call in state.calls:
        status = call()
        if status:
            raise mh.MaceHipError(status, context().last_error())
    return state.outputs
