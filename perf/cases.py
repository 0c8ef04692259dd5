"""The work a user of this library has it do, as cases that can be timed: the call sequences a generated Session issues
through the C ABI (include/sofie_hip.h) on device-resident tensors, for whole networks and for single operators.

A state is what a Session owns: a context that made the constant-weights promise, weights laid out the way the emitter
lays them out (QLinearMatMul weights [N,K], QLinearConv weights [OC][KH][KW][C], int8 activations channels-last), one
buffer per tensor, and the list of calls of one inference. All contexts launch on one stream, as the Sessions of a
program that runs its models one after the other.

A case is a dict with a "kind" and its sizes:
  mlp        fp32 multilayer perceptron, one sofie_hip_mlp_f32 call            batch, widths
  gemm_f32   fp32 Gemm operator                                               M, N, K, transA, transB, bias, relu
  conv_f32   fp32 Conv operator, NCHW, bias + ReLU                             N, C, H, W, OC, k, s, p
  convt_f32  fp32 ConvTranspose operator                                      N, C, H, W, OC, k, s, p
  cnn_f32    the fp32 image classifier, layer by layer                         batch
  qgemm      int8 QLinearMatMul                                               M, N, K, transB, bias, relu, out
  gemm_fp8   e4m3 GEMM with bias, bf16 or fp32 out                             M, N, K, transB, out
  qconv      int8 QLinearConv, ReLU, optionally 2x2 max pooling behind it      N, C, H, W, OC, k, s, p, pool
             (first = True: QuantizeLinear of the float NCHW input in the same call)
  qcnn       the int8 image classifier, layer by layer                         batch
"""
import ctypes as C
import math

import torch

from sofie_amd import lib as L
from sofie_amd import ops

CONV_F32_FLOPS = 2 * 256 * 128 * 3136 * 576      # the largest fp32 case
ONE_BYTE_FLOPS = 2 * 8192 * 8192 * 4096          # the largest one-byte case


def listed():
    return [
        # a multilayer perceptron on a batch of events: a launch and nothing else
        {"name": "mlp_b256", "kind": "mlp", "batch": 256, "widths": "64-128-64-8"},
        # a fully connected layer whose sizes nobody rounded
        {"name": "gemm_f32_ragged", "kind": "gemm_f32", "M": 1500, "N": 1001, "K": 1111, "transA": False, "transB": False,
         "bias": True, "relu": True},
        # the float classifier on an ordinary batch: eight launches of every size
        {"name": "cnn_f32_b256", "kind": "cnn_f32", "batch": 256},
        # a wide 3x3 layer in the middle of a network, training-sized batch: the largest fp32 work
        {"name": "conv_f32_56", "kind": "conv_f32", "N": 256, "C": 64, "H": 56, "W": 56, "OC": 128, "k": 3, "s": 1, "p": 1},
        # the first layer of an image network: three channels, a large strided kernel
        {"name": "conv_f32_first", "kind": "conv_f32", "N": 16, "C": 3, "H": 224, "W": 224, "OC": 64, "k": 7, "s": 2, "p": 3},
        # an upsampling layer (the decoder direction)
        {"name": "convt_f32_28", "kind": "convt_f32", "N": 64, "C": 128, "H": 28, "W": 28, "OC": 64, "k": 4, "s": 2, "p": 1},
        # QLinearMatMul on two run-time operands, the benchmark's headline
        {"name": "qgemm_4096", "kind": "qgemm", "M": 4096, "N": 4096, "K": 4096, "transB": False, "bias": False, "relu": False,
         "out": "s8"},
        # a quantized layer of 1000 features and 1000 classes on a batch of 256
        {"name": "qgemm_1000", "kind": "qgemm", "M": 256, "N": 1000, "K": 1000, "transB": True, "bias": True, "relu": False,
         "out": "f32"},
        # the benchmark's FP8 product, the largest one-byte work
        {"name": "gemm_fp8_8192", "kind": "gemm_fp8", "M": 8192, "N": 8192, "K": 4096, "transB": True, "out": "bf16"},
        # the quantized classifier at the benchmark's batch and on a small one (latency)
        {"name": "qcnn_b4096", "kind": "qcnn", "batch": 4096},
        {"name": "qcnn_b64", "kind": "qcnn", "batch": 64},
        # a strided quantized layer whose channel counts fit no tile
        {"name": "qconv_48_80", "kind": "qconv", "N": 16, "C": 48, "H": 35, "W": 29, "OC": 80, "k": 3, "s": 2, "p": 1, "pool": False,
         "first": False},
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _size(rng, lo, hi):
    """A size spread over the logarithm of its range: half of them as drawn, half rounded to a multiple of 8, 16 or 64."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        q = rng.choice([8, 16, 64])
        v = max(q, v // q * q) if v >= q else v
    return max(lo, min(hi, v))


def _draw_gemm_sizes(rng, flops, lo_n, bytes_per):
    while True:
        M, N, K = _size(rng, 1, 8192), _size(rng, lo_n, 8192), _size(rng, 16, 8192)
        if 2 * M * N * K <= flops and bytes_per * (M * K + K * N + M * N) <= 1 << 30:
            return M, N, K


def _draw_conv(rng, flops, batch, transposed):
    while True:
        c = {"N": _size(rng, 1, batch), "C": rng.choice([1, 3]) if not transposed and rng.random() < 0.25 else _size(rng, 4, 256),
             "H": _size(rng, 5, 56 if transposed else 224)}
        c["W"] = c["H"] if rng.random() < 0.6 else _size(rng, 5, 56 if transposed else 224)
        c["OC"] = _size(rng, 8, 256)
        if transposed:
            c["k"], c["s"], c["p"] = rng.choice([(2, 2, 0), (3, 2, 1), (4, 2, 1)])
        else:
            c["k"] = rng.choice([1, 3, 3, 3, 5, 7])
            c["s"] = rng.choice([1, 1, 1, 2])
            c["p"] = c["k"] // 2
        oh, ow = _conv_out(c, transposed)
        madds = c["N"] * c["C"] * c["OC"] * c["k"] ** 2 * (c["H"] * c["W"] if transposed else oh * ow)
        if 2 * madds <= flops and 4 * c["N"] * (c["C"] * c["H"] * c["W"] + c["OC"] * oh * ow) <= 1 << 30:
            return c


def draw(rng):
    kind = rng.choice(["mlp", "gemm_f32", "cnn_f32", "conv_f32", "conv_f32", "convt_f32", "qgemm", "qgemm", "gemm_fp8", "qcnn", "qconv",
                       "qconv"])
    if kind == "mlp":
        while True:
            batch = _size(rng, 1, 16384)
            widths = [_size(rng, 8, 512) for _ in range(rng.randint(2, 5))] + [rng.randint(1, 64)]
            if batch * sum(a * b for a, b in zip(widths, widths[1:])) <= 1 << 29:      # above it the emitter keeps the layers apart
                return {"kind": kind, "batch": batch, "widths": "-".join(map(str, widths))}
    if kind in ("cnn_f32", "qcnn"):
        while True:
            batch = _size(rng, 1, 1024 if kind == "cnn_f32" else 4096)
            if batch not in (64, 256, 4096):      # these are listed
                return {"kind": kind, "batch": batch}
    if kind == "gemm_f32":
        M, N, K = _draw_gemm_sizes(rng, CONV_F32_FLOPS, 1, 4)
        return {"kind": kind, "M": M, "N": N, "K": K, "transA": rng.random() < 0.2, "transB": rng.random() < 0.5, "bias": rng.random() < 0.8,
                "relu": rng.random() < 0.5}
    if kind == "qgemm":
        M, N, K = _draw_gemm_sizes(rng, ONE_BYTE_FLOPS // 4, 1, 4)
        return {"kind": kind, "M": M, "N": N, "K": K, "transB": rng.random() < 0.7, "bias": rng.random() < 0.8, "relu": rng.random() < 0.5,
                "out": rng.choice(["s8", "s8", "f32"])}
    if kind == "gemm_fp8":
        M, N, K = _draw_gemm_sizes(rng, ONE_BYTE_FLOPS, 8, 2)
        return {"kind": kind, "M": M, "N": N, "K": K, "transB": rng.random() < 0.7, "out": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "qconv":
        c = _draw_conv(rng, CONV_F32_FLOPS, 256, False)
        oh, ow = _conv_out(c, False)
        first = c["C"] <= 3
        return dict(c, kind=kind, pool=min(oh, ow) >= 2 and rng.random() < 0.4, first=first)
    return dict(_draw_conv(rng, CONV_F32_FLOPS, 256, kind == "convt_f32"), kind=kind)


# ------------------------------------------------------------------------------------------------ shapes and work
def _conv_out(c, transposed=False):
    k, s, p = c["k"], c["s"], c["p"]
    if transposed:
        return s * (c["H"] - 1) + k - 2 * p, s * (c["W"] - 1) + k - 2 * p
    return (c["H"] + 2 * p - k) // s + 1, (c["W"] + 2 * p - k) // s + 1


CNN_LAYERS = ((1, 32, 40, True), (32, 64, 20, True), (64, 128, 10, False))      # channels in and out, size, pooled
CNN_FC = ((12800, 256), (256, 5))
CNN_MADDS = sum(ci * co * 9 * hw * hw for ci, co, hw, _ in CNN_LAYERS) + sum(k * n for k, n in CNN_FC)
CNN_WEIGHTS = sum(ci * co * 9 for ci, co, _, _ in CNN_LAYERS) + sum(k * n for k, n in CNN_FC)
OUT_BYTES = {"s8": 1, "f32": 4, "bf16": 2}


def work(case):
    k = case["kind"]
    if k == "mlp":
        w = [int(v) for v in case["widths"].split("-")]
        madds, b = sum(a * c for a, c in zip(w, w[1:])), case["batch"]
        return {"bytes": 4 * (b * (w[0] + w[-1]) + madds + sum(w[1:])), "flops": 2 * b * madds}
    if k in ("gemm_f32", "qgemm", "gemm_fp8"):
        M, N, K = case["M"], case["N"], case["K"]
        e = 4 if k == "gemm_f32" else 1
        o = 4 if k == "gemm_f32" else OUT_BYTES[case["out"]]
        return {"bytes": e * (M * K + K * N) + o * M * N + 8 * N, "flops": 2 * M * N * K}
    if k in ("cnn_f32", "qcnn"):
        b = case["batch"]
        return {"bytes": b * (1600 + 5) * 4 + CNN_WEIGHTS * (4 if k == "cnn_f32" else 1), "flops": 2 * b * CNN_MADDS}
    n, c, h, w, oc, ks = (case[x] for x in ("N", "C", "H", "W", "OC", "k"))
    oh, ow = _conv_out(case, k == "convt_f32")
    flops = 2 * n * c * oc * ks * ks * (h * w if k == "convt_f32" else oh * ow)
    if k == "qconv":
        ph, pw = (oh // 2, ow // 2) if case["pool"] else (oh, ow)
        return {"bytes": n * (c * h * w * (4 if case["first"] else 1) + oc * ph * pw) + c * oc * ks * ks + 8 * oc, "flops": flops}
    return {"bytes": 4 * (n * (c * h * w + oc * oh * ow) + c * oc * ks * ks + oc), "flops": flops}


def tolerance(case):
    # the integer paths have one right answer; a float output of theirs is one product of an exact int32 and a scale
    if case["kind"] in ("qgemm", "qconv", "qcnn"):
        return "exact"
    # the others: about four times the distance of the results from the same product in 64 bits
    if case["kind"] == "gemm_fp8":
        # e4m3 products summed in fp32 (the matrix instruction drops what lies 2^-14 below the largest of eight: 1.5e-5 seen
        # over K = 4096), then one bf16 rounding, which can fall to either side
        return {"rel": 6e-3, "max": 1.6e-2} if case["out"] == "bf16" else {"rel": 6e-5, "max": 3e-4}
    return {"rel": 7e-6, "max": 5e-5}      # fp32 sums: 2e-7 .. 1.8e-6 seen over K = 147 .. 12544


# ------------------------------------------------------------------------------------------------ states
_stream = None


class State:
    """The context, the tensors and the calls of one model."""

    def __init__(self, seed):
        global _stream
        if _stream is None:
            _stream = torch.cuda.Stream()
        self.ctx = ops.Context(0, guard=False, stream=_stream)
        self.ctx.check(self.ctx.lib.sofie_hip_constant_weights(self.ctx.h, 1))
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.calls, self.keep, self.out = [], [], None

    # -- tensors
    def hold(self, t):
        t = t.contiguous()
        self.keep.append(t)
        return t

    def randn(self, *shape, std=1.0):
        return self.hold(torch.randn(*shape, device="cuda", generator=self.gen) * std)

    def rand(self, *shape, lo=0.0, hi=1.0):
        return self.hold(torch.rand(*shape, device="cuda", generator=self.gen) * (hi - lo) + lo)

    def empty(self, *shape, dtype=torch.float32):
        return self.hold(torch.empty(*shape, device="cuda", dtype=dtype))

    def relu_s8(self, *shape):
        """Quantized activations behind a ReLU: half of them at the zero-point -128, the rest half-normal over the range."""
        x = torch.randn(*shape, device="cuda", generator=self.gen).clamp_(0) * 64.0
        return self.hold((torch.round(x).clamp_(max=255.0) - 128.0).to(torch.int8))

    def quantized_weights(self, *shape):
        """Kaiming-normal weights, symmetric int8 per row of the first dimension; and the rows' scales."""
        w = torch.randn(*shape, device="cuda", generator=self.gen) * (2.0 / math.prod(shape[1:])) ** 0.5
        s = w.reshape(shape[0], -1).abs().amax(1).clamp_(min=1e-6) / 127.0
        q = torch.round(w / s.view(-1, *[1] * (len(shape) - 1))).clamp_(-127, 127).to(torch.int8)
        return self.hold(q), s

    def folded(self, q, bias, s_in, s_w, zp=-128):
        """int32 bias with the input's zero-point folded in, as the emitter stores it."""
        b = torch.round(bias / (s_in * s_w)).to(torch.int64) - zp * q.reshape(q.shape[0], -1).to(torch.int64).sum(1)
        return self.hold(b.to(torch.int32))

    # -- calls
    def call(self, name, *args):
        conv = [a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args]
        self.calls.append((getattr(self.ctx.lib, name), (self.ctx.h, *conv)))


def prepare(case, seed):
    st = State(seed)
    {"mlp": _mlp, "gemm_f32": _gemm_f32, "conv_f32": _conv_f32, "convt_f32": _convt_f32, "cnn_f32": _cnn_f32, "qgemm": _qgemm,
     "gemm_fp8": _gemm_fp8, "qconv": _qconv, "qcnn": _qcnn}[case["kind"]](st, case)
    torch.cuda.synchronize()      # the inputs were made on another stream
    return st


def run(state):
    for fn, args in state.calls:
        rc = fn(*args)
        if rc:
            state.ctx.check(rc)
    return state.out


def _mlp(st, case):
    w = [int(v) for v in case["widths"].split("-")]
    n, b = len(w) - 1, case["batch"]
    x, y = st.randn(b, w[0]), st.empty(b, w[-1])
    W = [st.rand(a, c, lo=-math.sqrt(6.0 / (a + c)), hi=math.sqrt(6.0 / (a + c))) for a, c in zip(w, w[1:])]
    B = [st.randn(c, std=0.05) for c in w[1:]]
    arrays = ((C.c_int * (n + 1))(*w), (C.c_void_p * n)(*[t.data_ptr() for t in W]), (C.c_void_p * n)(*[t.data_ptr() for t in B]),
              (C.c_int * n)(*[L.ACT_RELU] * (n - 1) + [L.ACT_NONE]))
    st.call("sofie_hip_mlp_f32", n, *arrays, x, w[0], y, w[-1], b)
    st.out = y


def _gemm_f32(st, case):
    M, N, K, ta, tb = case["M"], case["N"], case["K"], int(case["transA"]), int(case["transB"])
    A = st.randn(K, M) if ta else st.randn(M, K)
    B = st.randn(N, K, std=K ** -0.5) if tb else st.randn(K, N, std=K ** -0.5)
    bias = st.randn(N, std=0.1) if case["bias"] else None
    y = st.empty(M, N)
    st.call("sofie_hip_gemm_f32", ta, tb, M, N, K, 1.0, A, A.shape[1], B, B.shape[1], 1.0 if case["bias"] else 0.0, bias,
            L.BIAS_ROW if case["bias"] else L.BIAS_NONE, y, N, L.ACT_RELU if case["relu"] else L.ACT_NONE)
    st.out = y


def _conv_call(st, x, w, bias, y, n, c, h, wd, oc, k, s, p):
    st.call("sofie_hip_conv2d_f32", x, w, bias, y, n, c, h, wd, oc, k, k, p, p, p, p, s, s, 1, 1, 1, L.ACT_RELU)


def _conv_f32(st, case):
    n, c, h, wd, oc, k = (case[v] for v in ("N", "C", "H", "W", "OC", "k"))
    oh, ow = _conv_out(case)
    x, w = st.rand(n, c, h, wd), st.randn(oc, c, k, k, std=(2.0 / (c * k * k)) ** 0.5)
    y = st.empty(n, oc, oh, ow)
    _conv_call(st, x, w, st.randn(oc, std=0.1), y, n, c, h, wd, oc, k, case["s"], case["p"])
    st.out = y


def _convt_f32(st, case):
    n, c, h, wd, oc, k, s, p = (case[v] for v in ("N", "C", "H", "W", "OC", "k", "s", "p"))
    oh, ow = _conv_out(case, True)
    x, w = st.rand(n, c, h, wd), st.randn(c, oc, k, k, std=(2.0 * s * s / (c * k * k)) ** 0.5)
    y = st.empty(n, oc, oh, ow)
    st.call("sofie_hip_conv_transpose2d_f32", x, w, st.randn(oc, std=0.1), y, n, c, h, wd, oc, k, k, p, p, s, s, 1, 1, 1, oh, ow,
            L.ACT_NONE)
    st.out = y


def _cnn_f32(st, case):
    b = case["batch"]
    a = st.rand(b, 1, 40, 40)
    for ci, co, hw, pool in CNN_LAYERS:
        y = st.empty(b, co, hw, hw)
        _conv_call(st, a, st.randn(co, ci, 3, 3, std=(2.0 / (9 * ci)) ** 0.5), st.randn(co, std=0.05), y, b, ci, hw, hw, co, 3, 1, 1)
        a = y
        if pool:
            a = st.empty(b, co, hw // 2, hw // 2)
            st.call("sofie_hip_maxpool2d_f32", y, a, b * co, hw, hw, 2, 2, 0, 0, 0, 0, 2, 2)
    for k, n in CNN_FC:
        y = st.empty(b, n)
        st.call("sofie_hip_gemm_f32", 0, 0, b, n, k, 1.0, a, k, st.randn(k, n, std=(2.0 / k) ** 0.5), n, 1.0, st.randn(n, std=0.05),
                L.BIAS_ROW, y, n, L.ACT_RELU if n > 5 else L.ACT_NONE)
        a = y
    st.out = a


def _qgemm(st, case):
    M, N, K, tb = case["M"], case["N"], case["K"], int(case["transB"])
    A = st.hold(torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda", generator=st.gen))
    B = st.hold(torch.randint(-127, 128, (N, K) if tb else (K, N), dtype=torch.int8, device="cuda", generator=st.gen))
    # outputs spread over the int8 range: uniform operands have a root mean square of 73.3
    scale = st.rand(N, lo=20.0 / (73.3 ** 2 * K ** 0.5), hi=60.0 / (73.3 ** 2 * K ** 0.5))
    bias = None
    if case["bias"]:
        bias = st.hold(torch.round(torch.randn(N, device="cuda", generator=st.gen) * (73.3 ** 2 * K ** 0.5)).to(torch.int32))
    y = st.empty(M, N, dtype=torch.int8 if case["out"] == "s8" else torch.float32)
    st.call("sofie_hip_qgemm_s8", tb, M, N, K, A, K, B, B.shape[1], scale, bias, 0, L.ACT_RELU if case["relu"] else L.ACT_NONE, y, N,
            L.OUT_S8 if case["out"] == "s8" else L.OUT_F32)
    st.out = y


def _gemm_fp8(st, case):
    M, N, K, tb = case["M"], case["N"], case["K"], int(case["transB"])

    def e4m3(*shape):
        t = torch.randn(*shape, device="cuda", generator=st.gen)
        s = float(t.abs().max()) / 448.0
        return st.hold((t / s).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)), s
    A, sa = e4m3(M, K)
    B, sb = e4m3(N, K) if tb else e4m3(K, N)
    bias = st.randn(N)
    y = st.empty(M, N, dtype=torch.bfloat16 if case["out"] == "bf16" else torch.float32)
    st.call("sofie_hip_gemm_fp8", tb, M, N, K, A, K, B, B.shape[1], sa, sb, bias, y, N, L.OUT_BF16 if case["out"] == "bf16" else L.OUT_F32)
    st.out = y


def _qconv(st, case):
    n, c, h, wd, oc, k, s, p = (case[v] for v in ("N", "C", "H", "W", "OC", "k", "s", "p"))
    oh, ow = _conv_out(case)
    if case["pool"]:
        oh, ow = oh // 2, ow // 2
    w, sw = st.quantized_weights(oc, k, k, c)
    s_in = 1.0 / 255.0 if case["first"] else 4.0 / 255.0
    scale, bias = st.hold(sw * s_in / (6.0 / 255.0)), st.folded(w, torch.randn(oc, device="cuda", generator=st.gen) * 0.1, s_in, sw)
    y = st.empty(n, oh, ow, oc, dtype=torch.int8)
    geometry = (n, c, h, wd, oc, k, k, p, p, p, p, s, s, 1)
    pool = (2, 2, 2, 2) if case["pool"] else (0, 0, 0, 0)
    if case["first"]:
        st.call("sofie_hip_quantize_qconv2d_s8", st.rand(n, c, h, wd), s_in, -128, w, L.LAYOUT_NHWC, bias, scale, y, L.LAYOUT_NHWC,
                *geometry, -128, L.ACT_RELU, *pool)
    elif case["pool"]:
        st.call("sofie_hip_qconv2d_pool_s8", st.relu_s8(n, h, wd, c), L.LAYOUT_NHWC, w, L.LAYOUT_NHWC, bias, scale, y, L.LAYOUT_NHWC,
                *geometry, -128, -128, L.ACT_RELU, *pool)
    else:
        st.call("sofie_hip_qconv2d_s8", st.relu_s8(n, h, wd, c), L.LAYOUT_NHWC, w, L.LAYOUT_NHWC, bias, scale, y, L.LAYOUT_NHWC,
                *geometry, -128, -128, L.ACT_RELU, L.OUT_S8)
    st.out = y


def _qcnn(st, case):
    b = case["batch"]
    s_act = (1.0 / 255.0, 4.0 / 255.0, 8.0 / 255.0, 12.0 / 255.0, 12.0 / 255.0)      # the ranges the layers' outputs have
    x = st.rand(b, 1, 40, 40)

    def conv(i):
        ci, co, hw, pool = CNN_LAYERS[i]
        w, sw = st.quantized_weights(co, 3, 3, ci)
        bias = st.folded(w, torch.randn(co, device="cuda", generator=st.gen) * 0.05, s_act[i], sw)
        scale = st.hold(sw * s_act[i] / s_act[i + 1])
        o = hw // 2 if pool else hw
        return w, bias, scale, st.empty(b, o, o, co, dtype=torch.int8)
    w, bias, scale, a = conv(0)
    st.call("sofie_hip_quantize_qconv2d_s8", x, s_act[0], -128, w, L.LAYOUT_NHWC, bias, scale, a, L.LAYOUT_NHWC, b, 1, 40, 40, 32, 3, 3,
            1, 1, 1, 1, 1, 1, 1, -128, L.ACT_RELU, 2, 2, 2, 2)
    layers = (L.QConvLayer * 2)()
    head = a
    for d, i in zip(layers, (1, 2)):
        ci, co, hw, pool = CNN_LAYERS[i]
        w, bias, scale, a = conv(i)
        pk = 2 if pool else 0
        for name, v in dict(w=w.data_ptr(), w_layout=L.LAYOUT_NHWC, bias=bias.data_ptr(), scale=scale.data_ptr(), y=a.data_ptr(),
                            y_layout=L.LAYOUT_NHWC, C=ci, H=hw, W=hw, OC=co, KH=3, KW=3, pad_top=1, pad_left=1, pad_bottom=1,
                            pad_right=1, stride_h=1, stride_w=1, groups=1, zp_x=-128, zp_y=-128, act=L.ACT_RELU, pool_kh=pk, pool_kw=pk,
                            pool_stride_h=pk, pool_stride_w=pk).items():
            setattr(d, name, v)
    st.call("sofie_hip_qconv2d_s8_chain", head, L.LAYOUT_NHWC, b, 2, layers)
    (k1, n1), (_, n2) = CNN_FC
    w1, sw1 = st.quantized_weights(n1, k1)
    w2, sw2 = st.quantized_weights(n2, n1)
    q1 = st.folded(w1, torch.randn(n1, device="cuda", generator=st.gen) * 0.05, s_act[3], sw1)
    q2 = st.folded(w2, torch.randn(n2, device="cuda", generator=st.gen) * 0.05, s_act[4], sw2)
    mid, y = st.empty(b, n1, dtype=torch.int8), st.empty(b, n2)
    st.call("sofie_hip_qgemm_s8_pair", b, k1, a, k1, n1, w1, k1, st.hold(sw1 * s_act[3] / s_act[4]), q1, -128, L.ACT_RELU, mid, n1, n2,
            w2, n1, st.hold(sw2 * s_act[4]), q2, 0, L.ACT_NONE, y, n2, L.OUT_F32)
    st.out = y
