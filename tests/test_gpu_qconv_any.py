"""int8 convolutions of any channel counts, kernel sizes, strides, pads and layouts (k_qconv_any): bit-exact against the oracle.

The shapes cover the input read in place (channels-last, C a multiple of 16) with and without pads, the padded copy from
channels-last, channel-plane and float input, the three sizes of workgroup (whole tiles with the weights in LDS, small tiles, K
dealt to four or eight wavefronts), one to four tiles of 16 channels per workgroup and remainders of all of them, and the fused 2x2
pooling with scales of both signs."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle
from sofie_amd import lib as L

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


# N, C, H, W, OC, KH, KW, strides, pads
SHAPES = [
    (1, 16, 5, 5, 16, 3, 3, (1, 1), (1, 1)),        # one tile, in place, every row at a border
    (2, 48, 35, 29, 80, 3, 3, (2, 2), (1, 1)),      # in place, five channel tiles, stride
    (3, 16, 9, 7, 17, 1, 1, (1, 1), (0, 0)),        # one K-step that is a quarter full, no bounds
    (1, 32, 7, 9, 33, 5, 5, (1, 1), (2, 2)),        # K dealt to wavefronts, 13 K-steps
    (1, 1, 6, 5, 8, 3, 3, (1, 1), (1, 1)),          # one channel
    (2, 3, 31, 33, 24, 7, 7, (2, 2), (3, 3)),       # three channels, a kernel row of 28 bytes
    (2, 5, 12, 11, 9, 2, 3, (1, 2), (0, 1)),        # K of 30 bytes, uneven kernel, stride and pads
    (4, 45, 20, 18, 136, 3, 3, (1, 1), (1, 1)),     # 45 channels, nine channel tiles
    (1, 65, 6, 6, 20, 3, 3, (2, 2), (1, 1)),        # pixels rounded up to 80 bytes
    (40, 24, 30, 31, 12, 3, 3, (1, 1), (1, 1)),     # large tiles, one channel tile
    (24, 48, 40, 40, 30, 3, 3, (1, 1), (1, 1)),     # large tiles in place, two channel tiles
    (20, 20, 41, 39, 40, 3, 3, (1, 1), (0, 1)),     # large tiles, three channel tiles
    (20, 64, 41, 39, 61, 5, 5, (1, 1), (2, 2)),     # large tiles, more weights than a third of the LDS
    (9, 128, 33, 33, 100, 7, 7, (1, 1), (3, 3)),    # weights of one channel tile of seven are all that would fit the LDS
    (84, 128, 20, 20, 16, 7, 7, (1, 1), (3, 3)),    # those of one channel tile, which is all there is
    (13, 32, 48, 60, 188, 3, 3, (1, 1), (1, 1)),    # half a round of large tiles, five K-steps
    # the short sums above once more with the pixels from which on they are this kernel's
    (3, 16, 90, 70, 17, 1, 1, (1, 1), (0, 0)),      # one K-step that is a quarter full, no bounds
    (9, 1, 140, 130, 8, 5, 5, (1, 1), (2, 2)),      # one channel
    (20, 5, 62, 61, 9, 2, 3, (1, 2), (0, 1)),       # K of 30 bytes, uneven kernel, stride and pads
    (6, 64, 9, 8, 37, 7, 7, (1, 1), (3, 3)),        # pooled in place, few tiles: K dealt to eight wavefronts
]


def make(r, n, c, h, w, oc, kh, kw, negative):
    x = r.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = r.integers(-127, 128, (oc, c, kh, kw)).astype(np.int8)
    scale = (r.uniform(20.0, 60.0, oc) / (73.3 * 73.3 * np.sqrt(c * kh * kw))).astype(np.float32)
    if negative:
        scale[::3] *= -1.0
    return x, wt, scale, r.integers(-3000, 3000, oc).astype(np.int32)


@pytest.mark.parametrize("shape", SHAPES)
def test_qconv_of_any_shape(ops, shape):
    n, c, h, w, oc, kh, kw, strides, pads = shape
    x, wt, scale, bias = make(np.random.default_rng(c * 100 + oc), n, c, h, w, oc, kh, kw, False)
    want = oracle.qconv2d_s8(x, wt, scale, bias, pads, strides, 1, 7, -9, True)
    kw_ = dict(scale=scale, bias=bias, pads=pads, strides=strides, zpx=7, zpy=-9, relu=True)
    xl, wl = np.ascontiguousarray(x.transpose(0, 2, 3, 1)), np.ascontiguousarray(wt.transpose(0, 2, 3, 1))
    got = ops.qconv2d_s8(xl, wl, x_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC, **kw_)
    assert np.array_equal(got.transpose(0, 3, 1, 2), want)
    assert np.array_equal(ops.qconv2d_s8(x, wt, **kw_), want)


@pytest.mark.parametrize("shape", SHAPES)
def test_qconv_of_any_shape_with_pooling(ops, shape):
    n, c, h, w, oc, kh, kw, strides, pads = shape
    x, wt, scale, bias = make(np.random.default_rng(c * 100 + oc + 1), n, c, h, w, oc, kh, kw, True)
    conv = oracle.qconv2d_s8(x, wt, scale, bias, pads, strides, 1, -128, 3, False)
    xl = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    for pool, step in ((2, 2), (3, 2)):
        if min(conv.shape[2:]) < pool:
            continue
        oh, ow = (conv.shape[2] - pool) // step + 1, (conv.shape[3] - pool) // step + 1
        want = np.max([conv[:, :, i:i + step * (oh - 1) + 1:step, j:j + step * (ow - 1) + 1:step] for i in range(pool) for j in range(pool)], 0)
        got = ops.qconv2d_pool_s8(xl, wt, scale, bias, pads, strides, 1, -128, 3, False, (pool, pool), (step, step),
                                  x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC)
        assert np.array_equal(got.transpose(0, 3, 1, 2), want), pool


@pytest.mark.parametrize("shape", [s for s in SHAPES if s[1] < 48 and s[0] < 40])
def test_float_input_is_quantized_into_the_copy(ops, shape):
    n, c, h, w, oc, kh, kw, strides, pads = shape
    r = np.random.default_rng(c + oc)
    _, wt, scale, bias = make(r, n, c, h, w, oc, kh, kw, False)
    x = r.uniform(-0.2, 1.3, (n, c, h, w)).astype(np.float32)
    q = oracle.quantize_f32_s8(x, 1.0 / 255.0, -128)
    want = oracle.qconv2d_s8(q, wt, scale, bias, pads, strides, 1, -128, -128, True)
    got = ops.quantize_qconv2d_s8(x, 1.0 / 255.0, -128, wt, scale, bias, pads, strides, 1, -128, True, y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(got.transpose(0, 3, 1, 2), want)


@pytest.mark.parametrize("shape,kernels", [((8, 9, 11, 11, 85, 1, 1), ("k_qconv_simple", "k_qconv_simple")),
                                           ((2, 9, 12, 12, 50, 3, 3), ("k_qconv_any", "k_qconv_any")),
                                           ((1, 6, 10, 10, 20, 3, 3), ("k_qconv_simple", "k_qconv_any")),
                                           ((1, 16, 14, 14, 32, 3, 3), ("k_qconv_any", "k_qconv_any"))])
def test_small_layers_take_the_shorter_way(ops, shape, kernels):
    """The kernel of a small layer without and with kept weights, at the second call; bytes against the oracle."""
    n, c, h, w, oc, kh, kw = shape
    p = kh // 2
    x, wt, scale, bias = make(np.random.default_rng(c), n, c, h, w, oc, kh, kw, False)
    want = oracle.qconv2d_s8(x, wt, scale, bias, (p, p), (1, 1), 1, 0, -9, False).transpose(0, 2, 3, 1)
    for promise, kernel in zip((0, 1), kernels):
        ctx = ops.Context(0)
        assert ctx.lib.sofie_hip_constant_weights(ctx.h, promise) == 0
        xd, wd = ctx.dev(np.ascontiguousarray(x.transpose(0, 2, 3, 1))), ctx.dev(np.ascontiguousarray(wt.transpose(0, 2, 3, 1)))
        sd, bd, y = ctx.dev(scale), ctx.dev(bias), ctx.empty(want.shape, torch.int8)
        buf, m = C.create_string_buffer(4096), C.c_int(-1)
        for _ in range(2):
            ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
            ctx.check(ctx.lib.sofie_hip_qconv2d_s8(ctx.h, ctx.ptr(xd), L.LAYOUT_NHWC, ctx.ptr(wd), L.LAYOUT_NHWC, ctx.ptr(bd), ctx.ptr(sd), ctx.ptr(y),
                                                   L.LAYOUT_NHWC, n, c, h, w, oc, kh, kw, p, p, p, p, 1, 1, 1, 0, -9, L.ACT_NONE, L.OUT_S8))
            ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(m)))
            ctx.sync()
            assert np.array_equal(y.cpu().numpy(), want)
        assert [line.split()[0] for line in buf.value.decode().splitlines()][-1] == kernel
        ctx.close()


@pytest.mark.parametrize("promise", [0, 1])
@pytest.mark.parametrize("warm", [False, True])
def test_recorded_calls(ops, promise, warm):
    """A call recorded on a fresh context (no scratch buffer exists and none may be made: the plain kernel runs) and on one
    that has made the call before (the buffer and, under the promise, the copy of the weights exist); every replay gives
    the oracle's bytes."""
    n, c, h, w, oc, kh, kw, strides, pads = 2, 21, 17, 19, 35, 3, 3, (1, 1), (1, 1)
    x, wt, scale, bias = make(np.random.default_rng(5), n, c, h, w, oc, kh, kw, False)
    want = oracle.qconv2d_s8(x, wt, scale, bias, pads, strides, 1, 0, 0, False)
    ctx = ops.Context(0, stream=torch.cuda.Stream())
    assert ctx.lib.sofie_hip_constant_weights(ctx.h, promise) == 0
    xd, wd, sd, bd, y = ctx.dev(x), ctx.dev(wt), ctx.dev(scale), ctx.dev(bias), ctx.empty(want.shape, torch.int8)
    torch.cuda.synchronize()

    def call():
        return ctx.lib.sofie_hip_qconv2d_s8(ctx.h, ctx.ptr(xd), L.LAYOUT_NCHW, ctx.ptr(wd), L.LAYOUT_NCHW, ctx.ptr(bd), ctx.ptr(sd),
                                            ctx.ptr(y), L.LAYOUT_NCHW, n, c, h, w, oc, kh, kw, 1, 1, 1, 1, 1, 1, 1, 0, 0, L.ACT_NONE,
                                            L.OUT_S8)
    for _ in range(2 if warm else 0):
        y.zero_()
        torch.cuda.synchronize()
        ctx.check(call())
        ctx.sync()
        assert np.array_equal(y.cpu().numpy(), want)
    graph = C.c_void_p()
    ctx.check(ctx.lib.sofie_hip_capture_begin(ctx.h))
    rc = call()
    ctx.check(ctx.lib.sofie_hip_capture_end(ctx.h, C.byref(graph)))
    ctx.check(rc)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        ctx.check(ctx.lib.sofie_hip_graph_launch(ctx.h, graph))
        ctx.sync()
        assert np.array_equal(y.cpu().numpy(), want)
    ctx.check(ctx.lib.sofie_hip_graph_destroy(ctx.h, graph))
    ctx.close()


@pytest.mark.parametrize("steps", [1, 3, 4, 5, 15, 16, 17, 32, 33])
@pytest.mark.parametrize("n,h,w,oc", [(1, 5, 9, 7), (3, 20, 23, 40), (9, 22, 25, 72)])
@pytest.mark.parametrize("pool", [False, True])
def test_few_tiles_by_steps_of_k(ops, steps, n, h, w, oc, pool):
    """Weights from memory: K of up to as many steps as a wavefront requests at once, and of one more, dealt to one, four and eight."""
    c = 64 * steps - 16 * (steps % 2)
    x, wt, scale, bias = make(np.random.default_rng(steps + oc), n, c, h, w, oc, 1, 1, pool)
    want = oracle.qconv2d_s8(x, wt, scale, bias, (0, 0), (1, 1), 1, 7, -9, False)
    xl, wl = np.ascontiguousarray(x.transpose(0, 2, 3, 1)), np.ascontiguousarray(wt.transpose(0, 2, 3, 1))
    if pool:
        oh, ow = h // 2, w // 2
        want = np.max([want[:, :, i:2 * oh:2, j:2 * ow:2] for i in (0, 1) for j in (0, 1)], 0)
        got = ops.qconv2d_pool_s8(xl, wt, scale, bias, (0, 0), (1, 1), 1, 7, -9, False, (2, 2), (2, 2), x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC)
    else:
        got = ops.qconv2d_s8(xl, wl, x_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC, scale=scale, bias=bias,
                             pads=(0, 0), strides=(1, 1), zpx=7, zpy=-9, relu=False)
    assert np.array_equal(got.transpose(0, 3, 1, 2), want)
