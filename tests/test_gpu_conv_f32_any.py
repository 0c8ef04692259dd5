"""fp32 convolutions of any channels, kernels, strides, dilations, groups and pads, and transposed ones, against float64: every
form of k_conv_f32_any (16 to 96 channels x 16 or 32 pixels per wavefront, K shared by one to eight wavefronts, the three kinds of
stores), the tables of all taps, of four channels' taps and of finished offsets, and kernels it leaves to k_conv2d_f32."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


@pytest.fixture(scope="module")
def kept(ops):
    """A context that keeps its weights in the kernels' layouts: small layers run on k_conv_f32_any there, too."""
    ctx = ops.Context(0)
    ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, 1))
    yield ctx
    ctx.close()


# N, C, H, W, OC, KH, KW, stride, (top, left, bottom, right), dilation, groups
CONV = [
    (1, 1, 1, 1, 1, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1),          # one value
    (1, 3, 5, 5, 16, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),         # 27 k: the last step is not full
    (2, 61, 15, 15, 12, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),      # K over eight wavefronts, all taps in one table
    (3, 75, 9, 7, 33, 3, 3, (2, 1), (1, 0, 0, 2), (1, 1), 1),        # blocks of four channels, the last of three; uneven pads
    (2, 130, 6, 6, 20, 7, 7, (1, 1), (3, 3, 3, 3), (1, 1), 1),       # windows larger than the image
    (5, 8, 17, 13, 24, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1),       # no bounds
    (4, 24, 30, 31, 48, 1, 1, (2, 3), (0, 0, 0, 0), (1, 1), 1),
    (2, 12, 20, 18, 30, 3, 2, (1, 1), (2, 1, 2, 1), (2, 3), 3),      # groups, dilations
    (3, 16, 11, 10, 16, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 16),     # depthwise
    (1, 2, 1, 70, 5, 1, 15, (1, 2), (0, 7, 0, 7), (1, 1), 1),        # the widest kernel
    (1, 2, 1, 70, 5, 1, 16, (1, 1), (0, 8, 0, 7), (1, 1), 1),        # one wider: the general kernel
    (1, 2, 40, 3, 5, 16, 2, (1, 1), (8, 0, 8, 1), (1, 1), 1),
    (16, 5, 41, 43, 17, 5, 5, (1, 1), (2, 2, 2, 2), (1, 1), 1),
    (40, 16, 33, 35, 64, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),     # pixels run on across images
    (64, 20, 31, 33, 81, 3, 3, (1, 1), (0, 1, 0, 1), (1, 1), 1),
    (70, 70, 28, 28, 128, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),    # the largest tiles
    (50, 9, 50, 51, 96, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),
]


def close(y, ref):
    """1e-5 of the largest output: sums of fp32 products in another order differ by about sqrt(K) 2^-24 of the terms' root
    mean square times sqrt(K)."""
    return float((y.double() - ref).abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("shape", CONV)
def test_conv_of_any_kind(ops, kept, shape):
    n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
    g = torch.Generator(device="cuda").manual_seed(n * 1000 + c * 10 + oc)
    x = torch.randn(n, c, h, w, device="cuda", generator=g)
    wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * (c // groups * kh * kw) ** -0.5
    bias = torch.randn(oc, device="cuda", generator=g)
    torch.cuda.synchronize()
    t, l, b, r = pads
    ref = torch.nn.functional.conv2d(torch.nn.functional.pad(x.cpu().double(), (l, r, t, b)), wt.cpu().double(), None, s, 0, d, groups)
    for ctx in (ops.default_context(), kept):
        y = ops.conv2d_f32(x, wt, bias, pads, s, d, groups, relu=True, ctx=ctx)
        z = ops.conv2d_f32(x, wt, None, pads, s, d, groups, ctx=ctx)
        ctx.sync()
        assert close(z.cpu(), ref)
        assert close(y.cpu(), (ref + bias.cpu().double()[:, None, None]).clamp(min=0))
    kept.check(kept.lib.sofie_hip_constant_weights(kept.h, 0))      # this tensor's memory is freed
    kept.check(kept.lib.sofie_hip_constant_weights(kept.h, 1))


# N, C, H, W, OC/groups, KH, KW, stride, (top, left, bottom, right), dilation, groups, output padding
CONVT = [
    (1, 1, 1, 1, 1, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1, (0, 0)),
    (2, 7, 6, 5, 19, 3, 3, (2, 2), (1, 1, 1, 1), (1, 1), 1, (0, 0)),     # phases of one, two and four taps
    (2, 7, 6, 5, 19, 3, 3, (2, 2), (1, 1, 1, 1), (1, 1), 1, (1, 1)),
    (3, 30, 9, 8, 32, 4, 4, (2, 2), (1, 1, 1, 1), (1, 1), 1, (0, 0)),
    (2, 18, 5, 7, 10, 2, 2, (2, 2), (0, 0, 0, 0), (1, 1), 2, (0, 0)),    # groups, one tap per phase
    (2, 9, 5, 7, 10, 5, 4, (3, 3), (2, 0, 1, 1), (1, 1), 1, (0, 0)),     # nine phases: a launch each
    (2, 9, 5, 7, 10, 3, 3, (1, 1), (1, 1, 1, 1), (2, 2), 1, (0, 0)),     # unit stride
    (1, 4, 5, 7, 6, 3, 3, (2, 2), (1, 1, 1, 1), (2, 2), 1, (0, 0)),      # stride and dilation: the general kernel
    (30, 40, 20, 21, 70, 3, 3, (2, 2), (1, 1, 1, 1), (1, 1), 1, (0, 0)),
]


@pytest.mark.parametrize("shape", CONVT)
def test_conv_transpose_of_any_kind(ops, kept, shape):
    n, c, h, w, ocg, kh, kw, s, pads, d, groups, extra = shape
    g = torch.Generator(device="cuda").manual_seed(n * 1000 + c * 10 + ocg)
    x = torch.randn(n, c, h, w, device="cuda", generator=g)
    wt = torch.randn(c, ocg, kh, kw, device="cuda", generator=g) * (c // groups * kh * kw) ** -0.5
    bias = torch.randn(ocg * groups, device="cuda", generator=g)
    torch.cuda.synchronize()
    ys = []
    for ctx in (ops.default_context(), kept):
        ys.append(ops.conv_transpose2d_f32(x, wt, bias, pads, s, d, groups, extra, ctx=ctx))
        ctx.sync()
    kept.check(kept.lib.sofie_hip_constant_weights(kept.h, 0))      # this tensor's memory is freed
    kept.check(kept.lib.sofie_hip_constant_weights(kept.h, 1))
    full = torch.nn.functional.conv_transpose2d(x.cpu().double(), wt.cpu().double(), bias.cpu().double(), s, 0, 0, groups, d)
    full = torch.nn.functional.pad(full, (0, max(0, extra[1] - pads[3]), 0, max(0, extra[0] - pads[2])))
    if full.shape != (n, ocg * groups, s[0] * (h - 1) + d[0] * (kh - 1) + 1, s[1] * (w - 1) + d[1] * (kw - 1) + 1):
        full[:, :, s[0] * (h - 1) + d[0] * (kh - 1) + 1:] = bias.cpu().double()[:, None, None]
        full[:, :, :, s[1] * (w - 1) + d[1] * (kw - 1) + 1:] = bias.cpu().double()[:, None, None]
    for y in ys:
        assert close(y.cpu(), full[:, :, pads[0]:pads[0] + y.shape[2], pads[1]:pads[1] + y.shape[3]])


# (shape as above), the last kernel of a second call without and with kept weights
ROUTES = [
    ((1, 10, 28, 28, 10, 1, 1, 1), ("k_conv2d_f32", "k_conv_f32_any")),              # one launch against a pass over the weights and one
    ((16, 3, 32, 32, 24, 3, 3, 1), ("k_conv2d_f32", "k_conv_f32_any")),
    ((1, 256, 14, 14, 256, 3, 3, 256), ("k_conv2d_f32", "k_conv_f32_any")),
    ((1, 33, 33, 33, 33, 3, 3, 1), ("k_conv_f32_any", "k_conv_f32_any")),            # a long sum: the pass pays
    ((32, 5, 60, 60, 40, 3, 3, 1), ("k_conv_f32_any", "k_conv_f32_any")),            # many tiles
    # short sums on an even number of channels
    ((55, 16, 60, 60, 64, 3, 3, 1), ("k_conv2d_f32_dma_pairs", "k_conv2d_f32_dma_pairs")),
    ((1, 10, 101, 101, 64, 3, 3, 1), ("k_conv_f32_split_finish", "k_conv_f32_any")),
]


@pytest.mark.parametrize("shape,kernels", ROUTES)
def test_layers_take_the_shorter_way(ops, shape, kernels):
    n, c, h, w, oc, kh, kw, groups = shape
    g = torch.Generator(device="cuda").manual_seed(n * 1000 + c * 10 + oc)
    x, wt = torch.randn(n, c, h, w, device="cuda", generator=g), torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g)
    torch.cuda.synchronize()
    ref = torch.nn.functional.conv2d(x.cpu().double(), wt.cpu().double(), None, 1, kh // 2, 1, groups)
    buf, m = C.create_string_buffer(4096), C.c_int(-1)
    for promise, kernel in zip((0, 1), kernels):
        ctx = ops.Context(0)
        ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, promise))
        for _ in range(2):
            ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
            y = ops.conv2d_f32(x, wt, None, (kh // 2, kh // 2), (1, 1), (1, 1), groups, ctx=ctx)
            ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(m)))
            ctx.sync()
            assert close(y.cpu(), ref)
        assert [line.split()[0] for line in buf.value.decode().splitlines()][-1] == kernel
        ctx.close()


@pytest.mark.parametrize("shape,kernels", [((5, 3, 20, 20, 12, 3, 2), ("k_conv2d_f32_phases", "k_conv_f32_any")),
                                           ((5, 61, 20, 20, 12, 3, 2), ("k_conv_f32_any", "k_conv_f32_any")),
                                           ((9, 1, 39, 16, 16, 4, 1), ("k_conv2d_f32", "k_conv_f32_any")),
                                           ((5, 3, 65, 64, 4, 3, 3), ("k_conv2d_f32", "k_conv_f32_any"))])
def test_transposed_layers_take_the_shorter_way(ops, shape, kernels):
    n, c, h, w, oc, k, s = shape
    g = torch.Generator(device="cuda").manual_seed(c)
    x, wt = torch.randn(n, c, h, w, device="cuda", generator=g), torch.randn(c, oc, k, k, device="cuda", generator=g)
    torch.cuda.synchronize()
    ref = torch.nn.functional.conv_transpose2d(x.cpu().double(), wt.cpu().double(), None, s, 1)
    buf, m = C.create_string_buffer(4096), C.c_int(-1)
    for promise, kernel in zip((0, 1), kernels):
        ctx = ops.Context(0)
        ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, promise))
        for _ in range(2):
            ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
            y = ops.conv_transpose2d_f32(x, wt, None, (1, 1, 1, 1), (s, s), (1, 1), 1, (0, 0), ctx=ctx)
            ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(m)))
            ctx.sync()
            assert close(y.cpu(), ref)
        assert [line.split()[0] for line in buf.value.decode().splitlines()][-1] == kernel
        ctx.close()


def test_a_value_outside_the_sum_stays_outside(ops):
    """Infinities and NaN in one image and channel plane reach the outputs whose windows hold them, and no others: taps outside
    the image, steps behind K and channels of another block ask for nothing."""
    x = torch.zeros(3, 75, 9, 9)
    x[1, 74, 8, 8], x[1, 3, 0, 0] = float("inf"), float("nan")
    w = torch.ones(17, 75, 3, 3)
    y = ops.conv2d_f32(x.numpy(), w.numpy(), None, (1, 1))
    ref = torch.nn.functional.conv2d(x, w, None, 1, 1)
    assert torch.equal(torch.isnan(torch.from_numpy(y)), torch.isnan(ref)) and torch.equal(torch.isinf(torch.from_numpy(y)), torch.isinf(ref))


@pytest.mark.parametrize("n,c,h,w,oc,k", [(40, 32, 56, 56, 128, 3), (40, 30, 56, 56, 70, 3), (90, 33, 40, 40, 32, 1), (300, 8, 20, 20, 20, 5)])
def test_many_rounds_of_workgroups_store_whole_numbers(ops, n, c, h, w, oc, k):
    """Many wavefronts per SIMD and several 16 x 16 pieces stored one behind the other, four pixels at a time: sums of small whole
    numbers, which fp32 holds exactly, every value of every image compared."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randint(-3, 4, (n, c, h, w), device="cuda", generator=g).float()
    wt = torch.randint(-3, 4, (oc, c, k, k), device="cuda", generator=g).float()
    torch.cuda.synchronize()
    y = ops.conv2d_f32(x, wt, None, (k // 2, k // 2))
    ops.default_context().sync()
    for i in range(0, n, 10):
        assert torch.equal(y[i:i + 10].cpu(), torch.nn.functional.conv2d(x[i:i + 10].cpu(), wt.cpu(), None, 1, k // 2)), i


def test_constant_weights_and_repeated_calls_give_the_same_bits(ops):
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = torch.randn(2, 70, 9, 9, device="cuda", generator=g), torch.randn(40, 70, 3, 3, device="cuda", generator=g)
    torch.cuda.synchronize()
    once = ops.conv2d_f32(x, w, None, (1, 1)).clone()
    ops.default_context().sync()
    ctx = ops.Context(0)
    ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, 1))
    for _ in range(2):
        y = ops.conv2d_f32(x, w, None, (1, 1), ctx=ctx)
        ctx.sync()
        assert torch.equal(y, once)
    ctx.close()
