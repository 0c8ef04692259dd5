"""fp32 convolutions of one to nine products per output on k_conv_f32_short: every number of products, strides, dilations, uneven pads, groups,
odd planes, a last channel block that is not full, against float64; values that are not finite."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


def names_of(ctx, call):
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
    out = call()
    ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
    ctx.sync()
    return out, [line.split()[0] for line in buf.value.decode().splitlines()]


# N, C, H, W, OC, KH, KW, stride, (top, left, bottom, right), dilation, groups
CONV = [
    (256, 1, 40, 40, 32, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),       # the float classifier's first layer
    (84, 1, 111, 109, 70, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1),
    (90, 1, 91, 53, 67, 2, 1, (1, 2), (1, 0, 1, 0), (3, 1), 1),        # odd planes, dilated rows, a last block of three channels
    (61, 3, 64, 61, 65, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1),
    (40, 8, 80, 72, 40, 2, 1, (1, 1), (0, 1, 1, 0), (1, 1), 4),        # groups of ten channels, pads on one side
    (200, 5, 30, 62, 33, 1, 1, (2, 1), (0, 0, 0, 0), (1, 1), 1),
    (300, 1, 23, 40, 130, 2, 3, (1, 1), (1, 2, 0, 1), (1, 2), 1),
    (100, 7, 50, 50, 50, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1),
    (150, 2, 47, 33, 90, 2, 2, (1, 1), (1, 1, 1, 1), (1, 1), 1),
    (3000, 1, 3, 7, 129, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),       # a wavefront's pixels on many images
    (2, 9, 301, 303, 100, 1, 1, (1, 1), (0, 0, 0, 0), (1, 1), 1),
    (8, 1, 64, 64, 165, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),        # two pixels per lane (four above), stores through the L2
]


@pytest.mark.parametrize("shape", CONV)
def test_short_sums(ops, shape):
    """Nine products summed in fp32: 9 roundings of 2^-24 on the sum of the absolute products."""
    n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
    t, l, b, r = pads
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    x = torch.randn(n, c, h, w, device="cuda", generator=g)
    wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g)
    bias = torch.randn(oc, device="cuda", generator=g)
    torch.cuda.synchronize()
    for relu in (False, True):
        ctx = ops.Context(0)
        y, names = names_of(ctx, lambda: ops.conv2d_f32(x, wt, bias if relu else None, pads, s, d, groups, relu=relu, ctx=ctx))
        assert names == ["k_conv_f32_short"], names
        pad = torch.nn.functional.pad(x.cpu().double(), (l, r, t, b))
        ref = torch.nn.functional.conv2d(pad, wt.cpu().double(), bias.cpu().double() if relu else None, s, 0, d, groups)
        size = torch.nn.functional.conv2d(pad.abs(), wt.cpu().double().abs(), bias.cpu().double().abs() if relu else None, s, 0, d, groups)
        ref = ref.clamp(min=0) if relu else ref
        assert bool(((y.cpu().double() - ref).abs() <= 10 * 2.0 ** -24 * size).all())
        ctx.close()


def test_values_that_are_not_finite_stay_in_their_windows(ops):
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(300, 1, 40, 39, generator=g), torch.randn(40, 1, 3, 3, generator=g)
    x[3, 0, 4, 7], x[3, 0, 39, 38], x[9, 0, 0, 13], x[299, 0, 39, 0] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[7, 0, 2, 2], w[39, 0, 0, 0], w[11] = 1e38, float("inf"), 0.0
    ref = torch.nn.functional.conv2d(torch.nn.functional.pad(x, (1, 1, 1, 1)), w)
    xd, wd = x.cuda(), w.cuda()
    torch.cuda.synchronize()
    ctx = ops.Context(0)
    y, names = names_of(ctx, lambda: ops.conv2d_f32(xd, wd, None, (1, 1), (1, 1), (1, 1), 1, False, ctx=ctx))
    assert names == ["k_conv_f32_short"]
    y = y.cpu()
    ctx.close()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(torch.sign(y[~fin & ~torch.isnan(ref)]), torch.sign(ref[~fin & ~torch.isnan(ref)]))
