"""fp32 convolutions of few channels and a large kernel on k_conv_f32_split, a row of the kernel as a cell: strides, dilations, uneven pads,
groups, kernels of four to eight columns, ragged planes and channels, against float64; values that are not finite."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


@pytest.fixture()
def kept(ops):
    ctx = ops.Context(0)
    ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, 1))
    yield ctx
    ctx.close()


def names_of(ctx, call):
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
    out = call()
    ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
    ctx.sync()
    return out, [line.split()[0] for line in buf.value.decode().splitlines()]


# N, C, H, W, OC, KH, KW, stride, (top, left, bottom, right), dilation, groups
CONV = [
    (16, 3, 224, 224, 64, 7, 7, (2, 2), (3, 3, 3, 3), (1, 1), 1),
    (60, 1, 64, 64, 90, 7, 7, (1, 1), (3, 3, 3, 3), (1, 1), 1),        # one channel: seven chunks
    (50, 3, 61, 47, 33, 7, 7, (1, 1), (3, 3, 3, 3), (1, 1), 1),        # odd planes, one channel behind a block of 32
    (40, 4, 50, 70, 40, 5, 8, (1, 2), (2, 3, 2, 4), (2, 1), 1),        # eight columns, every other column, dilated rows
    (40, 5, 80, 72, 17, 6, 6, (1, 1), (0, 5, 3, 1), (1, 2), 1),        # dilated columns, uneven pads
    (30, 8, 90, 40, 64, 9, 7, (1, 1), (4, 3, 4, 3), (1, 1), 2),        # groups of four channels
    (200, 3, 9, 130, 70, 7, 8, (1, 1), (3, 3, 3, 4), (1, 1), 1),       # images of little more than a tile
]


@pytest.mark.parametrize("shape", CONV)
def test_rows_as_cells(ops, kept, shape):
    """Products of split numbers lose at most 2^-24 each (2^-27 in the mean), sums are rounded once per 32 k: 1e-5 of the largest output as for the other fp32
    kernels, 3e-7 in the 2-norm."""
    n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
    t, l, b, r = pads
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    x = torch.randn(n, c, h, w, device="cuda", generator=g)
    wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * (c // groups * kh * kw) ** -0.5
    bias = torch.randn(oc, device="cuda", generator=g)
    torch.cuda.synchronize()
    for ctx in (kept, ops.Context(0)):
        y, names = names_of(ctx, lambda: ops.conv2d_f32(x, wt, bias, pads, s, d, groups, relu=ctx is kept, ctx=ctx))
        assert "k_conv_f32_split" in names or ctx is not kept, names
        for i in sorted({0, n // 3, n // 2, n - 1}):
            ref = torch.nn.functional.conv2d(torch.nn.functional.pad(x[i:i + 1].cpu().double(), (l, r, t, b)), wt.cpu().double(), bias.cpu().double(), s, 0, d, groups)
            ref = ref.clamp(min=0) if ctx is kept else ref
            err = y[i:i + 1].cpu().double() - ref
            assert float(err.abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())), i
            assert "k_conv_f32_split" not in names or float(err.norm()) <= 3e-7 * float(ref.norm()), i


@pytest.mark.parametrize("shape", CONV)
def test_sums_that_are_repeated(ops, kept, shape):
    """Operands of 2^60: every sum passes 2^95 on the way and is formed again with fp32 instructions from the operands as they were given. A
    rounding of 2^-24 for each of K products, which add as their square root."""
    n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
    t, l, b, r = pads
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    products = c // groups * kh * kw
    x = torch.randn(n, c, h, w, device="cuda", generator=g) * 2.0 ** 60
    wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * products ** -0.5 * 2.0 ** 60
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv2d_f32(x, wt, None, pads, s, d, groups, ctx=kept))
    assert "k_conv_f32_split" in names, names
    for i in sorted({0, n // 2, n - 1}):
        conv = lambda a, v: torch.nn.functional.conv2d(torch.nn.functional.pad(a, (l, r, t, b)), v, None, s, 0, d, groups)
        xi, wi = x[i:i + 1].cpu().double(), wt.cpu().double()
        assert bool(((y[i:i + 1].cpu().double() - conv(xi, wi)).abs() <= products ** 0.5 * 2.0 ** -24 * conv(xi.abs(), wi.abs())).all()), i


def test_values_that_are_not_finite_stay_in_their_windows(ops, kept):
    """The eighth value of a cell, a column the kernel does not have, is no factor: an infinity there leaves the pixel alone."""
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(40, 3, 64, 60, generator=g), torch.randn(70, 3, 7, 7, generator=g)
    x[3, 0, 4, 7], x[3, 2, 63, 59], x[9, 1, 0, 13], x[39, 2, 63, 0] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[:, 2] = w[:, 2].clamp(-0.5, 0.5)
    w[7, 1, 2, 2], w[69, 0, 6, 6], w[11] = 1e38, float("inf"), 0.0
    ref = torch.nn.functional.conv2d(torch.nn.functional.pad(x, (3, 3, 3, 3)), w)
    xd, wd = x.cuda(), w.cuda()
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv2d_f32(xd, wd, None, (3, 3), (1, 1), (1, 1), 1, False, ctx=kept))
    assert names[-1] == "k_conv_f32_split"
    y = y.cpu()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(torch.sign(y[~fin & ~torch.isnan(ref)]), torch.sign(ref[~fin & ~torch.isnan(ref)]))
    zeros = torch.zeros(())
    scale = torch.nn.functional.conv2d(torch.where(torch.isfinite(x), x, zeros).abs().double(), torch.where(torch.isfinite(w), w, zeros).abs().double(), None, 1, 3)
    assert bool(((y.double() - ref.double()).abs()[fin] <= 1e-5 * scale[fin] + 1e-30).all())
