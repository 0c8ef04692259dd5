"""fp32 convolutions on k_conv_f32_split (operands as three bf16 numbers): every tile size, slots of 16 and 32 channels, steps that reach
into the next slot, strips, groups, phases and ragged ends, against float64; error against the fp32 instructions'; values that are
not finite."""
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
    """A context that keeps its weights in the kernels' layouts."""
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
    (64, 64, 56, 56, 128, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),      # 128 channels x 128 pixels, tiles end with an image
    (120, 32, 20, 20, 64, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),      # pixels run on across images
    (256, 64, 10, 10, 128, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),
    (90, 35, 41, 37, 70, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),       # odd planes (4-byte stores), three channels of the last eight
    (64, 51, 40, 64, 93, 5, 5, (1, 1), (2, 2, 2, 2), (1, 1), 1),       # 96 channels
    (17, 64, 168, 38, 28, 7, 7, (1, 1), (3, 3, 3, 3), (1, 1), 1),      # 32 channels, 49 taps
    (16, 64, 32, 32, 65, 7, 7, (1, 1), (3, 3, 3, 3), (1, 1), 1),       # one channel behind two blocks of 32
    (7, 64, 158, 64, 231, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),
    (5, 16, 58, 58, 192, 5, 5, (1, 1), (2, 2, 2, 2), (1, 1), 1),       # a slot and nothing else
    (192, 12, 16, 64, 66, 5, 5, (1, 1), (2, 2, 2, 2), (1, 1), 1),      # part of a slot
    (64, 64, 56, 40, 128, 3, 3, (2, 1), (1, 1, 1, 1), (1, 1), 1),      # every other row
    (20, 90, 60, 61, 96, 3, 3, (1, 1), (2, 0, 1, 3), (2, 3), 2),       # groups, dilations, uneven pads
    (30, 128, 30, 225, 64, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1),     # wide rows in strips, the last one short
    (300, 24, 7, 5, 160, 5, 4, (1, 1), (2, 2, 2, 1), (1, 1), 1),       # images smaller than a tile
]


def reference(x, w, bias, s, pads, d, groups):
    t, l, b, r = pads
    return torch.nn.functional.conv2d(torch.nn.functional.pad(x.cpu().double(), (l, r, t, b)), w.cpu().double(), bias.cpu().double(), s, 0, d, groups)


@pytest.mark.parametrize("shape", CONV)
def test_conv_in_three_parts(ops, kept, shape):
    """Products of split numbers lose at most 2^-24 each (2^-27 in the mean) and sums are rounded once per 32 k at their own size, where fp32
    products in a row are rounded K times: 1e-5 of the largest output, as for the other fp32 kernels, and 3e-7 in the 2-norm (they show up to
    1e-6 at these K)."""
    n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    x = torch.randn(n, c, h, w, device="cuda", generator=g)
    wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * (c // groups * kh * kw) ** -0.5
    bias = torch.randn(oc, device="cuda", generator=g)
    torch.cuda.synchronize()
    for ctx in (kept, ops.Context(0)):
        y, names = names_of(ctx, lambda: ops.conv2d_f32(x, wt, bias, pads, s, d, groups, relu=ctx is kept, ctx=ctx))
        assert "k_conv_f32_split" in names or ctx is not kept, names
        # some images, the first and the last among them
        for i in sorted({0, n // 3, n // 2, n - 1}):
            ref = reference(x[i:i + 1], wt, bias, s, pads, d, groups)
            ref = ref.clamp(min=0) if ctx is kept else ref
            err = y[i:i + 1].cpu().double() - ref
            assert float(err.abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())), i
            assert "k_conv_f32_split" not in names or float(err.norm()) <= 3e-7 * float(ref.norm()), i


# Layers of stride 2 in slots of eight channels (tests/test_conv_f32_split_plan.py: where the kernel takes them, it is in these): an odd number of chunks in a slot (9, 25, 49), an even one; one slot, several, the last one in part
EIGHTS = [
    (33, 128, 99, 99, 128, 3, 3, (2, 2), (1, 1, 1, 1), (1, 1), 1), (60, 48, 37, 37, 112, 3, 3, (2, 2), (1, 1, 1, 1), (1, 1), 1),
    (46, 61, 40, 64, 27, 5, 5, (2, 2), (2, 2, 2, 2), (1, 1), 1), (48, 81, 144, 11, 190, 7, 7, (2, 2), (3, 3, 3, 3), (1, 1), 1),
    (64, 120, 64, 60, 128, 4, 4, (2, 2), (1, 1, 2, 1), (1, 1), 1), (40, 96, 33, 50, 96, 5, 5, (2, 1), (2, 2, 2, 2), (1, 1), 2),
    (224, 8, 57, 57, 48, 5, 5, (2, 2), (2, 2, 2, 2), (1, 1), 1), (30, 40, 60, 60, 64, 5, 5, (2, 2), (3, 2, 2, 3), (1, 2), 1)]


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("shape", EIGHTS)
def test_strided_layers_in_slots_of_eight(ops, kept, shape, large):
    """Bounds as above; operands of 2^60, whose sums are formed again in fp32, a rounding for each product."""
    n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    big, products = 2.0 ** 60 if large else 1.0, c // groups * kh * kw
    x = torch.randn(n, c, h, w, device="cuda", generator=g) * big
    wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * products ** -0.5 * big
    zero = torch.zeros(oc, device="cuda")
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv2d_f32(x, wt, None, pads, s, d, groups, ctx=kept))
    assert "k_conv_f32_split" in names, names
    for i in sorted({0, n // 2, n - 1}):
        ref = reference(x[i:i + 1], wt, zero, s, pads, d, groups)
        err = y[i:i + 1].cpu().double() - ref
        if large:
            assert bool((err.abs() <= products ** 0.5 * 2.0 ** -24 * reference(x[i:i + 1].abs(), wt.abs(), zero, s, pads, d, groups)).all()), i
        else:
            assert float(err.abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())) and float(err.norm()) <= 3e-7 * float(ref.norm()), i


@pytest.mark.parametrize("n,c,h,w,oc,k,s", [(64, 128, 28, 28, 64, 4, 2), (30, 143, 32, 34, 181, 4, 2), (30, 64, 26, 15, 93, 4, 2),
                                            (60, 87, 19, 21, 40, 3, 2), (64, 120, 20, 20, 90, 3, 1)])
def test_transposed_conv_in_three_parts(ops, kept, n, c, h, w, oc, k, s):
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    x, wt = torch.randn(n, c, h, w, device="cuda", generator=g), torch.randn(c, oc, k, k, device="cuda", generator=g) * (c * k * k) ** -0.5
    bias = torch.randn(oc, device="cuda", generator=g)
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv_transpose2d_f32(x, wt, bias, (1, 1, 1, 1), (s, s), (1, 1), 1, (0, 0), ctx=kept))
    assert "k_conv_f32_split" in names or (k == 3 and s == 2), names
    for i in sorted({0, n // 2, n - 1}):
        ref = torch.nn.functional.conv_transpose2d(x[i:i + 1].cpu().double(), wt.cpu().double(), bias.cpu().double(), s, 1)
        assert float((y[i:i + 1].cpu().double() - ref).abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())), i


# N, C, H, W, OC, k, (pad, right and bottom pad), groups: all four phases by one workgroup (as above, by its choice); 16-byte stores where W is whole fours and the output
# twice as wide; phases of equal and of unequal length and extent; one slot and several, the last one in part; blocks of 16 to 64 channels
TOGETHER = [
    (64, 128, 28, 28, 64, 4, (1, 1), 1), (48, 54, 31, 29, 40, 4, (1, 1), 1), (60, 33, 24, 20, 48, 4, (0, 0), 1), (128, 32, 24, 24, 17, 2, (0, 0), 1),
    (30, 70, 31, 33, 60, 2, (0, 0), 1), (60, 46, 24, 23, 64, 3, (1, 0), 1), (60, 46, 20, 24, 70, 3, (1, 1), 1), (24, 40, 23, 26, 96, 5, (2, 1), 1),
    (200, 24, 9, 8, 130, 3, (1, 0), 1), (16, 20, 70, 72, 16, 6, (2, 2), 1),
    (40, 96, 28, 28, 64, 4, (1, 1), 2), (40, 96, 24, 27, 32, 4, (1, 1), 2), (60, 92, 27, 28, 66, 3, (1, 0), 2), (40, 92, 27, 25, 34, 3, (1, 0), 2)]      # groups, 16 and 4 bytes


# phases of a workgroup each, or not, by a little
APART = [(48, 54, 31, 29, 64, 4, (1, 1), 1), (40, 33, 24, 20, 48, 4, (0, 0), 1), (30, 96, 20, 20, 128, 4, (1, 1), 2)]


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("shape", TOGETHER + APART)
def test_phases_of_one_workgroup(ops, kept, shape, large):
    """Bounds as above: 1e-5 of the largest output and 3e-7 in the 2-norm; operands of 2^60, whose sums are formed again in fp32, a rounding for each
    product."""
    n, c, h, w, oc, k, (before, behind), groups = shape
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    big = 2.0 ** 60 if large else 1.0
    x, wt = torch.randn(n, c, h, w, device="cuda", generator=g) * big, torch.randn(c, oc // groups, k, k, device="cuda", generator=g) * (c * k * k) ** -0.5 * big
    torch.cuda.synchronize()
    pads = (before, before, behind, behind)
    y, names = names_of(kept, lambda: ops.conv_transpose2d_f32(x, wt, None, pads, (2, 2), (1, 1), groups, (0, 0), ctx=kept))
    assert "k_conv_f32_split" in names, names
    H, W = y.shape[2:]
    conv = lambda a, b: torch.nn.functional.conv_transpose2d(a, b, None, 2, 0, 0, groups)[:, :, before:before + H, before:before + W]
    for i in sorted({0, n // 2, n - 1}):
        xi, wi = x[i:i + 1].cpu().double(), wt.cpu().double()
        ref = conv(xi, wi)
        err = y[i:i + 1].cpu().double() - ref
        if large:
            assert bool((err.abs() <= (c * k * k) ** 0.5 * 2.0 ** -24 * conv(xi.abs(), wi.abs())).all()), i
        else:
            assert float(err.abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())) and float(err.norm()) <= 3e-7 * float(ref.norm()), i


@pytest.mark.parametrize("shape,up", [(s, False) for s in EIGHTS[:3] + EIGHTS[5:6]] + [(s, True) for s in TOGETHER[:7] + TOGETHER[10:]])
def test_bias_and_relu_of_strided_and_transposed_layers(ops, kept, shape, up):
    """A bias for every channel, in 16-byte and in 4-byte stores, in the exchange between two phases and behind sums that are formed again; ReLU; bounds
    as above. One image has an infinity, which meets its own window alone: NaN or an infinity there, the rest as without it."""
    if up:
        n, c, h, w, oc, k, (before, behind), groups = shape
        g = torch.Generator(device="cuda").manual_seed(n + oc)
        wt = torch.randn(c, oc // groups, k, k, device="cuda", generator=g) * (c // groups * k * k / 4) ** -0.5
        call = lambda x, relu: ops.conv_transpose2d_f32(x, wt, bias, (before, before, behind, behind), (2, 2), (1, 1), groups, (0, 0), relu=relu, ctx=kept)
    else:
        n, c, h, w, oc, kh, kw, s, pads, d, groups = shape
        g = torch.Generator(device="cuda").manual_seed(n + oc)
        wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * (c // groups * kh * kw) ** -0.5
        call = lambda x, relu: ops.conv2d_f32(x, wt, bias, pads, s, d, groups, relu=relu, ctx=kept)
    x, bias = torch.randn(n, c, h, w, device="cuda", generator=g), torch.randn(oc, device="cuda", generator=g)
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: call(x, True))
    plain, _ = names_of(kept, lambda: call(x, False))
    assert names[-1] == "k_conv_f32_split", names
    assert torch.equal(y, plain.clamp(min=0)) and bool((plain < 0).any())
    H, W = y.shape[2:]
    for i in sorted({0, n // 2, n - 1}):
        xi = x[i:i + 1].cpu().double()
        if up:
            ref = torch.nn.functional.conv_transpose2d(xi, wt.cpu().double(), None, 2, 0, 0, groups)[:, :, before:before + H, before:before + W] + bias.cpu().double().view(1, -1, 1, 1)
        else:
            ref = reference(x[i:i + 1], wt, bias, s, pads, d, groups)
        err = plain[i:i + 1].cpu().double() - ref
        assert float(err.abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())) and float(err.norm()) <= 3e-7 * float(ref.norm()), i
    x[n // 2, 0, h // 2, w // 2] = float("inf")
    torch.cuda.synchronize()
    z, names = names_of(kept, lambda: call(x, False))
    assert names[-1] == "k_conv_f32_split", names
    bad = ~z[n // 2].isfinite()
    assert bool(bad.any()) and not bool((~z.isfinite()).sum() != bad.sum())
    rows, cols = bad.any(0).any(1).nonzero(), bad.any(0).any(0).nonzero()
    size = (k, k) if up else ((kh - 1) // s[0] + 1, (kw - 1) // s[1] + 1)
    assert int(rows.max() - rows.min()) < max(size[0], 1) * (1 if up else d[0]) + 1 and int(cols.max() - cols.min()) < max(size[1], 1) * (1 if up else d[1]) + 1
    keep = z.isfinite()
    assert float((z[keep] - plain[keep]).abs().max()) <= 2e-5 * max(1.0, float(plain.abs().max()))      # (the two sums' bounds together)


@pytest.mark.parametrize("n,c,h,oc,k,s,up", [(300, 1, 96, 100, 7, 1, False), (230, 128, 99, 128, 3, 2, False), (1400, 128, 28, 64, 4, 2, True), (300, 32, 99, 96, 3, 1, False)])
def test_images_of_more_than_a_launch(ops, kept, n, c, h, oc, k, s, up):
    """Above 1 GiB of images: full launches and one of the rest, whose form is chosen anew (rows of a kernel as cells, slots of eight channels, all
    phases by one workgroup, a plain layer); the images on both sides of the line, bound as above."""
    g = torch.Generator(device="cuda").manual_seed(n)
    pad = (k - 1) // 2
    x, wt = torch.randn(n, c, h, h, device="cuda", generator=g), torch.randn(*((c, oc) if up else (oc, c)), k, k, device="cuda", generator=g) * (c * k * k) ** -0.5
    torch.cuda.synchronize()
    if up:
        y, names = names_of(kept, lambda: ops.conv_transpose2d_f32(x, wt, None, (pad,) * 4, (s, s), (1, 1), 1, (0, 0), ctx=kept))
    else:
        y, names = names_of(kept, lambda: ops.conv2d_f32(x, wt, None, (pad,) * 4, (s, s), (1, 1), 1, ctx=kept))
    assert names.count("k_conv_f32_split") == 2, names
    per = ((1 << 30) - (16 << 20)) // (4 * max(x[0].numel(), y[0].numel()))
    assert per < n < 2 * per
    f = torch.nn.functional.conv_transpose2d if up else torch.nn.functional.conv2d
    for i in (0, per - 1, per, n - 1):
        ref = f(x[i:i + 1].cpu().double(), wt.cpu().double(), None, s, pad)
        assert float((y[i:i + 1].cpu().double() - ref).abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max())), i


@pytest.mark.parametrize("shape", CONV + [
    (64, 128, 28, 28, 64, 4, 2), (30, 143, 32, 34, 181, 4, 2), (120, 87, 19, 21, 256, 3, 2), (64, 120, 20, 20, 90, 3, 1)])      # transposed: k, stride
def test_sums_that_are_repeated_in_every_form(ops, kept, shape):
    """Operands of 2^60: every sum passes 2^95 on the way and is formed again with fp32 instructions from the operands as they were given, flipped
    and strided kernels of transposed layers among them. A rounding of 2^-24 for each of K products, which add as their square root."""
    transposed = len(shape) == 7
    n, c, h, w, oc = shape[:5]
    g = torch.Generator(device="cuda").manual_seed(n + c + oc)
    x = torch.randn(n, c, h, w, device="cuda", generator=g) * 2.0 ** 60
    if transposed:
        k, s = shape[5:]
        wt = torch.randn(c, oc, k, k, device="cuda", generator=g) * (c * k * k) ** -0.5 * 2.0 ** 60
        products = c * k * k
        conv = lambda a, b: torch.nn.functional.conv_transpose2d(a, b, None, s, 1)
        call = lambda: ops.conv_transpose2d_f32(x, wt, None, (1, 1, 1, 1), (s, s), (1, 1), 1, (0, 0), ctx=kept)
    else:
        kh, kw, s, (t, l, b, r), d, groups = shape[5:]
        products = c // groups * kh * kw
        wt = torch.randn(oc, c // groups, kh, kw, device="cuda", generator=g) * products ** -0.5 * 2.0 ** 60
        conv = lambda a, v: torch.nn.functional.conv2d(torch.nn.functional.pad(a, (l, r, t, b)), v, None, s, 0, d, groups)
        call = lambda: ops.conv2d_f32(x, wt, None, (t, l, b, r), s, d, groups, ctx=kept)
    torch.cuda.synchronize()
    y, names = names_of(kept, call)
    assert "k_conv_f32_split" in names or (transposed and k == 3 and s == 2), names
    for i in sorted({0, n // 2, n - 1}):
        xi, wi = x[i:i + 1].cpu().double(), wt.cpu().double()
        assert bool(((y[i:i + 1].cpu().double() - conv(xi, wi)).abs() <= products ** 0.5 * 2.0 ** -24 * conv(xi.abs(), wi.abs())).all()), i


@pytest.mark.parametrize("c,relu", [(72, False), (16, True)])
def test_values_that_are_not_finite_stay_in_their_windows(ops, kept, c, relu):
    """Infinities and NaN in cells, weights and products: the parts of a split infinity are no numbers, but its sums are the fp32
    kernels' again. Zeros, signs and the largest finite numbers, which a rounded bf16 would leave, among them."""
    g = torch.Generator().manual_seed(c)
    x, w = torch.randn(40, c, 28, 28, generator=g), torch.randn(96, c, 5, 5, generator=g)
    x[3, 0, 4, 4], x[3, c - 1, 27, 27], x[9, 5, 0, 13], x[39, 2, 27, 0] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[7, 3, 2, 2], w[95, c - 1, 0, 0] = 1e38, float("inf")
    w[:, 2] = w[:, 2].clamp(-0.5, 0.5)
    w[11] = 0.0
    xp = torch.nn.functional.pad(x, (2, 2, 2, 2))      # zeros outside the image are factors like others: with an infinite weight they are NaN
    ref = torch.nn.functional.conv2d(xp, w)
    ref = torch.where(ref > 0, ref, torch.zeros(())) if relu else ref
    xd, wd = x.cuda(), w.cuda()
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv2d_f32(xd, wd, None, (2, 2), (1, 1), (1, 1), 1, relu, ctx=kept))
    assert names[-1] == "k_conv_f32_split"
    y = y.cpu()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(torch.sign(y[~fin & ~torch.isnan(ref)]), torch.sign(ref[~fin & ~torch.isnan(ref)]))
    scale = torch.nn.functional.conv2d(torch.where(torch.isfinite(x), x, torch.zeros(())).abs().double(), torch.where(torch.isfinite(w), w, torch.zeros(())).abs().double(), None, 1, 2)
    assert bool(((y.double() - ref.double()).abs()[fin] <= 1e-5 * scale[fin] + 1e-30).all())


def test_small_and_mixed_magnitudes_keep_their_bits(ops, kept):
    """Every cell is split by itself: rows 2^60 apart in one tile, and channels of weights 2^100 apart, are as exact as rows of ones."""
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(64, 64, 28, 28, device="cuda", generator=g) * torch.exp2(torch.randint(-30, 31, (64, 1, 28, 1), device="cuda", generator=g).float())
    w = torch.randn(96, 64, 3, 1, device="cuda", generator=g) * torch.exp2(torch.randint(-60, 40, (96, 1, 1, 1), device="cuda", generator=g).float())
    w[:, :, 0], w[:, :, 2] = 0.0, 0.0      # an output row depends on one row of cells
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv2d_f32(x, w, None, (1, 0), (1, 1), (1, 1), 1, ctx=kept))
    assert names[-1] == "k_conv_f32_split"
    ref = torch.nn.functional.conv2d(x.double(), w.double(), None, 1, (1, 0)).cpu()
    size = torch.nn.functional.conv2d(x.double().abs(), w.double().abs(), None, 1, (1, 0)).cpu()
    assert bool(((y.cpu().double() - ref).abs() <= 2.0 ** -21 * size).all())      # two roundings of 2^-24 per 32 k and 2^-24 per product


# exponents of cells and weights: the smallest numbers of fp32 (2^-149) against large ones, products near 2^-126, sums above 2^95 (which
# are repeated with fp32 instructions), and all of them next to each other (None)
EXPONENTS = [(-114, 100), (-126, 110), (-140, 108), (110, -126), (100, -140), (-60, -60), (60, 60), (112, 0), (None, 0), (0, None)]


@pytest.mark.parametrize("e,f", EXPONENTS)
@pytest.mark.parametrize("kind", ["3x3", "rows", "phases"])
def test_magnitudes_of_all_sizes_keep_their_bits(ops, kept, kind, e, f):
    """Whatever the exponents: each output as near to float64 as with operands of one size, where the lowest bits of cells and weights are
    below those of bf16's smallest number, too. 2^-21 of the sum of the products' sizes: a rounding of 2^-24 per 32 k (at most 32 here, and they
    add as their square root) and 2^-24 per product. Where all exponents meet, sums above 2^95 among them are repeated, a rounding of 2^-24 for
    each of K products, of the size of the largest: K^1/2 2^-24."""
    c, k = {"3x3": (64, 3), "rows": (3, 7), "phases": (64, 4)}[kind]
    g = torch.Generator().manual_seed(5)

    def scaled(t, exponent):
        s = torch.randint(-140, 120, t.shape, generator=g).double() if exponent is None else torch.full((), float(exponent), dtype=torch.float64)
        return (t.double() * torch.exp2(s)).float()
    x = scaled(torch.randn(48, c, 40, 40, generator=g), e)
    w = scaled(torch.randn((c, 64, k, k) if kind == "phases" else (96, c, k, k), generator=g) * (c * k * k) ** -0.5, f)
    xd, wd = x.cuda(), w.cuda()
    torch.cuda.synchronize()
    if kind == "phases":
        y, names = names_of(kept, lambda: ops.conv_transpose2d_f32(xd, wd, None, (1, 1, 1, 1), (2, 2), (1, 1), 1, (0, 0), ctx=kept))
        conv = lambda a, b: torch.nn.functional.conv_transpose2d(a, b, None, 2, 1)
    else:
        y, names = names_of(kept, lambda: ops.conv2d_f32(xd, wd, None, (k // 2, k // 2), ctx=kept))
        conv = lambda a, b: torch.nn.functional.conv2d(a, b, None, 1, k // 2)
    assert names[-1] == "k_conv_f32_split"
    bound = 2.0 ** -21 if None not in (e, f) else (c * k * k) ** 0.5 * 2.0 ** -24
    for i in (0, 20, 47):
        xi, wi = x[i:i + 1].double(), w.double()
        assert bool(((y[i:i + 1].cpu().double() - conv(xi, wi)).abs() <= bound * conv(xi.abs(), wi.abs()) + c * k * k * 2.0 ** -149).all()), i


def test_whole_numbers_are_exact(ops, kept):
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randint(-300, 301, (50, 48, 30, 30), device="cuda", generator=g).float()
    w = torch.randint(-9, 10, (80, 48, 3, 3), device="cuda", generator=g).float()
    torch.cuda.synchronize()
    y, names = names_of(kept, lambda: ops.conv2d_f32(x, w, None, (1, 1), ctx=kept))
    assert names[-1] == "k_conv_f32_split"
    assert torch.equal(y.cpu(), torch.nn.functional.conv2d(x.cpu(), w.cpu(), None, 1, 1))


@pytest.mark.parametrize("kind", ["cell of a strided layer", "cell of a transposed layer", "weight"])
def test_sums_are_formed_again_in_their_tiles_alone(ops, kept, kind):
    """An infinity in a cell that few windows hold, or in one weight: tiles of 16 pixels x 16 channels without a sum that is not finite keep every bit."""
    g = torch.Generator(device="cuda").manual_seed(9)
    up, s = kind == "cell of a transposed layer", 2 if kind == "cell of a strided layer" else 1
    n, c, h, w, oc, k = (64, 128, 28, 28, 64, 4) if up else EIGHTS[0][:6] if s == 2 else CONV[0][:6]
    x, wt = torch.randn(n, c, h, w, device="cuda", generator=g), torch.randn(*((c, oc) if up else (oc, c)), k, k, device="cuda", generator=g) * (c * k * k) ** -0.5
    torch.cuda.synchronize()
    if up:
        call = lambda ctx: ops.conv_transpose2d_f32(x, wt, None, (1, 1, 1, 1), (2, 2), (1, 1), 1, (0, 0), ctx=ctx)
    else:
        call = lambda ctx: ops.conv2d_f32(x, wt, None, (1, 1, 1, 1), (s, s), (1, 1), 1, ctx=ctx)
    y, names = names_of(kept, lambda: call(kept))
    assert names[-1] == "k_conv_f32_split"
    if kind == "weight":
        wt[70, 3, 1, 1] = float("inf")
    else:
        x[5, 2, 10, 12] = float("inf")
    torch.cuda.synchronize()
    other = ops.Context(0)      # (keeps no weights of the call before)
    other.check(other.lib.sofie_hip_constant_weights(other.h, 1))
    z, names = names_of(other, lambda: call(other))
    assert names[-1] == "k_conv_f32_split"
    differs, bad = z != y, ~z.isfinite()
    if kind == "weight":
        assert bool(bad[:, 70].all()) and not bool(differs[:, :64].any() or differs[:, 80:].any()) and not bool(bad[:, 71:].any())
    else:
        pixels = bad.any(1).sum()
        assert int(pixels) == (16 if up else 1) and int(differs.any(1).sum()) <= 16 * int(pixels) and not bool(differs[:5].any() or differs[6:].any())
    other.close()
