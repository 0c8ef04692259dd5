"""fp32 products on k_gemm_f32_split (operands as three bf16 numbers): every storage, 32, 64 and 96 rows per workgroup, K in slices, the
shortest K it is chosen for (two chunks per wavefront, one k in the last), rows, columns and K that are no whole fours, against float64;
values that are not finite."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from sofie_amd import lib as L  # noqa: E402


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


def product(ctx, a, b, tA, tB, bias, alpha=1.0, beta=1.0, relu=False, pad=0, kind=L.BIAS_ROW):
    """The call through the C ABI, rows of all operands `pad` floats further apart than they are long; the result and the kernels' names."""
    M, N, K = (a.shape[1] if tA else a.shape[0]), (b.shape[0] if tB else b.shape[1]), (a.shape[0] if tA else a.shape[1])

    def wide(t):
        if not pad:
            return t
        w = torch.full((t.shape[0], t.shape[1] + pad), float("nan"), device="cuda")
        w[:, :t.shape[1]] = t
        return w
    a, b, y = wide(a), wide(b), torch.full((M + 2, N + pad), 77.0, device="cuda")
    torch.cuda.synchronize()
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
    ctx.check(ctx.lib.sofie_hip_gemm_f32(ctx.h, tA, tB, M, N, K, alpha, a.data_ptr(), a.shape[1], b.data_ptr(), b.shape[1], beta if bias is not None else 0.0,
                                         bias.data_ptr() if bias is not None else None, kind if bias is not None else L.BIAS_NONE,
                                         y[1].data_ptr(), N + pad, L.ACT_RELU if relu else L.ACT_NONE))
    ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
    ctx.sync()
    assert bool((y[0] == 77.0).all() and (y[M + 1] == 77.0).all() and (y[:, N:] == 77.0).all())      # nothing around the result
    return y[1:M + 1, :N], [line.split()[0] for line in buf.value.decode().splitlines()]


# M, N, K: whether A stored along M takes the kernel, too (64 rows per workgroup or none); slices of K
SHAPES = [((64, 6208, 1106), False, 1), ((65, 6209, 1105), True, 1), ((112, 7656, 1284), True, 1), ((97, 6301, 1283), True, 1),
          ((1500, 1001, 1111), False, 1), ((1501, 1003, 1024), False, 1), ((1441, 1089, 1538), True, 1), ((1537, 1023, 2049), True, 1),
          ((1195, 1160, 481), False, 1), ((1757, 2409, 486), False, 1), ((4624, 133, 5187), True, 1), ((130, 3633, 4279), False, 2),
          ((2447, 107, 5990), True, 3), ((3001, 1001, 1113), True, 1)]


@pytest.mark.parametrize("shape,along_m,slices", SHAPES)
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_in_three_parts(ops, shape, along_m, slices, tA, tB):
    """Products of split numbers lose at most 2^-24 each (2^-27 in the mean) and sums are rounded once per 32 k at their own size, where fp32 products in a
    row are rounded K times: 3e-7 in the 2-norm and 1e-6 of the largest output (fp32 instructions show up to 1.2e-6 at these K).
    The same bits on a second call."""
    M, N, K = shape
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn((K, M) if tA else (M, K), device="cuda", generator=g)
    b = torch.randn((N, K) if tB else (K, N), device="cuda", generator=g) * K ** -0.5
    bias = torch.randn(N, device="cuda", generator=g)
    ref = (a.t() if tA else a).double().contiguous() @ (b.t() if tB else b).double().contiguous()
    ctx = ops.Context(0)
    y, names = product(ctx, a, b, tA, tB, bias)
    want = ref + bias.double()
    if not tA or along_m:
        assert names == ["k_gemm_f32_split"] + ["k_gemm_f32_skinny_finish"] * (slices > 1), names
        err = y.double() - want
        assert float(err.norm()) <= 3e-7 * float(want.norm()) and float(err.abs().max()) <= 1e-6 * float(want.abs().max())
    else:
        assert "k_gemm_f32_split" not in names, names
    assert torch.equal(y, product(ctx, a, b, tA, tB, bias)[0])
    y, _ = product(ctx, a, b, tA, tB, bias, alpha=-0.5, beta=2.0, relu=True, pad=3)
    want = (-0.5 * ref + 2.0 * bias.double()).clamp(min=0)
    assert float((y.double() - want).abs().max()) <= 1e-6 * float(want.abs().max())
    ctx.close()


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_in_three_parts_of_values_that_are_not_finite(ops, tA, tB):
    """Infinities, NaN and sums that overflow stay where fp32 products put them, and finite ones next to them stay right; numbers that
    bf16 would round up to infinity are finite."""
    M, N, K = 3001 if tA else 1500, 1001, 1111
    g = torch.Generator(device="cuda").manual_seed(5)
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(K, N, device="cuda", generator=g)
    a[3, 7], a[700, 1110], a[1499, 0], a[900, 50], b[50, 1000] = float("inf"), float("nan"), float("-inf"), 3.4e38, 0.25
    a[[3, 700, 900, 1499], 9] = 0.0      # (b[9, 33] below: two products that overflow with opposite signs are NaN in fp32)
    a[40, :] = 0.0
    a[40, 9], b[9, 33] = 1.0, 3.4028234e38
    a[41, :] = 3e38
    b[:, 500] = 1.0
    ctx = ops.Context(0)
    y, names = product(ctx, a.t().contiguous() if tA else a, b.t().contiguous() if tB else b, tA, tB, None)
    assert "k_gemm_f32_split" in names, names
    rows = [3, 40, 41, 700, 900, 1499, 0, 1, 64, 1498]
    ref = a[rows].cpu().double() @ b.cpu().double()
    got = y[rows].cpu()
    ref32 = torch.where(ref.abs() > 3.4028235e38, torch.sign(ref) * float("inf"), ref)
    for i, r in enumerate(rows):
        if r == 41:      # sums of 3e38 times anything: only the one that must overflow
            assert float(got[i, 500]) == float("inf")
            continue
        assert torch.equal(got[i].isnan(), ref32[i].isnan()), r
        assert torch.equal(got[i].isinf(), ref32[i].isinf()), r
        assert torch.equal(torch.sign(got[i][got[i].isinf()]).double(), torch.sign(ref32[i][ref32[i].isinf()])), r
        fin = ref32[i].isfinite()
        if bool(fin.any()):
            assert float((got[i][fin].double() - ref32[i][fin]).abs().max()) <= 1e-5 * float(ref32[i][fin].abs().max()), r
    ctx.close()


@pytest.mark.parametrize("e,f", [(-114, 100), (-126, 110), (-140, 108), (100, -140), (-60, -60), (60, 60), (112, 0), (None, 0), (0, None)])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0)])
def test_magnitudes_of_all_sizes_keep_their_bits(ops, tA, tB, e, f):
    """Whatever the exponents of a and b (None: all of them next to each other): each output as near to float64 as with operands of one size,
    where their lowest bits are below those of bf16's smallest number, too. 2^-21 of the sum of the products' sizes: a rounding of 2^-24 per
    32 k of a wavefront and for the wavefronts' sums, and 2^-24 per product."""
    M, N, K = (1500, 1001, 1111) if not tA else (4624, 640, 1111)
    g = torch.Generator(device="cuda").manual_seed(5)

    def scaled(shape, exponent):
        s = torch.randint(-140, 120, shape, device="cuda", generator=g).double() if exponent is None else torch.full((), float(exponent), dtype=torch.float64, device="cuda")
        return (torch.randn(shape, device="cuda", generator=g).double() * torch.exp2(s)).float()
    a, b = scaled((K, M) if tA else (M, K), e), scaled((N, K) if tB else (K, N), f)
    ctx = ops.Context(0)
    y, names = product(ctx, a, b, tA, tB, None)
    assert "k_gemm_f32_split" in names, names
    a, b = (a.t() if tA else a).double().contiguous(), (b.t() if tB else b).double().contiguous()
    assert bool(((y.double() - a @ b).abs() <= 2.0 ** -21 * (a.abs() @ b.abs()) + K * 2.0 ** -149).all())
    ctx.close()


@pytest.mark.parametrize("M,N,K", [(2710, 5088, 336), (2711, 5089, 337), (3185, 2559, 726), (5043, 4527, 451)])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_in_three_parts_on_shared_fragments(ops, M, N, K, tA, tB):
    """Tiles of 128 x 128 whose operands are split once for all wavefronts, whole ones and cut in all directions: bounds as above; an infinity, a NaN and
    sums that overflow stay where fp32 products put them, and sums next to them keep 2^-24 of each of K products, which add as their square root."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(K, N, device="cuda", generator=g) * K ** -0.5
    bias = torch.randn(N, device="cuda", generator=g)
    stored = lambda x, y: (x.t().contiguous() if tA else x, y.t().contiguous() if tB else y)
    ctx = ops.Context(0)
    y, names = product(ctx, *stored(a, b), tA, tB, bias, pad=3)
    assert names == ["k_gemm_f32_split_shared"], names
    want = a.double() @ b.double() + bias.double()
    err = y.double() - want
    assert float(err.norm()) <= 3e-7 * float(want.norm()) and float(err.abs().max()) <= 1e-6 * float(want.abs().max())
    a[3, 7], a[M - 1, K - 1], a[200, 0] = float("inf"), float("nan"), 3.4e38
    b[0, N - 1] = 1000.0
    y, names = product(ctx, *stored(a, b), tA, tB, None)
    assert names == ["k_gemm_f32_split_shared"], names
    rows = [0, 3, 63, 64, 127, 128, 199, 200, M - 5, M - 2, M - 1]
    ad, bd = a[rows].double(), b.double()
    ref = ad @ bd
    ref = torch.where(ref.abs() > 3.4028235e38, torch.sign(ref) * float("inf"), ref)
    got = y[rows].double()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    fin = ref.isfinite()
    assert bool(((got - ref).abs()[fin] <= (K ** 0.5 * 2.0 ** -24 * (ad.nan_to_num(0.0, 0.0, 0.0).abs() @ bd.abs()))[fin]).all())
    ctx.close()


@pytest.mark.parametrize("M,N,K,kernel", [(1441, 1089, 1538, "k_gemm_f32_split"), (1537, 1025, 2049, "k_gemm_f32_split"), (65, 6210, 1105, "k_gemm_f32_split"),
                                          (2753, 5121, 336, "k_gemm_f32_split_shared"), (2689, 5186, 337, "k_gemm_f32_split_shared")])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_an_infinity_in_the_last_tile_changes_no_bit_of_the_others(ops, M, N, K, kernel, tA, tB):
    """One or two columns (rows) in the last tile, and an infinity in the last one alone: its wavefront forms its sums again with fp32 instructions,
    those of the columns (rows) in front of its first, which it loads in fours with its own, among them. The tile before keeps what it has summed."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(K, N, device="cuda", generator=g)
    stored = lambda x, y: (x.t().contiguous() if tA else x, y.t().contiguous() if tB else y)
    ctx = ops.Context(0)
    y, names = product(ctx, *stored(a, b), tA, tB, None)
    assert names == [kernel], names
    for last in ("column", "row"):
        ai, bi = a.clone(), b.clone()
        if last == "column":
            bi[K // 2, N - 1] = float("inf")
        else:
            ai[M - 1, K // 2] = float("inf")
        for _ in range(3):
            yi, names = product(ctx, *stored(ai, bi), tA, tB, None)
            assert names == [kernel], names
            if last == "column":
                assert torch.equal(yi[:, :N // 64 * 64], y[:, :N // 64 * 64]) and not bool(yi[:, N - 1].isfinite().any())
            else:
                assert torch.equal(yi[:M // 64 * 64 if tA else M // 128 * 128], y[:M // 64 * 64 if tA else M // 128 * 128]) and not bool(yi[M - 1].isfinite().any())
    ctx.close()


@pytest.mark.parametrize("M,N,K", [(2711, 5089, 337), (5043, 4527, 451)])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("kind", [L.BIAS_NONE, L.BIAS_ROW, L.BIAS_COL])
def test_scale_bias_and_relu_on_shared_fragments(ops, M, N, K, tA, tB, kind):
    g = torch.Generator(device="cuda").manual_seed(M + kind)
    a, b = torch.randn(M, K, device="cuda", generator=g), torch.randn(K, N, device="cuda", generator=g) * K ** -0.5
    bias = None if kind == L.BIAS_NONE else torch.randn(N if kind == L.BIAS_ROW else M, device="cuda", generator=g)
    stored = (a.t().contiguous() if tA else a, b.t().contiguous() if tB else b)
    ctx = ops.Context(0)
    y, names = product(ctx, *stored, tA, tB, bias, alpha=-0.5, beta=2.0, relu=True, pad=3, kind=kind)
    assert names == ["k_gemm_f32_split_shared"], names
    want = -0.5 * (a.double() @ b.double())
    if bias is not None:
        want += 2.0 * (bias.double() if kind == L.BIAS_ROW else bias.double()[:, None])
    want = want.clamp(min=0)
    err = y.double() - want
    assert float(err.norm()) <= 3e-7 * float(want.norm()) and float(err.abs().max()) <= 1e-6 * float(want.abs().max())
    ctx.close()


# leading dimensions of A and of B (1: one matrix for all), M, N, K: 512 tiles of 128 x 128, the last ones cut
@pytest.mark.parametrize("la,lb,M,N,K", [((2,), (2,), 2041, 2047, 330), ((2, 4), (1, 4), 1021, 1019, 451), ((4, 1), (1, 2), 1021, 1019, 330), ((1,), (4,), 2045, 1017, 451)])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("relu", [False, True])
def test_stacks_on_shared_fragments(ops, la, lb, M, N, K, tA, tB, relu):
    """Stacked products, broadcast ones among them, each against float64; an infinity in one product's last row changes no other product."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    a, b = torch.randn(*la, M, K, device="cuda", generator=g), torch.randn(*lb, K, N, device="cuda", generator=g) * K ** -0.5
    lead = torch.broadcast_shapes(la, lb)
    n, strides = len(lead), lambda l, mat: [0 if l[i] == 1 else mat * int(torch.tensor(l[i + 1:]).prod()) for i in range(len(l))]
    ctx = ops.Context(0)

    def stacked(a, b):
        a, b = a.transpose(-1, -2).contiguous() if tA else a, b.transpose(-1, -2).contiguous() if tB else b
        y = torch.full((*lead, M, N), 77.0, device="cuda")
        torch.cuda.synchronize()
        buf, m = C.create_string_buffer(4096), C.c_int(-1)
        ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
        ctx.check(ctx.lib.sofie_hip_gemm_f32_stacked(ctx.h, tA, tB, M, N, K, -0.5, a.data_ptr(), a.shape[-1], b.data_ptr(), b.shape[-1], y.data_ptr(), N, n,
                                                     (C.c_int * n)(*lead), (C.c_longlong * n)(*strides(la, M * K)), (C.c_longlong * n)(*strides(lb, K * N)),
                                                     L.ACT_RELU if relu else L.ACT_NONE))
        ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(m)))
        ctx.sync()
        assert [line.split()[0] for line in buf.value.decode().splitlines()] == ["k_gemm_f32_split_shared"]
        return y.reshape(-1, M, N)
    y = stacked(a, b)
    af, bf = a.expand(*lead, M, K).reshape(-1, M, K), b.expand(*lead, K, N).reshape(-1, K, N)
    for i in range(y.shape[0]):
        want = -0.5 * (af[i].double() @ bf[i].double())
        want = want.clamp(min=0) if relu else want
        err = y[i].double() - want
        assert float(err.norm()) <= 3e-7 * float(want.norm()) and float(err.abs().max()) <= 1e-6 * float(want.abs().max()), i
    if la == lead:
        a[(-1,) * len(la) + (M - 1, K - 1)] = float("inf")
        z = stacked(a, b)
        assert torch.equal(z[:-1], y[:-1]) and torch.equal(z[-1, :M // 128 * 128 - 128], y[-1, :M // 128 * 128 - 128]) and not bool(z[-1, M - 1].isfinite().all())
    ctx.close()
