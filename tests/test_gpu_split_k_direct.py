"""int8 products of a long K on few tiles, K in slices: k_gemm_bytes_direct on 16 or 32 rows and columns with raw sums per slice, behind it
k_splitk_finish or k_splitk_finish_pair. Bit-exact against integer products in float64 (sums stay below 2^53)."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from sofie_amd import lib as L  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    from sofie_amd import ops
    c = ops.Context(0)
    yield c
    c.close()


def int8(gen, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, generator=gen)


def traced(ctx, call):
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
    ctx.check(call())
    ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
    ctx.sync()
    return [line.split()[0] for line in buf.value.decode().splitlines()]


def requantised(acc, scale, zp, relu):
    """round-to-nearest-even of the fp32 product of the sum and its column's scale, as the oracle has it"""
    v = torch.round(acc.to(torch.float32) * scale) + zp
    return v.clamp(max(-128, zp) if relu else -128, 127).to(torch.int8)


# tiles that end one row or column behind a boundary, columns that are no whole four, a last slice of one chunk of 16 and of whole
# chunks of 128, K with an odd number of slices; 64 x 256 x 12800 is the classifier's first fully connected layer at batch 64
@pytest.mark.parametrize("M,N,K", [(33, 65, 12288), (64, 256, 12800), (65, 77, 12304), (40, 90, 32784), (129, 73, 16000), (48, 70, 65552),
                                   (120, 250, 16400)])
def test_product_in_slices(ctx, M, N, K):
    gen = torch.Generator().manual_seed(M + N + K)
    a, b = int8(gen, M, K), int8(gen, N, K)
    scale = (torch.rand(N, generator=gen) + 0.5) * (40.0 / (73.3 ** 2 * K ** 0.5))
    bias = torch.randint(-2000, 2000, (N,), dtype=torch.int32, generator=gen)
    acc = (a.double() @ b.double().T).long() + bias
    ad, bd, sd, qd = (t.cuda() for t in (a, b, scale, bias))
    for out, want in ((L.OUT_S8, requantised(acc, scale, 3, True)), (L.OUT_S32, acc.int()), (L.OUT_F32, acc.float() * scale)):
        y = torch.full((M + 2, N), 77, dtype=want.dtype, device="cuda")
        torch.cuda.synchronize()
        names = traced(ctx, lambda: ctx.lib.sofie_hip_qgemm_s8(ctx.h, 1, M, N, K, ad.data_ptr(), K, bd.data_ptr(), K, sd.data_ptr(), qd.data_ptr(),
                                                               3 if out == L.OUT_S8 else 0, L.ACT_RELU if out == L.OUT_S8 else L.ACT_NONE,
                                                               y[1].data_ptr(), N, out))
        assert names == ["k_gemm_bytes_direct", "k_splitk_finish"], names
        assert torch.equal(y[1:M + 1].cpu(), want)
        assert bool((y[0] == 77).all() and (y[M + 1] == 77).all())


@pytest.mark.parametrize("M,N1,K,N2", [(64, 256, 12800, 5), (1, 256, 12800, 5), (30, 32, 24592, 8), (33, 128, 12304, 8), (130, 128, 16384, 1)])
def test_pair_in_slices(ctx, M, N1, K, N2):
    gen = torch.Generator().manual_seed(M + K)
    a, b1, b2 = int8(gen, M, K), int8(gen, N1, K), int8(gen, N2, N1)
    s1 = (torch.rand(N1, generator=gen) + 0.5) * (40.0 / (73.3 ** 2 * K ** 0.5))
    s2 = torch.rand(N2, generator=gen) + 0.5
    q1, q2 = (torch.randint(-2000, 2000, (n,), dtype=torch.int32, generator=gen) for n in (N1, N2))
    mid = requantised((a.double() @ b1.double().T).long() + q1, s1, -3, True)
    want = ((mid.double() @ b2.double().T).long() + q2).float() * s2
    d = [t.cuda() for t in (a, b1, b2, s1, s2, q1, q2)]
    m, y = torch.empty(M, N1, dtype=torch.int8, device="cuda"), torch.empty(M, N2, device="cuda")
    torch.cuda.synchronize()
    names = traced(ctx, lambda: ctx.lib.sofie_hip_qgemm_s8_pair(ctx.h, M, K, d[0].data_ptr(), K, N1, d[1].data_ptr(), K, d[3].data_ptr(),
                                                                d[5].data_ptr(), -3, L.ACT_RELU, m.data_ptr(), N1, N2, d[2].data_ptr(), N1,
                                                                d[4].data_ptr(), d[6].data_ptr(), 0, L.ACT_NONE, y.data_ptr(), N2, L.OUT_F32))
    assert names == ["k_gemm_bytes_direct", "k_splitk_finish_pair"], names
    assert torch.equal(y.cpu(), want)
