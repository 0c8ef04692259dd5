"""One-byte products on operands of any size and alignment: rows that start at any byte, K that is no multiple of 16, both
storage orders of B. Covers the kernels of small products (k_gemm_bytes_direct on 16 and 32 rows and columns, k_gemm_bytes
on 64 x 64 and 128 x 128 tiles, each for rows of whole dwords and of any bytes), the copies that large products make
(k_copy_operands), and the paths without memory for a copy."""
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


def rng(seed):
    return np.random.default_rng(seed)


def rows_at(ctx, a, ld, offset):
    """The matrix on the device with rows `ld` bytes apart, the first `offset` bytes into its buffer (which ends with the
    last row); returns (buffer, address)."""
    buf = np.full(offset + (a.shape[0] - 1) * ld + a.shape[1], 0x55, np.uint8)
    for i, row in enumerate(a.view(np.uint8)):
        buf[offset + i * ld:offset + i * ld + a.shape[1]] = row
    t = torch.from_numpy(buf).to(ctx.device)
    return t, t.data_ptr() + offset


# one K below and above a chunk of 16 and a step of 128, K whose last chunk holds one byte, single rows and columns, tiles
# that end one row or column behind a boundary
SHAPES = [(1, 4, 16), (1, 5, 17), (3, 1, 31), (16, 16, 127), (17, 33, 129), (33, 47, 50), (2, 300, 1000), (65, 66, 257), (5, 2, 4099),
          (70, 13, 1041), (256, 1000, 1000), (130, 300, 515), (300, 257, 2049), (700, 650, 397)]


@pytest.mark.parametrize("transB", [True, False])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8_product_of_any_rows(ops, M, N, K, transB):
    """Bit-exact against the oracle for the three output kinds; operands at an odd and at a four-byte offset."""
    r = rng(1000 + M + N + K)
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (N, K) if transB else (K, N)).astype(np.int8)
    scale = (r.uniform(20.0, 60.0, N) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-2000, 2000, N).astype(np.int32)
    acc = oracle.igemm_s8(A, B, transB) + bias[None, :]
    ctx = ops.default_context()
    sd, bd = ctx.dev(scale), ctx.dev(bias)
    for offset, pad in ((0, 0), (3, 2), (4, -K % 4)):
        (ta, pa), (tb, pb) = rows_at(ctx, A, K + pad, offset), rows_at(ctx, B, B.shape[1] + pad, offset)
        for out, want in ((L.OUT_S32, acc), (L.OUT_S8, oracle.qgemm_s8(A, B, scale, bias, transB, zpy=3, relu=True)),
                          (L.OUT_F32, oracle.qgemm_s8_f32out(A, B, scale, bias, transB, relu=True))):
            y = ctx.empty((M, N), {L.OUT_S32: torch.int32, L.OUT_S8: torch.int8, L.OUT_F32: torch.float32}[out])
            ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, int(transB), M, N, K, C.c_void_p(pa), K + pad, C.c_void_p(pb), B.shape[1] + pad,
                                                 ctx.ptr(sd), ctx.ptr(bd), 3, L.ACT_RELU, ctx.ptr(y), N, out))
            ctx.sync()
            assert np.array_equal(y.cpu().numpy(), want), (offset, pad, out)


@pytest.mark.parametrize("M,N,K,kernel", [(17, 287, 11888, "k_qgemm_few_rows"), (31, 1023, 24000, "k_qgemm_few_rows"),
                                          (32, 64, 40000, "k_qgemm_few_rows"), (33, 64, 40000, "k_gemm_bytes"),
                                          (20, 1300, 24000, "k_gemm_bytes"), (2, 64, 46736, "k_qgemm_few_rows"),
                                          (3, 3326, 16368, "k_qgemm_few_rows_whole")])
def test_up_to_32_rows_on_a_long_sum_are_a_pass_over_b(ops, M, N, K, kernel):
    r = rng(1500 + M)
    A, B = r.integers(-127, 128, (M, K)).astype(np.int8), r.integers(-127, 128, (N, K)).astype(np.int8)
    scale = (r.uniform(20.0, 60.0, N) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    ctx = ops.Context(0)
    a, b, sd, y = ctx.dev(A), ctx.dev(B), ctx.dev(scale), ctx.empty((M, N), torch.int8)
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
    ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, 1, M, N, K, ctx.ptr(a), K, ctx.ptr(b), K, ctx.ptr(sd), None, -3, L.ACT_NONE, ctx.ptr(y), N, L.OUT_S8))
    ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
    ctx.sync()
    names = [l.split()[0] for l in buf.value.decode().splitlines()]
    assert names[0] == kernel, names
    assert np.array_equal(y.cpu().numpy(), oracle.qgemm_s8(A, B, scale, None, True, zpy=-3))
    ctx.close()


# a size for each number of rows and columns of k_gemm_bytes_direct (16 x 16, 16 x 32, 32 x 16, 32 x 32)
@pytest.mark.parametrize("M,N", [(40, 100), (200, 500), (1088, 100), (500, 272)])
@pytest.mark.parametrize("K", [41, 45, 46, 47, 44, 300, 1001])
def test_last_chunk_of_every_direct_form(ops, M, N, K):
    """The bytes behind K are cut off by moving the last chunk of a row down: 1 to 15 bytes, in every form of the kernel and for every kind
    of output. int8 against the oracle bit by bit; e4m3 within 7 * 2^-13 of the sum of the products' magnitudes (the matrix
    instruction's own cut) and a rounding to bfloat16 (2^-8)."""
    r = rng(1050 + M + K)
    ctx = ops.default_context()
    A, B = r.integers(-127, 128, (M, K)).astype(np.int8), r.integers(-127, 128, (N, K)).astype(np.int8)
    scale = (r.uniform(20.0, 60.0, N) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-2000, 2000, N).astype(np.int32)
    a, b, sd, bd = ctx.dev(A), ctx.dev(B), ctx.dev(scale), ctx.dev(bias)
    for out, want in ((L.OUT_S32, oracle.igemm_s8(A, B, True) + bias[None, :]), (L.OUT_S8, oracle.qgemm_s8(A, B, scale, bias, True, zpy=3)),
                      (L.OUT_F32, oracle.qgemm_s8_f32out(A, B, scale, bias, True))):
        y = ctx.empty((M, N), {L.OUT_S32: torch.int32, L.OUT_S8: torch.int8, L.OUT_F32: torch.float32}[out])
        ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, 1, M, N, K, ctx.ptr(a), K, ctx.ptr(b), K, ctx.ptr(sd), ctx.ptr(bd), 3, L.ACT_NONE, ctx.ptr(y), N, out))
        ctx.sync()
        assert np.array_equal(y.cpu().numpy(), want), out
    fa, fb = (torch.from_numpy(r.standard_normal(s).astype(np.float32)).to(torch.float8_e4m3fn) for s in ((M, K), (N, K)))
    want, mag = fa.double() @ fb.double().t(), fa.double().abs() @ fb.double().abs().t()
    ad, bd8 = fa.view(torch.uint8).cuda(), fb.view(torch.uint8).cuda()
    for out, kind, rounding in ((L.OUT_F32, torch.float32, 0.0), (L.OUT_BF16, torch.bfloat16, 2.0 ** -8)):
        y = ctx.empty((M, N), kind)
        torch.cuda.synchronize()
        ctx.check(ctx.lib.sofie_hip_gemm_fp8(ctx.h, 1, M, N, K, ctx.ptr(ad), K, ctx.ptr(bd8), K, 1.0, 1.0, None, ctx.ptr(y), N, out))
        ctx.sync()
        assert bool(((y.cpu().double() - want).abs() <= 7 * 2.0 ** -13 * mag + rounding * want.abs()).all()), out


@pytest.mark.parametrize("transB", [True, False])
@pytest.mark.parametrize("M,N,K", [(2100, 4099, 131), (1025, 8200, 48)])
def test_large_int8_product_copies_ragged_operands(ops, M, N, K, transB):
    """Products of 128 tiles of 256 x 256 and more: operands copied into whole chunks (A alone where B has them), sampled rows
    against the oracle, with and without the constant-weights promise."""
    r = rng(1100 + K)
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (N, K) if transB else (K, N)).astype(np.int8)
    rows = np.concatenate([np.arange(0, 16), r.integers(0, M, 16), np.arange(M - 16, M)])
    want = oracle.igemm_s8(A[rows], B, transB)
    for promise in (0, 1):
        ctx = ops.Context(0)
        assert ctx.lib.sofie_hip_constant_weights(ctx.h, promise) == 0
        a, b = ctx.dev(A), ctx.dev(B)
        for _ in range(2):
            y = ctx.empty((M, N), torch.int32)
            ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, int(transB), M, N, K, ctx.ptr(a), K, ctx.ptr(b), B.shape[1], None, None, 0,
                                                 L.ACT_NONE, ctx.ptr(y), N, L.OUT_S32))
            ctx.sync()
            assert np.array_equal(y.cpu().numpy()[rows], want)
        ctx.close()


@pytest.mark.parametrize("M,N,K,transB", [(256, 1000, 1000, False), (40, 70, 333, False), (2100, 4099, 67, False), (2100, 4099, 67, True),
                                          (2048, 4096, 72, False)])
def test_operand_changed_between_calls_under_the_promise(ops, M, N, K, transB):
    """The constant-weights promise does not name the operands of these products: B rewritten in place between two calls (as a
    tensor that a program computes is) gives the product with what it holds then."""
    r = rng(1150 + K)
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    rows = np.unique(np.concatenate([np.arange(0, min(M, 16)), r.integers(0, M, 16), [M - 1]]))
    ctx = ops.Context(0)
    assert ctx.lib.sofie_hip_constant_weights(ctx.h, 1) == 0
    a, b = ctx.dev(A), ctx.empty((N, K) if transB else (K, N), torch.int8)
    for _ in range(3):
        B = r.integers(-127, 128, (N, K) if transB else (K, N)).astype(np.int8)
        b.copy_(torch.from_numpy(B))
        y = ctx.empty((M, N), torch.int32)
        torch.cuda.synchronize()
        ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, int(transB), M, N, K, ctx.ptr(a), K, ctx.ptr(b), B.shape[1], None, None, 0, L.ACT_NONE,
                                             ctx.ptr(y), N, L.OUT_S32))
        ctx.sync()
        assert np.array_equal(y.cpu().numpy()[rows], oracle.igemm_s8(A[rows], B, transB))
    ctx.close()


@pytest.mark.parametrize("M,N,K,kernels", [(1, 1, 16, ["k_gemm_bytes_simple"]), (53, 305, 23, ["k_gemm_bytes_simple"]),
                                           (8, 64, 34, ["k_gemm_bytes_simple"]), (40, 70, 333, ["k_copy_operands", "k_gemm_bytes_direct"])])
def test_short_sums_take_the_shorter_way(ops, M, N, K, kernels):
    """B [K,N] of odd rows: a thread per output where that is one launch of less time than the copy and the product."""
    r = rng(1300 + K)
    A, B = r.integers(-127, 128, (M, K)).astype(np.int8), r.integers(-127, 128, (K, N)).astype(np.int8)
    ctx = ops.Context(0)
    (a, pa), (b, pb), y = rows_at(ctx, A, K, 0), rows_at(ctx, B, N, 3), ctx.empty((M, N), torch.int32)
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
    ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, 0, M, N, K, C.c_void_p(pa), K, C.c_void_p(pb), N, None, None, 0, L.ACT_NONE, ctx.ptr(y), N, L.OUT_S32))
    ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
    ctx.sync()
    assert [l.split()[0] for l in buf.value.decode().splitlines()] == kernels
    assert np.array_equal(y.cpu().numpy(), oracle.igemm_s8(A, B, False))
    ctx.close()


def test_int8_product_of_a_billion_rows(ops):
    """2^30 rows: 64 x 64 tiles would be a launch of 2^32 threads."""
    M, N, K = 1 << 30, 17, 16
    r = rng(30)
    ctx = ops.default_context()
    a = torch.empty((M, K), dtype=torch.int8, device="cuda")
    a.view(torch.int64).random_()
    B = r.integers(-127, 128, (N, K)).astype(np.int8)
    scale = (r.uniform(20.0, 60.0, N) / (73.3 * 73.3 * 4.0)).astype(np.float32)
    b, sd, y = ctx.dev(B), ctx.dev(scale), torch.zeros((M, N), dtype=torch.int8, device="cuda")
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, 1, M, N, K, ctx.ptr(a), K, ctx.ptr(b), K, ctx.ptr(sd), None, 0, L.ACT_NONE, ctx.ptr(y), N,
                                         L.OUT_S8))
    ctx.sync()
    pick = torch.from_numpy(np.concatenate([np.arange(200), r.integers(0, M, 500), np.arange(M - 200, M)])).cuda()
    assert np.array_equal(y[pick].cpu().numpy(), oracle.qgemm_s8(a[pick].cpu().numpy(), B, scale, None, True))


@pytest.mark.parametrize("M,N,K,transB", [(40, 70, 333, False), (9, 3, 100, False), (1024, 16, 16384, True), (300, 5, 32768, True)])
def test_any_rows_without_memory_for_a_copy(ops, M, N, K, transB):
    """B [K,N] of odd rows, and a long K on at most 16 columns, in a call that is recorded on a fresh context (no scratch buffer
    exists and none may be made): a kernel that reads B where it lies and writes no partial sums runs, and every replay
    gives the oracle's result."""
    r = rng(1200 + K)
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (N, K) if transB else (K, N)).astype(np.int8)
    want = oracle.igemm_s8(A, B, transB)
    ctx = ops.Context(0, stream=torch.cuda.Stream())
    a, b, y = ctx.dev(A), ctx.dev(B), ctx.empty((M, N), torch.int32)
    torch.cuda.synchronize()
    graph = C.c_void_p()
    ctx.check(ctx.lib.sofie_hip_capture_begin(ctx.h))
    rc = ctx.lib.sofie_hip_qgemm_s8(ctx.h, int(transB), M, N, K, ctx.ptr(a), K, ctx.ptr(b), B.shape[1], None, None, 0, L.ACT_NONE, ctx.ptr(y), N,
                                    L.OUT_S32)
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


@pytest.mark.parametrize("M,N,K", [(256, 4096, 8320), (300, 4100, 8208), (64, 4100, 8208)])
def test_aligned_product_whose_b_may_not_be_copied(ops, M, N, K):
    """B [K,N] of more bytes than the entry point that allocates nothing has scratch memory: read where it lies, on 128 x 128
    tiles (whole and ragged ones) or on 64 x 64 tiles; sampled rows against the oracle."""
    r = rng(1270 + M)
    A, B = r.integers(-127, 128, (M, K)).astype(np.int8), r.integers(-127, 128, (K, N)).astype(np.int8)
    rows = np.unique(np.concatenate([np.arange(0, 4), r.integers(0, M, 6), [M - 1]]))
    ctx = ops.default_context()
    a, b, y = ctx.dev(A), ctx.dev(B), ctx.empty((M, N), torch.int32)
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_qgemm_s8_noalloc(ctx.h, 0, M, N, K, ctx.ptr(a), K, ctx.ptr(b), N, None, None, 0, L.ACT_NONE, ctx.ptr(y), N, L.OUT_S32))
    ctx.sync()
    assert np.array_equal(y.cpu().numpy()[rows], oracle.igemm_s8(A[rows], B))


def test_few_rows_that_lie_far_apart(ops):
    """16 rows of A 300 MB apart, on a B that the kernel for few rows takes otherwise: its offsets are 32 bits wide."""
    M, N, K, lda = 16, 2048, 1024, 300_000_000
    r = rng(1250)
    A, B = r.integers(-127, 128, (M, K)).astype(np.int8), r.integers(-127, 128, (N, K)).astype(np.int8)
    ctx = ops.default_context()
    a = torch.zeros((M - 1) * lda + K, dtype=torch.int8, device=ctx.device)
    for i in range(M):
        a[i * lda:i * lda + K] = torch.from_numpy(A[i]).to(ctx.device)
    b, y = ctx.dev(B), ctx.empty((M, N), torch.int32)
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, 1, M, N, K, ctx.ptr(a), lda, ctx.ptr(b), K, None, None, 0, L.ACT_NONE, ctx.ptr(y), N, L.OUT_S32))
    ctx.sync()
    assert np.array_equal(y.cpu().numpy(), oracle.igemm_s8(A, B, True))


@pytest.mark.parametrize("transB", [True, False])
@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (17, 33, 129), (33, 47, 50), (256, 500, 1001), (300, 1030, 333), (1, 9, 4001), (2100, 4099, 67)])
def test_fp8_product_of_any_rows(ops, M, N, K, transB):
    """Against the float64 product of the same e4m3 operands: |d| <= 7 * 2^-13 * sum|a_k b_k| (what the matrix instruction's sums of
    eight products may drop), plus 2^-8 |ref| for a bf16 result."""
    g = torch.Generator(device="cuda").manual_seed(1300 + M + N + K)
    A = torch.randn(M, K, device="cuda", generator=g).to(torch.float8_e4m3fn)
    B = torch.randn(*((N, K) if transB else (K, N)), device="cuda", generator=g).to(torch.float8_e4m3fn)
    bias = torch.randn(N, device="cuda", generator=g)
    a, b = A.double(), (B.t() if transB else B).double().contiguous()
    ref, mag = a @ b + bias.double(), a.abs() @ b.abs()
    for out in (L.OUT_F32, L.OUT_BF16):
        y = ops.gemm_fp8(A.view(torch.uint8), B.view(torch.uint8), 1.0, 1.0, bias, transB, out)
        tol = (2.0 ** -8 if out == L.OUT_BF16 else 2.0 ** -23) * ref.abs() + 7 * 2.0 ** -13 * mag
        assert bool(((y.double() - ref).abs() <= tol).all())
