"""fp32 products of any size, alignment and storage: k_gemm_f32_direct (16 and 32 rows and columns per workgroup) and
k_gemm_f32 (tiles of 32 x 32 to 128 x 128, K in one piece or in slices), every transposition, against float64."""
import ctypes as C

import numpy as np
import pytest

from sofie_amd import lib as L

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


# (M, N, K): a single element, K below the four of a load, one k and one row or column behind a chunk (4, 32), a tile
# (16, 32, 64, 96, 128) or a wavefront's share; K long enough for slices (few tiles) and a size for each tile shape
SIZES = [(1, 1, 1), (3, 5, 2), (16, 16, 32), (17, 33, 31), (33, 17, 65), (65, 129, 100), (130, 67, 19), (97, 64, 33), (64, 64, 2049),
         (300, 200, 1025), (10, 1000, 999), (700, 33, 77), (1100, 1000, 130), (2050, 1030, 67)]
# rows and columns that are no whole fours, K in whole steps of 32: the last step of an operand stored along M or N must not be
# requested 16 bytes at a time, and it is the last one of a round of stages (two: an odd number of steps, three: 2 mod 3)
STRADDLING = [(1501, 1001, 1024), (301, 1003, 256), (130, 1002, 160), (2049, 1031, 96), (258, 257, 4096)]


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", SIZES + STRADDLING)
def test_gemm_f32_of_any_kind(ops, M, N, K, tA, tB):
    """1e-5 of the largest output: sums of fp32 products in another order differ by about sqrt(K) 2^-24 of the terms' root
    mean square times sqrt(K). Leading dimensions equal to the sizes and three floats wider, every bias kind."""
    g = torch.Generator(device="cuda").manual_seed(100 * M + 10 * N + K)
    ctx = ops.default_context()

    def matrix(rows, cols, pad):
        return torch.randn(rows, cols + pad, device="cuda", generator=g)
    for pad, kind in ((0, L.BIAS_ROW), (3, L.BIAS_NONE), (0, L.BIAS_FULL), (3, L.BIAS_COL)):
        A = matrix(K, M, pad) if tA else matrix(M, K, pad)
        B = matrix(N, K, pad) if tB else matrix(K, N, pad)
        a = A[:, :M].t() if tA else A[:, :K]
        b = B[:, :K].t() if tB else B[:, :N]
        bias = {L.BIAS_NONE: None, L.BIAS_ROW: torch.randn(N, device="cuda", generator=g), L.BIAS_FULL: torch.randn(M, N, device="cuda", generator=g),
                L.BIAS_COL: torch.randn(M, device="cuda", generator=g)}[kind]
        beta = 0.0 if bias is None else 2.0
        y = ctx.empty((M, N), torch.float32)
        torch.cuda.synchronize()
        ctx.check(ctx.lib.sofie_hip_gemm_f32(ctx.h, tA, tB, M, N, K, 0.5, ctx.ptr(A), A.shape[1], ctx.ptr(B), B.shape[1], beta, ctx.ptr(bias), kind,
                                             ctx.ptr(y), N, L.ACT_RELU))
        ctx.sync()
        ref = 0.5 * (a.double().contiguous() @ b.double().contiguous())
        if bias is not None:
            ref = ref + beta * (bias.double()[:, None] if kind == L.BIAS_COL else bias.double())
        ref = ref.clamp(min=0)
        assert float((y.double() - ref).abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max()))


def test_gemm_f32_slices_give_the_same_bits_twice(ops):
    """Few tiles and a long K without alignment: slices of K in a fixed order."""
    r = np.random.default_rng(7)
    A, B = r.standard_normal((70, 6001)).astype(np.float32), r.standard_normal((6001, 90)).astype(np.float32)
    y = ops.gemm_f32(A, B, beta=0.0)
    assert np.array_equal(y, ops.gemm_f32(A, B, beta=0.0))
    assert np.max(np.abs(y - A.astype(np.float64) @ B.astype(np.float64))) <= 1e-5 * np.max(np.abs(y))


@pytest.mark.parametrize("M,N,K,tA,tB,lda,ldb,kernel",
                         [(37, 70, 50, 0, 0, 1 << 22, 1 << 22, "k_gemm_f32_direct"), (300, 250, 200, 0, 1, (1 << 22) + 1, (1 << 22) - 3, "k_gemm_f32_direct"),
                          (4000, 650, 64, 0, 0, 0, (1 << 24) - 1, "k_gemm_f32"), (4000, 650, 64, 1, 0, (1 << 24) + 1, (1 << 22) + 2, "k_gemm_f32_direct"),
                          (40, 100, 64, 0, 1, (1 << 24) - 1, (1 << 23) + 1, "k_gemm_f32_direct"), (9, 20, 3, 0, 0, 0, (1 << 24) + 3, "k_gemm_f32_plain"),
                          (21, 9, 7, 1, 1, (1 << 22) + 1, 0, "k_gemm_f32_plain")])
def test_gemm_f32_rows_far_apart(ops, M, N, K, tA, tB, lda, ldb, kernel):
    """Leading dimensions around those where a tile's 32-bit offsets end (2^22 to 2^24 floats): the kernel that takes them, a row
    bias and (not where a thread per output is the rule) a full one, against float64."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    ctx = ops.Context(0)

    def strided(rows, cols, ld):
        ld = ld or cols
        buf = torch.empty((rows - 1) * ld + cols, device="cuda")
        view = torch.as_strided(buf, (rows, cols), (ld, 1))
        view.copy_(torch.randn(rows, cols, device="cuda", generator=g))
        return buf, view, ld
    a, av, lda = strided(*((K, M) if tA else (M, K)), lda)
    b, bv, ldb = strided(*((N, K) if tB else (K, N)), ldb)
    ref = (av.t() if tA else av).double().contiguous() @ (bv.t() if tB else bv).double().contiguous()
    y = ctx.empty((M, N), torch.float32)
    buf, n = C.create_string_buffer(4096), C.c_int(-1)
    for kind, bias in ((L.BIAS_ROW, torch.randn(N, device="cuda", generator=g)), (L.BIAS_FULL, torch.randn(M, N, device="cuda", generator=g))):
        y.zero_()
        torch.cuda.synchronize()
        ctx.check(ctx.lib.sofie_hip_trace_begin(ctx.h))
        ctx.check(ctx.lib.sofie_hip_gemm_f32(ctx.h, tA, tB, M, N, K, 1.0, ctx.ptr(a), lda, ctx.ptr(b), ldb, 1.0, ctx.ptr(bias), kind, ctx.ptr(y), N,
                                             L.ACT_NONE))
        ctx.check(ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)))
        names = [line.split()[0] for line in buf.value.decode().splitlines()]
        ctx.sync()
        want = ref + bias.double()
        assert float((y.double() - want).abs().max()) <= 1e-5 * float(want.abs().max())
        assert kind == L.BIAS_FULL or names[0] == kernel, names
        assert K < 8 or "k_gemm_f32_plain" not in names, names
    ctx.close()


@pytest.mark.parametrize("tA,tB", [(0, 0), (1, 1)])
def test_gemm_f32_without_memory_for_slices(ops, tA, tB):
    """A long K on few tiles, recorded on a context that has no scratch buffer, and called while the graph is alive, when the
    buffer may not grow: K stays in one piece. Every replay and the eager call against float64; the slices come back with
    the graph gone."""
    M, N, K = 70, 90, 6001
    r = np.random.default_rng(11)
    A, B = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    ctx = ops.Context(0, stream=torch.cuda.Stream())
    a, b = ctx.dev(np.ascontiguousarray(A.T) if tA else A), ctx.dev(np.ascontiguousarray(B.T) if tB else B)
    y = ctx.empty((M, N), torch.float32)

    def call():
        return ctx.lib.sofie_hip_gemm_f32(ctx.h, tA, tB, M, N, K, 1.0, ctx.ptr(a), a.shape[1], ctx.ptr(b), b.shape[1], 0.0, None, L.BIAS_NONE,
                                          ctx.ptr(y), N, L.ACT_NONE)

    def check(run):
        y.zero_()
        torch.cuda.synchronize()
        ctx.check(run())
        ctx.sync()
        assert np.max(np.abs(y.cpu().numpy() - ref)) <= 1e-5 * np.max(np.abs(ref))
    graph = C.c_void_p()
    ctx.check(ctx.lib.sofie_hip_capture_begin(ctx.h))
    rc = call()
    ctx.check(ctx.lib.sofie_hip_capture_end(ctx.h, C.byref(graph)))
    ctx.check(rc)
    for _ in range(3):
        check(lambda: ctx.lib.sofie_hip_graph_launch(ctx.h, graph))
        check(call)
    ctx.check(ctx.lib.sofie_hip_graph_destroy(ctx.h, graph))
    check(call)
    ctx.close()
