"""GPU parity: every entry point of the C ABI against the CPU oracle on the same seeded
inputs, the reference's known-answer fixtures through the HIP path, and size-independent
properties at the full benchmark sizes. Bit-exact for int8 / index work; fp32 within 1e-5
relative (max |d| / max |ref|); FP8 within the tolerance written in the test."""
import json
import os
import sys

import numpy as np
import pytest
import torch

from sofie_amd import onnx_wire
import replay
from oracle import oracle

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
with open(os.path.join(GOLD, "expected.json")) as f:
    EXPECTED = json.load(f)


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    o.default_context()
    return o


@pytest.fixture(autouse=True)
def _announce(request):
    print("\n[case] %s" % request.node.nodeid, flush=True)
    sys.stdout.flush()
    yield


def rng(seed):
    return np.random.default_rng(seed)


def rel_err(y, ref):
    return float(np.max(np.abs(y.astype(np.float64) - ref.astype(np.float64))) / max(np.max(np.abs(ref)), 1e-30))


FP32_TOL = 1e-5
# FP8 GEMM: the share of sum|a_k b_k| that the matrix instruction's sums of eight products may drop (seven products of
# a group, each cut below 2^-13 of the group's largest: test_fp8_matrix_instruction_sums_groups_of_eight)
FP8_SUM_SLACK = 7 * 2.0 ** -13


# --------------------------------------------------------------------------- fixtures
@pytest.mark.parametrize("name", sorted(EXPECTED))
def test_reference_known_answers_through_hip(ops, name):
    entry = EXPECTED[name]
    graph = onnx_wire.load(os.path.join(GOLD, "onnx", name + ".onnx"))
    feeds = replay.fixture_feeds(entry, graph)
    y = replay.run_graph(graph, feeds, ops)
    want = np.array(entry["expected"], np.float32)
    assert y.size == want.size
    assert np.max(np.abs(y.reshape(-1) - want)) <= 1e-3   # the reference's own tolerance
    yo = replay.run_graph(graph, feeds, oracle)
    assert rel_err(y, yo) <= FP32_TOL
    if name.startswith("Conv") or name.startswith("MaxPool") or name.startswith("Einsum") or name.startswith("AvgPool"):
        assert np.array_equal(y, yo)


# --------------------------------------------------------------------------- fp32 transposed convolution
@pytest.mark.parametrize("cfg", [
    dict(N=2, C=4, H=5, W=6, OC=6, k=(3, 3), s=(2, 2), p=(1, 1, 1, 1), d=(1, 1), g=1, op=(0, 0)),
    dict(N=1, C=6, H=4, W=4, OC=4, k=(2, 3), s=(3, 2), p=(0, 1, 0, 1), d=(2, 1), g=2, op=(1, 1)),
    dict(N=2, C=3, H=7, W=5, OC=5, k=(4, 4), s=(2, 2), p=(1, 1, 1, 1), d=(1, 1), g=1, op=(1, 0)),
    dict(N=3, C=64, H=14, W=14, OC=96, k=(4, 4), s=(2, 2), p=(1, 1, 1, 1), d=(1, 1), g=1, op=(0, 0)),   # 128-channel tile
    dict(N=4, C=128, H=28, W=28, OC=64, k=(4, 4), s=(2, 2), p=(1, 1, 1, 1), d=(1, 1), g=1, op=(0, 0)),  # the benchmark's layer: phases on gathered sub-kernels
    dict(N=2, C=24, H=9, W=10, OC=16, k=(4, 4), s=(2, 2), p=(1, 1, 1, 1), d=(1, 1), g=2, op=(1, 1)),     # ... with groups and output padding
    dict(N=2, C=32, H=9, W=11, OC=32, k=(3, 3), s=(1, 1), p=(1, 1, 1, 1), d=(1, 1), g=4, op=(0, 0)),    # stride 1, groups
    dict(N=1, C=8, H=6, W=6, OC=8, k=(3, 3), s=(2, 2), p=(2, 2, 2, 2), d=(1, 1), g=1, op=(1, 1)),       # pad = kernel - 1
    dict(N=1, C=4, H=5, W=5, OC=4, k=(2, 2), s=(1, 1), p=(2, 2, 2, 2), d=(1, 1), g=1, op=(0, 0)),       # pad beyond the kernel
    dict(N=1, C=2, H=3, W=40, OC=3, k=(1, 9), s=(1, 4), p=(0, 2, 0, 2), d=(1, 1), g=1, op=(0, 3)),
    dict(N=1, C=2, H=2, W=2, OC=2, k=(31, 31), s=(1, 1), p=(0, 0, 0, 0), d=(1, 1), g=1, op=(0, 0)),     # large kernel
    dict(N=2, C=4, H=6, W=5, OC=6, k=(3, 4), s=(2, 3), p=(0, 2, 1, 0), d=(1, 1), g=2, op=(1, 2)),       # begin != end pads
    dict(N=1, C=3, H=5, W=7, OC=2, k=(3, 3), s=(2, 1), p=(2, 0, 0, 1), d=(2, 2), g=1, op=(0, 0)),
])
def test_conv_transpose2d_f32(ops, cfg):
    """ConvTranspose through the implicit-GEMM kernel over the zero-interleaved input against the oracle's
    GEMM + col2im restatement of the reference: strides, dilations, groups, begin/end pads (also larger than
    the kernel reach), output padding, bias and ReLU. Tolerance 1e-5 relative (accumulation order differs)."""
    r = rng(40 + cfg["C"] + cfg["H"])
    x = r.standard_normal((cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.float32)
    w = (r.standard_normal((cfg["C"], cfg["OC"] // cfg["g"]) + cfg["k"]) * 0.2).astype(np.float32)
    b = r.standard_normal(cfg["OC"]).astype(np.float32)
    for bias, relu in ((b, False), (None, True)):
        y = ops.conv_transpose2d_f32(x, w, bias, cfg["p"], cfg["s"], cfg["d"], cfg["g"], cfg["op"], relu)
        ref = oracle.conv_transpose2d_f32(x, w, bias, cfg["p"], cfg["s"], cfg["d"], cfg["g"], cfg["op"], relu)
        assert y.shape == ref.shape
        assert rel_err(y, ref) <= FP32_TOL


def test_conv_transpose2d_f32_is_the_adjoint_of_conv2d(ops):
    """<conv(x, w), y> = <x, conv_transpose(y, w)> for matching geometry, at a size the oracle would take long for."""
    r = rng(41)
    N, C, H, W, OC = 4, 48, 28, 28, 64
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((OC, C, 4, 4)) * 0.1).astype(np.float32)
    cy = ops.conv2d_f32(x, w, None, (1, 1), (2, 2))
    y = r.standard_normal(cy.shape).astype(np.float32)
    # conv weights [OC, C, kh, kw] are ConvTranspose weights for an input with OC channels and C outputs
    ty = ops.conv_transpose2d_f32(y, w, None, (1, 1, 1, 1), (2, 2))
    assert ty.shape == x.shape
    lhs = float(np.sum(cy.astype(np.float64) * y))
    rhs = float(np.sum(x.astype(np.float64) * ty))
    assert abs(lhs - rhs) <= 1e-5 * max(abs(lhs), abs(rhs), 1.0) * 10


# --------------------------------------------------------------------------- batch normalisation
@pytest.mark.parametrize("shape", [(3, 5, 7, 6), (4, 9), (2, 3, 10), (2, 64, 56, 56), (70000, 2), (1, 1, 1, 1)])
def test_batchnorm_f32(ops, shape):
    """Same rounding steps as the oracle's restatement of the reference (subtract, multiply by the folded scale, add):
    identical bits, with and without the fused ReLU; vector and scalar planes, more planes than one launch holds."""
    r = rng(60 + len(shape) + shape[1])
    C = shape[1]
    x = (r.standard_normal(shape) * 3).astype(np.float32)
    g, b = r.uniform(0.5, 2, C).astype(np.float32), r.standard_normal(C).astype(np.float32)
    m, v = r.standard_normal(C).astype(np.float32), r.uniform(0.1, 3, C).astype(np.float32)
    for eps, relu in ((1e-5, False), (1e-3, True)):
        y = ops.batchnorm_f32(x, g, b, m, v, eps, relu)
        assert np.array_equal(y, oracle.batchnorm_f32(x, g, b, m, v, eps, relu))


# --------------------------------------------------------------------------- fp32 gemm
@pytest.mark.parametrize("M,N,K,tA,tB,alpha,beta,relu", [
    (256, 128, 64, 0, 0, 1.0, 1.0, True),      # MLP layer 1 of the fp32 configuration
    (256, 64, 128, 0, 0, 1.0, 1.0, True),
    (256, 8, 64, 0, 0, 1.0, 1.0, False),
    (37, 29, 53, 0, 1, 1.0, 1.0, False),
    (130, 67, 19, 1, 0, 0.5, 2.0, True),
    (65, 130, 33, 1, 1, -1.25, 0.0, False),
    (1, 1, 1, 0, 0, 1.0, 0.0, False),
    (700, 900, 257, 0, 1, 1.0, 1.0, True),
    (2048, 2304, 512, 0, 0, 1.0, 1.0, False),  # large enough for the 128x128 tiles
])
def test_gemm_f32(ops, M, N, K, tA, tB, alpha, beta, relu):
    r = rng(100 + M + N + K)
    A = r.standard_normal((K, M) if tA else (M, K)).astype(np.float32)
    B = r.standard_normal((N, K) if tB else (K, N)).astype(np.float32)
    bias = r.standard_normal(N).astype(np.float32) if beta != 0.0 else None
    y = ops.gemm_f32(A, B, bias, alpha, beta, bool(tA), bool(tB), relu)
    if M * N * K <= 64 * 1024 * 1024:
        ref = oracle.gemm_f32(A, B, bias, alpha, beta, bool(tA), bool(tB), relu)
    else:
        a = (A.T if tA else A).astype(np.float64)
        b = (B.T if tB else B).astype(np.float64)
        ref = alpha * (a @ b) + (beta * bias if bias is not None else 0.0)
        ref = np.maximum(ref, 0) if relu else ref
    assert y.shape == ref.shape
    assert rel_err(y, ref) <= FP32_TOL


@pytest.mark.parametrize("M,N,K,tB,alpha,beta,relu,kern", [
    # the kernel that fetches its operands by LDS-DMA: ragged tiles along M and N, one K step and an odd number of them,
    # B as [K,N] and as [N,K], with and without a bias row
    (2100, 2052, 96, 0, 1.0, 1.0, True, "k_gemm_f32_dma"),
    (2100, 2052, 96, 1, -0.5, 2.0, False, "k_gemm_f32_dma"),
    (2048, 2304, 32, 1, 1.0, 0.0, False, "k_gemm_f32_dma"),
    (2304, 2048, 64, 0, 1.0, 0.0, True, "k_gemm_f32_dma"),
    (4096, 2048, 160, 1, 1.0, 1.0, True, "k_gemm_f32_dma"),
    # ... with 64 x 64 tiles where there are fewer than 256 tiles of 128 x 128
    (700, 900, 256, 1, 1.0, 1.0, True, "k_gemm_f32_dma64"),
    (700, 900, 96, 0, 0.25, -1.0, False, "k_gemm_f32_dma64"),
    (1024, 1024, 1024, 0, 1.0, 1.0, True, "k_gemm_f32_dma64"),
    (300, 520, 32, 1, 1.0, 0.0, False, "k_gemm_f32_dma64"),
    # ... and what it leaves to the register-staged kernel: K that is no multiple of 32, N that is no multiple of 4 with B [K,N]
    (2100, 2052, 100, 1, 1.0, 1.0, True, "k_gemm_f32"),
    (2100, 2050, 96, 0, 1.0, 1.0, True, "k_gemm_f32"),
])
def test_gemm_f32_large(ops, M, N, K, tB, alpha, beta, relu, kern):
    r = rng(900 + M + N + K + tB)
    A = r.standard_normal((M, K)).astype(np.float32)
    B = r.standard_normal((N, K) if tB else (K, N)).astype(np.float32)
    bias = r.standard_normal(N).astype(np.float32) if beta != 0.0 else None
    y, names = _kernels_of(ops, lambda: ops.gemm_f32(A, B, bias, alpha, beta, False, bool(tB), relu))
    assert names == [kern], names
    ref = alpha * (A.astype(np.float64) @ (B.T if tB else B).astype(np.float64)) + (beta * bias if bias is not None else 0.0)
    ref = np.maximum(ref, 0) if relu else ref
    assert y.shape == ref.shape
    assert rel_err(y, ref) <= FP32_TOL
    # sampled rows against the oracle's own summation (the C restatement of the reference's sgemm_ call)
    rows = np.concatenate([np.arange(0, 8), r.integers(0, M, 8), np.arange(M - 8, M)])
    assert rel_err(y[rows], oracle.gemm_f32(A[rows], B, bias, alpha, beta, False, bool(tB), relu)) <= FP32_TOL


def test_gemm_f32_large_integer_data_is_exact_with_a_column_bias(ops):
    """Integer operands make every order of summation exact: the LDS-DMA kernel against int64 numpy, with the bias as a
    column (one value per row of the output), through the C ABI."""
    from sofie_amd import lib as L
    r = rng(901)
    M, N, K = 2200, 2048, 128
    A = r.integers(-8, 9, (M, K)).astype(np.float32)
    B = r.integers(-8, 9, (N, K)).astype(np.float32)
    col = r.integers(-50, 50, M).astype(np.float32)
    ctx = ops.default_context()
    a, b, c = ctx.dev(A), ctx.dev(B), ctx.dev(col)
    y = ctx.empty((M, N), torch.float32)
    ctx.check(ctx.lib.sofie_hip_gemm_f32(ctx.h, 0, 1, M, N, K, 2.0, ctx.ptr(a), K, ctx.ptr(b), K, 3.0, ctx.ptr(c), L.BIAS_COL,
                                         ctx.ptr(y), N, L.ACT_RELU))
    ctx.sync()
    ref = np.maximum(2 * (A.astype(np.int64) @ B.astype(np.int64).T) + 3 * col.astype(np.int64)[:, None], 0)
    assert np.array_equal(y.cpu().numpy(), ref)


@pytest.mark.parametrize("M,N,K,tB", [
    (1, 1024, 1024, 0), (8, 4096, 2048, 0), (5, 1000, 260, 0), (32, 516, 1028, 0), (33, 768, 512, 0), (64, 2048, 4096, 0),
    (1, 1024, 1024, 1), (7, 1003, 516, 1), (32, 130, 2048, 1), (40, 999, 1000, 1), (64, 4096, 1024, 1), (16, 256, 256, 0),
])
def test_gemm_f32_few_rows(ops, M, N, K, tB):
    """A layer on a small batch (at most 64 rows of A) runs as a pass over B with K cut into slices
    (k_gemm_f32_skinny, and k_gemm_f32_skinny_finish where there is more than one slice): both layouts of B, ragged
    column blocks, K that is no multiple of a wavefront's chunk of 8 or of a slice, every bias kind, alpha, beta, ReLU;
    1e-5 relative against the oracle's own summation and against float64."""
    r = rng(930 + M + N + K + tB)
    A = r.standard_normal((M, K)).astype(np.float32)
    B = r.standard_normal((N, K) if tB else (K, N)).astype(np.float32)
    for kind in range(3):
        bias = [None, r.standard_normal(N).astype(np.float32), r.standard_normal((M, N)).astype(np.float32)][kind]
        alpha, beta, relu = [1.0, 0.5, -2.0][kind], (0.0 if bias is None else [1.0, 0.25][kind % 2]), kind != 1
        y, names = _kernels_of(ops, lambda: ops.gemm_f32(A, B, bias, alpha, beta, False, bool(tB), relu))
        assert names in (["k_gemm_f32_skinny"], ["k_gemm_f32_skinny", "k_gemm_f32_skinny_finish"]), names
        ref = alpha * (A.astype(np.float64) @ (B.T if tB else B).astype(np.float64)) + (beta * bias if bias is not None else 0.0)
        ref = np.maximum(ref, 0) if relu else ref
        assert y.shape == ref.shape
        assert rel_err(y, ref) <= FP32_TOL
        assert rel_err(y, oracle.gemm_f32(A, B, bias, alpha, beta, False, bool(tB), relu)) <= FP32_TOL


@pytest.mark.parametrize("M,N,K,tB", [(128, 1024, 4096, 0), (200, 520, 2048, 1), (96, 2048, 1024, 0), (512, 260, 8192, 1)])
def test_gemm_f32_few_tiles_long_k_in_slices(ops, M, N, K, tB):
    """Products whose 64 x 64 tiles cover less than half of the compute units, with a long K: the LDS-DMA kernel runs
    on slices of K and the pass of the few-rows kernel adds them in order (the trace shows both); every bias kind,
    1e-5 relative against float64 and against the oracle, and the same bits on a second call."""
    r = rng(940 + M + N + K + tB)
    A = r.standard_normal((M, K)).astype(np.float32)
    B = r.standard_normal((N, K) if tB else (K, N)).astype(np.float32)
    for kind in range(3):
        bias = [None, r.standard_normal(N).astype(np.float32), r.standard_normal((M, N)).astype(np.float32)][kind]
        alpha, beta, relu = [1.0, 0.5, -2.0][kind], (0.0 if bias is None else [1.0, 0.25][kind % 2]), kind != 1
        y, names = _kernels_of(ops, lambda: ops.gemm_f32(A, B, bias, alpha, beta, False, bool(tB), relu))
        # (a bias given for every output element is not a case of the LDS-DMA kernel)
        assert names == (["k_gemm_f32"] if kind == 2 else ["k_gemm_f32_dma64", "k_gemm_f32_skinny_finish"]), names
        ref = alpha * (A.astype(np.float64) @ (B.T if tB else B).astype(np.float64)) + (beta * bias if bias is not None else 0.0)
        ref = np.maximum(ref, 0) if relu else ref
        assert rel_err(y, ref) <= FP32_TOL
        assert rel_err(y, oracle.gemm_f32(A, B, bias, alpha, beta, False, bool(tB), relu)) <= FP32_TOL
        assert np.array_equal(y, ops.gemm_f32(A, B, bias, alpha, beta, False, bool(tB), relu))


def test_gemm_f32_few_rows_integer_data_is_exact_with_a_column_bias(ops):
    """Integer operands make every order of summation exact: the sliced pass over B against int64 numpy, bias as a
    column (one value per row), rows of A and Y wider than the matrices, through the C ABI."""
    from sofie_amd import lib as L
    r = rng(931)
    M, N, K = 48, 1536, 2052
    A = np.zeros((M, K + 12), dtype=np.float32)
    A[:, :K] = r.integers(-8, 9, (M, K))
    A[:, K:] = np.nan                                     # what lies behind K in a row must not reach the sums
    B = r.integers(-8, 9, (K, N)).astype(np.float32)
    col = r.integers(-50, 50, M).astype(np.float32)
    ctx = ops.default_context()
    a, b, c = ctx.dev(A), ctx.dev(B), ctx.dev(col)
    y = ctx.empty((M, N + 4), torch.float32)
    y.fill_(-7.0)
    ctx.check(ctx.lib.sofie_hip_gemm_f32(ctx.h, 0, 0, M, N, K, 2.0, ctx.ptr(a), K + 12, ctx.ptr(b), N, 3.0, ctx.ptr(c), L.BIAS_COL,
                                         ctx.ptr(y), N + 4, L.ACT_RELU))
    ctx.sync()
    ref = np.maximum(2 * (A[:, :K].astype(np.int64) @ B.astype(np.int64)) + 3 * col.astype(np.int64)[:, None], 0)
    got = y.cpu().numpy()
    assert np.array_equal(got[:, :N], ref)
    assert np.all(got[:, N:] == -7.0)


def test_gemm_f32_full_bias_and_error_path(ops):
    r = rng(7)
    A = r.standard_normal((50, 20)).astype(np.float32)
    B = r.standard_normal((20, 30)).astype(np.float32)
    Cfull = r.standard_normal((50, 30)).astype(np.float32)
    assert rel_err(ops.gemm_f32(A, B, Cfull), oracle.gemm_f32(A, B, Cfull)) <= FP32_TOL
    with pytest.raises(ops.SofieHipError, match="beta"):
        ops.gemm_f32(A, B, None, 1.0, 1.0)


def test_gemm_f32_integer_data_is_exact(ops):
    r = rng(8)
    A = r.integers(-8, 9, (96, 200)).astype(np.float32)
    B = r.integers(-8, 9, (200, 72)).astype(np.float32)
    assert np.array_equal(ops.gemm_f32(A, B, beta=0.0), A.astype(np.int64) @ B.astype(np.int64))


# --------------------------------------------------------------------------- fp32 conv
@pytest.mark.parametrize("cfg", [
    dict(N=2, C=3, H=7, W=6, OC=4, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, bias=True, relu=True),
    dict(N=1, C=4, H=9, W=8, OC=6, k=(3, 2), p=(0, 1), s=(2, 1), d=(1, 1), g=2, bias=False, relu=False),
    dict(N=2, C=2, H=8, W=8, OC=2, k=(2, 2), p=(1, 1), s=(2, 2), d=(1, 1), g=1, bias=True, relu=False),
    dict(N=1, C=2, H=10, W=9, OC=3, k=(3, 3), p=(2, 2), s=(1, 1), d=(2, 2), g=1, bias=True, relu=True),
    dict(N=3, C=16, H=20, W=20, OC=70, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, bias=True, relu=True),
    dict(N=2, C=64, H=56, W=56, OC=128, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, bias=True, relu=True),
    dict(N=2, C=1, H=40, W=40, OC=32, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, bias=True, relu=True),
    dict(N=1, C=8, H=12, W=300, OC=16, k=(1, 1), p=(0, 0), s=(1, 1), d=(1, 1), g=1, bias=False, relu=False),
    dict(N=1, C=3, H=30, W=30, OC=5, k=(7, 7), p=(3, 3), s=(2, 2), d=(1, 1), g=1, bias=True, relu=False),
    # channel blocks staged under the matrix loop (the kernel with two LDS buffers): two groups with 64-channel tiles
    # and a stride; a dilation with a ragged second channel tile; a last pixel tile that is nearly empty
    dict(N=2, C=16, H=9, W=19, OC=96, k=(3, 3), p=(1, 1), s=(2, 2), d=(1, 1), g=2, bias=True, relu=True),
    dict(N=1, C=8, H=12, W=12, OC=130, k=(3, 3), p=(2, 2), s=(1, 1), d=(2, 2), g=1, bias=True, relu=False),
    dict(N=3, C=12, H=13, W=10, OC=64, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, bias=False, relu=True),
    # begin pads that differ from the end pads (top, left, bottom, right), as SAME_UPPER / SAME_LOWER make them for
    # even kernels: the oracle convolves the explicitly padded tensor
    dict(N=2, C=3, H=8, W=8, OC=4, k=(4, 4), p=(1, 1, 2, 2), s=(1, 1), d=(1, 1), g=1, bias=True, relu=False),
    dict(N=2, C=3, H=8, W=8, OC=4, k=(4, 4), p=(2, 2, 1, 1), s=(1, 1), d=(1, 1), g=1, bias=True, relu=True),
    dict(N=1, C=4, H=7, W=6, OC=6, k=(3, 2), p=(0, 2, 1, 0), s=(1, 1), d=(1, 1), g=2, bias=True, relu=False),
    dict(N=2, C=16, H=15, W=18, OC=96, k=(3, 3), p=(0, 0, 1, 1), s=(2, 2), d=(1, 1), g=1, bias=True, relu=True),
    dict(N=1, C=8, H=12, W=12, OC=130, k=(3, 3), p=(3, 0, 1, 4), s=(1, 1), d=(2, 2), g=1, bias=False, relu=False),
])
def test_conv2d_f32(ops, cfg):
    r = rng(200 + cfg["C"] + cfg["OC"])
    x = r.uniform(0, 1, (cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.float32)
    fan = cfg["C"] // cfg["g"] * cfg["k"][0] * cfg["k"][1]
    w = (r.standard_normal((cfg["OC"], cfg["C"] // cfg["g"]) + cfg["k"]) * np.sqrt(2.0 / fan)).astype(np.float32)
    b = (r.standard_normal(cfg["OC"]) * 0.1).astype(np.float32) if cfg["bias"] else None
    y = ops.conv2d_f32(x, w, b, cfg["p"], cfg["s"], cfg["d"], cfg["g"], cfg["relu"])
    ref = oracle.conv2d_f32(x, w, b, cfg["p"], cfg["s"], cfg["d"], cfg["g"], cfg["relu"])
    assert y.shape == ref.shape
    assert rel_err(y, ref) <= FP32_TOL


def _kernels_of(ops, call):
    """Names of the kernels that `call` launches on the default context (sofie_hip_trace_begin / _end)."""
    import ctypes as C
    ctx = ops.default_context()
    buf = C.create_string_buffer(4096)
    n = C.c_int(-1)
    assert ctx.lib.sofie_hip_trace_begin(ctx.h) == 0
    try:
        out = call()
    finally:
        assert ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)) == 0
    return out, [l.split()[0] for l in buf.value.decode().splitlines()]


@pytest.mark.parametrize("cfg", [
    # channel counts that are no multiple of 4 (the copied weights' rows are padded), a ragged second channel tile,
    # groups, a stride and a dilation, asymmetric pads, one or several patch requests per thread, a nearly empty last
    # pixel tile, a grid small enough for more than three workgroups per compute unit
    # ... kernels 1 to 3 columns wide take the loop without a table of offsets (K ordered by channel pairs); a dilation
    # along the columns, an odd number of channels per group and a kernel 5 columns wide take the general loop
    dict(N=3, C=16, H=20, W=20, OC=70, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, pairs=True),
    dict(N=2, C=16, H=9, W=19, OC=98, k=(3, 3), p=(1, 1), s=(2, 2), d=(1, 1), g=2, pairs=True),
    dict(N=1, C=8, H=12, W=12, OC=130, k=(3, 3), p=(3, 0, 1, 4), s=(1, 1), d=(2, 2), g=1, pairs=False),
    dict(N=2, C=64, H=56, W=56, OC=128, k=(3, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, pairs=True),
    dict(N=5, C=24, H=17, W=33, OC=33, k=(5, 2), p=(2, 0, 2, 1), s=(1, 1), d=(1, 1), g=1, pairs=True),
    dict(N=2, C=12, H=14, W=11, OC=40, k=(2, 3), p=(0, 1, 1, 1), s=(1, 2), d=(2, 1), g=2, pairs=True),
    dict(N=40, C=32, H=6, W=6, OC=64, k=(1, 1), p=(0, 0), s=(1, 1), d=(1, 1), g=1, pairs=True),
    dict(N=2, C=20, H=9, W=12, OC=24, k=(3, 1), p=(1, 0, 1, 0), s=(1, 1), d=(2, 3), g=1, pairs=True),
    dict(N=3, C=9, H=13, W=10, OC=20, k=(2, 3), p=(1, 1), s=(1, 1), d=(1, 1), g=1, pairs=False),
    dict(N=2, C=4, H=11, W=16, OC=8, k=(2, 5), p=(1, 2, 0, 2), s=(1, 1), d=(1, 1), g=1, pairs=False),
])
def test_conv2d_f32_operands_by_lds_dma(ops, cfg):
    """The kernel that fetches both operands by LDS-DMA from weights copied into the [K][channel] order: the trace names
    it (and which of its two matrix loops ran), and its results are the oracle's within the fp32 tolerance (1e-5
    relative), with and without bias and ReLU."""
    r = rng(230 + cfg["C"] + cfg["OC"])
    x = r.standard_normal((cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.float32)
    fan = cfg["C"] // cfg["g"] * cfg["k"][0] * cfg["k"][1]
    w = (r.standard_normal((cfg["OC"], cfg["C"] // cfg["g"]) + cfg["k"]) * np.sqrt(2.0 / fan)).astype(np.float32)
    b = (r.standard_normal(cfg["OC"]) * 0.1).astype(np.float32)
    for bias, relu in ((b, True), (None, False)):
        y, names = _kernels_of(ops, lambda: ops.conv2d_f32(x, w, bias, cfg["p"], cfg["s"], cfg["d"], cfg["g"], relu))
        # (a layer of fewer tiles than compute units is cut into slices of channel blocks, which a second pass adds)
        assert names[:2] == ["k_transpose_weights", "k_conv2d_f32_dma_pairs" if cfg["pairs"] else "k_conv2d_f32_dma"], names
        assert names[2:] in ([], ["k_conv_f32_split_finish"]), names
        ref = oracle.conv2d_f32(x, w, bias, cfg["p"], cfg["s"], cfg["d"], cfg["g"], relu)
        assert y.shape == ref.shape
        assert rel_err(y, ref) <= FP32_TOL


@pytest.mark.parametrize("N,C,H,W,OC,k,g", [(1, 64, 56, 56, 128, 3, 1), (2, 48, 20, 30, 70, 3, 1), (1, 64, 28, 28, 64, 1, 1),
                                            (3, 32, 14, 14, 96, 3, 2), (1, 128, 9, 9, 40, 2, 1)])
def test_conv2d_f32_on_few_images_sums_channel_slices(ops, N, C, H, W, OC, k, g):
    """A layer with fewer tiles than the device has compute units runs on 64 x 64 tiles with its channel blocks dealt
    to slices (k_conv2d_f32_dma writes raw sums, k_conv_f32_split_finish adds them in slice order, then bias and
    ReLU): the trace shows the second pass, the results are the oracle's within 1e-5 relative, and a second call
    gives the same bits (the order of the sums is fixed)."""
    r = rng(260 + C + OC + k)
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((OC, C // g, k, k)) * np.sqrt(2.0 / (C // g * k * k))).astype(np.float32)
    b = (r.standard_normal(OC) * 0.1).astype(np.float32)
    pads = (k // 2, k // 2)
    for bias, relu in ((b, True), (None, False)):
        y, names = _kernels_of(ops, lambda: ops.conv2d_f32(x, w, bias, pads, (1, 1), (1, 1), g, relu))
        assert names[-1] == "k_conv_f32_split_finish" and names[-2].startswith("k_conv2d_f32_dma"), names
        ref = oracle.conv2d_f32(x, w, bias, pads, (1, 1), (1, 1), g, relu)
        assert y.shape == ref.shape
        assert rel_err(y, ref) <= FP32_TOL
        assert np.array_equal(y, ops.conv2d_f32(x, w, bias, pads, (1, 1), (1, 1), g, relu))


def test_conv_transpose2d_f32_phases_by_lds_dma(ops):
    """The benchmark's upsampling layer (4x4, stride 2) runs as four phases in one launch of the LDS-DMA kernel on
    gathered sub-kernels; an odd output size gives the phases different extents."""
    r = rng(77)
    for (N, C, H, W, OC, op, k, kern) in ((3, 128, 28, 28, 64, (0, 0), 4, "k_conv2d_f32_dma_pairs_phases"),
                                          (2, 24, 9, 10, 18, (1, 1), 4, "k_conv2d_f32_dma_pairs_phases"),
                                          (2, 16, 9, 10, 18, (1, 1), 3, "k_conv2d_f32_dma_phases")):   # phases 2 and 1 columns wide
        x = r.standard_normal((N, C, H, W)).astype(np.float32)
        w = (r.standard_normal((C, OC, k, k)) * 0.2).astype(np.float32)
        b = r.standard_normal(OC).astype(np.float32)
        y, names = _kernels_of(ops, lambda: ops.conv_transpose2d_f32(x, w, b, (1, 1, 1, 1), (2, 2), (1, 1), 1, op, True))
        # (the small layers have fewer tiles than the device has compute units: their channel blocks are cut into
        # slices that a second pass adds)
        assert names[:2] == ["k_gather_phase_weights", kern] and names[2:] in ([], ["k_conv_f32_split_finish"]), names
        ref = oracle.conv_transpose2d_f32(x, w, b, (1, 1, 1, 1), (2, 2), (1, 1), 1, op, True)
        assert rel_err(y, ref) <= FP32_TOL


def test_constant_weights_keep_the_kernels_layout_of_a_weight_tensor(ops):
    """sofie_hip_constant_weights: with the promise made, the copy of a weight tensor in the kernel's layout is made by
    the first call only (the trace shows the small kernel once), results stay what they were, a second geometry on
    the same tensor gets a copy of its own, taking the promise back returns to a copy per call, and a graph recorded
    with the promise made holds the convolution alone and replays to the same result."""
    import ctypes as C
    from sofie_amd import lib as L
    r = rng(4242)
    ctx = ops.Context(0)
    x = r.standard_normal((3, 16, 20, 20)).astype(np.float32)
    w = (r.standard_normal((40, 16, 3, 3)) * 0.1).astype(np.float32)
    b = r.standard_normal(40).astype(np.float32)
    xt = r.standard_normal((2, 24, 9, 10)).astype(np.float32)
    wt = (r.standard_normal((24, 18, 4, 4)) * 0.2).astype(np.float32)
    dx, dw, db, dxt, dwt = ctx.dev(x), ctx.dev(w), ctx.dev(b), ctx.dev(xt), ctx.dev(wt)
    ctx.sync()

    def traced(call):
        buf = C.create_string_buffer(4096)
        n = C.c_int(-1)
        assert ctx.lib.sofie_hip_trace_begin(ctx.h) == 0
        out = call()
        assert ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)) == 0
        # (layers this small are cut into slices of channel blocks; the pass that adds them is not what this test is about)
        return out, [l.split()[0] for l in buf.value.decode().splitlines() if l.split()[0] != "k_conv_f32_split_finish"]

    conv = lambda pads=(1, 1): ops.conv2d_f32(dx, dw, db, pads, (1, 1), (1, 1), 1, True, ctx=ctx)
    convt = lambda: ops.conv_transpose2d_f32(dxt, dwt, None, (1, 1, 1, 1), (2, 2), (1, 1), 1, (0, 0), False, ctx=ctx)
    y0, names = traced(conv)
    assert names == ["k_transpose_weights", "k_conv2d_f32_dma_pairs"]
    t0, names = traced(convt)
    assert names == ["k_gather_phase_weights", "k_conv2d_f32_dma_pairs_phases"]
    ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, 1))
    y1, names = traced(conv)
    assert names == ["k_transpose_weights", "k_conv2d_f32_dma_pairs"]          # the first call with the promise lays it out
    for _ in range(2):
        y2, names = traced(conv)
        assert names == ["k_conv2d_f32_dma_pairs"] and torch.equal(y2, y0)
    t1, names = traced(convt)
    assert names == ["k_gather_phase_weights", "k_conv2d_f32_dma_pairs_phases"]
    t2, names = traced(convt)
    assert names == ["k_conv2d_f32_dma_pairs_phases"] and torch.equal(t2, t0)
    # the same tensor read as a grouped convolution's weights: another layout, another copy
    wg_ = ctx.dev((r.standard_normal((40, 8, 3, 3)) * 0.1).astype(np.float32))
    yg0 = ops.conv2d_f32(dx, wg_, db, (1, 1), (1, 1), (1, 1), 2, False, ctx=ctx)
    yg1, names = traced(lambda: ops.conv2d_f32(dx, wg_, db, (1, 1), (1, 1), (1, 1), 2, False, ctx=ctx))
    assert names == ["k_conv2d_f32_dma_pairs"] and torch.equal(yg1, yg0)
    # recorded with the promise made: the graph holds the convolution alone
    y3 = ctx.empty(tuple(y0.shape), torch.float32)
    call = lambda: ctx.check(ctx.lib.sofie_hip_conv2d_f32(ctx.h, ctx.ptr(dx), ctx.ptr(dw), ctx.ptr(db), ctx.ptr(y3), 3, 16, 20, 20, 40,
                                                          3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1))
    ctx.check(ctx.lib.sofie_hip_capture_begin(ctx.h))
    call()
    graph = C.c_void_p()
    ctx.check(ctx.lib.sofie_hip_capture_end(ctx.h, C.byref(graph)))
    assert ctx.lib.sofie_hip_constant_weights(ctx.h, 0) == L.EINVAL          # the graph may hold a kept copy's address
    for _ in range(2):
        y3.zero_()
        ctx.sync()
        ctx.check(ctx.lib.sofie_hip_graph_launch(ctx.h, graph))
        ctx.sync()
        assert torch.equal(y3, y0)
    ctx.check(ctx.lib.sofie_hip_graph_destroy(ctx.h, graph))
    ctx.check(ctx.lib.sofie_hip_constant_weights(ctx.h, 0))
    y4, names = traced(conv)
    assert names == ["k_transpose_weights", "k_conv2d_f32_dma_pairs"] and torch.equal(y4, y0)
    assert rel_err(y0.cpu().numpy(), oracle.conv2d_f32(x, w, b, (1, 1), relu=True)) <= FP32_TOL


def test_conv2d_f32_integer_data_is_exact(ops):
    r = rng(9)
    x = r.integers(-6, 7, (2, 8, 11, 13)).astype(np.float32)
    w = r.integers(-4, 5, (10, 8, 3, 3)).astype(np.float32)
    y = ops.conv2d_f32(x, w, None, (1, 1))
    assert np.array_equal(y, oracle.conv2d_f32(x, w, None, (1, 1)))


def test_relu_and_maxpool_f32(ops):
    r = rng(10)
    x = r.standard_normal((3, 5, 17, 19)).astype(np.float32)
    assert np.array_equal(ops.relu_f32(x), oracle.relu_f32(x))
    odd = r.standard_normal(1027).astype(np.float32)
    assert np.array_equal(ops.relu_f32(odd), np.maximum(odd, 0))
    for k, s, p in [((2, 2), (2, 2), (0, 0, 0, 0)), ((3, 2), (1, 1), (0, 0, 0, 0)), ((3, 3), (2, 2), (1, 1, 1, 1))]:
        assert np.array_equal(ops.maxpool2d(x, k, s, p), oracle.maxpool2d(x, k, s, p))


@pytest.mark.parametrize("cfg", [
    dict(shape=(2, 3, 6, 7, 8), k=(2, 3, 2), s=(2, 1, 2), p=(0, 0, 0, 0, 0, 0)),
    dict(shape=(1, 2, 5, 5, 5), k=(3, 3, 3), s=(1, 1, 1), p=(1, 1, 1, 1, 1, 1)),
    dict(shape=(3, 5, 9, 6, 11), k=(2, 2, 4), s=(1, 2, 3), p=(1, 0, 2, 0, 1, 3)),
    dict(shape=(1, 1, 4, 4, 4), k=(4, 4, 4), s=(1, 1, 1), p=(0, 0, 0, 0, 0, 0)),        # the global pooling
])
def test_pool3d_f32(ops, cfg):
    """Max and average pooling over three spatial axes against the oracle: the maximum exactly, the average exactly too
    (same order of additions, one division), with padding cells counted and not."""
    x = rng(60 + cfg["shape"][4]).standard_normal(cfg["shape"]).astype(np.float32)
    assert np.array_equal(ops.pool3d(x, cfg["k"], cfg["s"], cfg["p"]), oracle.pool3d(x, cfg["k"], cfg["s"], cfg["p"]))
    for include in (False, True):
        y = ops.pool3d(x, cfg["k"], cfg["s"], cfg["p"], average=True, count_include_pad=include)
        assert np.array_equal(y, oracle.pool3d(x, cfg["k"], cfg["s"], cfg["p"], average=True, count_include_pad=include))


def test_pool3d_refuses_what_it_cannot_do(ops):
    import ctypes as C
    from sofie_amd import lib as L
    ctx = ops.default_context()
    x = ctx.dev(np.zeros((1, 1, 4, 4, 4), np.float32))
    y = ctx.empty((1, 1, 4, 4, 4), torch.float32)
    arr = lambda *v: (C.c_int * len(v))(*v)
    # kernel larger than the padded volume; a pad as large as the window for an average over inside cells only
    assert ctx.lib.sofie_hip_maxpool3d_f32(ctx.h, ctx.ptr(x), ctx.ptr(y), 1, arr(4, 4, 4), arr(5, 1, 1), arr(0, 0, 0, 0, 0, 0), arr(1, 1, 1)) == L.EINVAL
    assert ctx.lib.sofie_hip_avgpool3d_f32(ctx.h, ctx.ptr(x), ctx.ptr(y), 1, arr(4, 4, 4), arr(2, 2, 2), arr(2, 0, 0, 0, 0, 0), arr(1, 1, 1), 0) == L.EINVAL
    assert ctx.lib.sofie_hip_avgpool3d_f32(ctx.h, ctx.ptr(x), ctx.ptr(y), 1, arr(4, 4, 4), arr(2, 2, 2), arr(0, 0, 0, 0, 0, 0), arr(1, 0, 1), 0) == L.EINVAL


# --------------------------------------------------------------------------- int8
def test_quantize_dequantize(ops):
    r = rng(11)
    x = np.concatenate([r.uniform(0, 1, 5001), (np.arange(-300, 300) + 0.5) / 255.0, [1e9, -1e9]]).astype(np.float32)
    s = np.float32(1 / 255)
    q = ops.quantize_f32_s8(x, s, -128)
    assert np.array_equal(q, oracle.quantize_f32_s8(x, s, -128))
    assert np.array_equal(ops.dequantize_s8_f32(q, s, -128), oracle.dequantize_s8_f32(q, s, -128))
    q8 = r.integers(-128, 128, (2, 6, 9, 8)).astype(np.int8)
    from sofie_amd import lib as L
    nhwc = ops.relayout_s8(q8, L.LAYOUT_NCHW, L.LAYOUT_NHWC)
    assert np.array_equal(nhwc, q8.transpose(0, 2, 3, 1))
    assert np.array_equal(ops.relayout_s8(nhwc, L.LAYOUT_NHWC, L.LAYOUT_NCHW), q8)
    assert np.array_equal(ops.maxpool2d(q8, (2, 2), (2, 2)), oracle.maxpool2d(q8, (2, 2), (2, 2)))
    pooled_nhwc = ops.maxpool2d(nhwc, (2, 2), (2, 2), layout=L.LAYOUT_NHWC)
    assert np.array_equal(pooled_nhwc.transpose(0, 3, 1, 2), oracle.maxpool2d(q8, (2, 2), (2, 2)))
    # channel counts that take the 16-channels-per-thread kernel, with pads and an overlapping window
    for shape, k, st, p in (((3, 32, 9, 11), (3, 3), (2, 2), (1, 1, 1, 1)), ((2, 48, 8, 8), (2, 2), (2, 2), (0, 0, 0, 0)),
                            ((1, 16, 5, 7), (3, 2), (1, 2), (1, 0, 0, 1))):
        q = r.integers(-128, 128, shape).astype(np.int8)
        got = ops.maxpool2d(np.ascontiguousarray(q.transpose(0, 2, 3, 1)), k, st, p, layout=L.LAYOUT_NHWC)
        assert np.array_equal(got.transpose(0, 3, 1, 2), oracle.maxpool2d(q, k, st, p))


QGEMM_SHAPES = [
    # M, N, K, transB
    (64, 64, 64, True), (64, 64, 64, False),
    (100, 72, 48, True), (100, 72, 48, False),          # ragged tiles, 128-tile kernel
    (300, 520, 272, True), (300, 520, 272, False),
    (512, 2048, 512, True), (512, 2048, 512, False),    # 128 x 128 tiles (the 256 x 256 kernel starts at M * N >= 2^23:
    (777, 1028, 1040, True), (777, 1028, 1040, False),  # test_qgemm_s8_large_b_as_k_by_n covers it), ragged
    (33, 47, 50, True), (33, 47, 50, False),            # K % 16 != 0: simple kernel
    (4096, 5, 256, True), (1, 16, 16, True),             # at most 16 columns: the dot-product kernel
    (70, 13, 1040, True), (5, 1, 32, True), (300, 9, 48, True),
    (512, 256, 12800, True),                             # long K, few tiles: K cut into slices
    (300, 130, 8464, True), (129, 40, 8208, True),       # ... with ragged tiles and a last slice that is shorter
    (1, 1024, 1024, True), (8, 4096, 2048, True),        # a small batch on a layer of some size: a pass over B [N,K] with K
    (16, 1000, 1040, True), (17, 66, 4096, True),        # in slices (k_qgemm_few_rows): ragged columns, K no multiple of a
    (32, 2050, 528, True), (31, 640, 8208, True),        # chunk of 64 or of a slice, one and two row tiles
    (13, 2060, 1104, True), (16, 4096, 4112, True),      # ... at most 16 rows and 2048 columns or more: one launch, K cut inside
]                                                        # the workgroups (k_qgemm_few_rows_whole): ragged columns, a last wavefront
                                                         # with a short share of K, more than eight chunks per wavefront


@pytest.mark.parametrize("M,N,K,transB", QGEMM_SHAPES)
def test_qgemm_s8_accumulators_and_requant(ops, M, N, K, transB):
    from sofie_amd import lib as L
    r = rng(300 + M + N + K)
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (N, K) if transB else (K, N)).astype(np.int8)
    acc = ops.igemm_s8(A, B, transB)
    ref = oracle.igemm_s8(A, B, transB)
    assert np.array_equal(acc, ref)
    sigma = 73.3 * 73.3 * np.sqrt(K)
    scale = r.uniform(20.0, 60.0, N).astype(np.float32) / np.float32(sigma)   # spread: few saturate
    bias = r.integers(-2000, 2000, N).astype(np.int32)
    for zpy, relu in [(0, False), (-128, True), (5, True)]:
        y = ops.qgemm_s8(A, B, scale, bias, transB, zpy=zpy, relu=relu)
        assert np.array_equal(y, oracle.qgemm_s8(A, B, scale, bias, transB, zpy=zpy, relu=relu))
    yf = ops.qgemm_s8(A, B, scale, bias, transB, relu=True, out=L.OUT_F32)
    assert np.array_equal(yf, oracle.qgemm_s8_f32out(A, B, scale, bias, transB, relu=True))
    # activation zero-point folded into the bias on the host
    yz = ops.qgemm_s8(A, B, scale, bias, transB, zpa=-128, zpy=-3)
    acc_z = (A.astype(np.int64) + 128) @ (B.T if transB else B).astype(np.int64) + bias
    want = np.empty((M, N), np.int8)
    flat = want.reshape(-1)
    az = acc_z.reshape(-1)
    sc = np.tile(scale, M)
    if M * N <= 40000:
        for i in range(flat.size):
            flat[i] = oracle.requant_one(int(az[i]), sc[i], -3, False)
        assert np.array_equal(yz, want)


def test_qgemm_s8_few_rows_kernels_and_constant_weights(ops):
    """Which kernels a quantised layer on a small batch runs on: B [N,K] takes the pass over B with K in slices; B [K,N]
    is transposed into the scratch buffer first and then runs on tiles, and with the constant-weights promise the
    transposed copy is made once and the small batch takes the pass over it. Bit-exact against the oracle each time."""
    r = rng(612)
    M, N, K = 8, 1536, 2048
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    Bnk = r.integers(-127, 128, (N, K)).astype(np.int8)
    Bkn = np.ascontiguousarray(Bnk.T)
    scale = (r.uniform(20.0, 60.0, N) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-2000, 2000, N).astype(np.int32)
    ref = oracle.qgemm_s8(A, Bnk, scale, bias, True, zpy=-128, relu=True)
    y, names = _kernels_of(ops, lambda: ops.qgemm_s8(A, Bnk, scale, bias, True, zpy=-128, relu=True))
    assert names == ["k_qgemm_few_rows", "k_splitk_finish"], names
    assert np.array_equal(y, ref)
    # 2048 columns or more and at most 16 rows: one launch, no partial sums in memory
    wide = r.integers(-127, 128, (4096, 1024)).astype(np.int8)
    ws = (r.uniform(20.0, 60.0, 4096) / (73.3 * 73.3 * 32)).astype(np.float32)
    yw, names = _kernels_of(ops, lambda: ops.qgemm_s8(A[:, :1024], wide, ws, None, True, zpy=3))
    assert names == ["k_qgemm_few_rows_whole"], names
    assert np.array_equal(yw, oracle.qgemm_s8(A[:, :1024], wide, ws, None, True, zpy=3))
    y, names = _kernels_of(ops, lambda: ops.qgemm_s8(A, Bkn, scale, bias, False, zpy=-128, relu=True))
    assert names == ["k_transpose_bytes", "k_gemm_bytes"], names
    assert np.array_equal(y, ref)
    ctx = ops.Context(0)
    try:
        assert ctx.lib.sofie_hip_constant_weights(ctx.h, 1) == 0
        a, b = ctx.dev(A, torch.int8), ctx.dev(Bkn, torch.int8)
        sd, bd = ctx.dev(scale, torch.float32), ctx.dev(bias, torch.int32)
        out = ctx.empty((M, N), torch.int8)
        from sofie_amd import lib as L
        import ctypes as C
        seen = []
        for _ in range(2):
            buf = C.create_string_buffer(4096)
            n = C.c_int(-1)
            assert ctx.lib.sofie_hip_trace_begin(ctx.h) == 0
            ctx.check(ctx.lib.sofie_hip_qgemm_s8(ctx.h, 0, M, N, K, ctx.ptr(a), K, ctx.ptr(b), N, ctx.ptr(sd), ctx.ptr(bd), -128,
                                                 L.ACT_RELU, ctx.ptr(out), N, L.OUT_S8))
            assert ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)) == 0
            seen.append([l.split()[0] for l in buf.value.decode().splitlines()])
            ctx.sync()
            assert np.array_equal(out.cpu().numpy(), ref)
        assert seen == [["k_transpose_bytes", "k_qgemm_few_rows", "k_splitk_finish"], ["k_qgemm_few_rows", "k_splitk_finish"]], seen
    finally:
        ctx.close()


def test_qgemm_s8_baseline_scales_saturate_identically(ops):
    """The benchmark's own scale range [1e-3, 1e-2] saturates most outputs; still bit-exact."""
    r = rng(12)
    M, N, K = 256, 512, 4096
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (K, N)).astype(np.int8)
    scale = r.uniform(1e-3, 1e-2, N).astype(np.float32)
    y = ops.qgemm_s8(A, B, scale)
    assert np.array_equal(y, oracle.qgemm_s8(A, B, scale))


def test_qgemm_s8_full_size_properties(ops):
    """M=N=K=4096: rows checked against the oracle, plus exact linearity of the accumulators."""
    r = rng(13)
    n = 4096
    A = r.integers(-127, 128, (n, n)).astype(np.int8)
    B = r.integers(-127, 128, (n, n)).astype(np.int8)
    scale = r.uniform(1e-3, 1e-2, n).astype(np.float32)
    spread = (r.uniform(20, 60, n) / (73.3 * 73.3 * 64)).astype(np.float32)
    At, Bt = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    y = ops.qgemm_s8(At, Bt, torch.from_numpy(scale).cuda()).cpu().numpy()
    ys = ops.qgemm_s8(At, Bt, torch.from_numpy(spread).cuda()).cpu().numpy()
    acc = ops.igemm_s8(At, Bt).cpu().numpy()
    rows = np.concatenate([np.arange(0, 24), r.integers(0, n, 24), np.arange(n - 16, n)])
    ref_acc = oracle.igemm_s8(A[rows], B)
    assert np.array_equal(acc[rows], ref_acc)
    assert np.array_equal(y[rows], oracle.qgemm_s8(A[rows], B, scale))
    assert np.array_equal(ys[rows], oracle.qgemm_s8(A[rows], B, spread))
    # checksum of checksums: sum over all accumulators equals (column sums of A) . (row sums of B)
    total = int(acc.astype(np.int64).sum())
    assert total == int(A.astype(np.int64).sum(axis=0) @ B.astype(np.int64).sum(axis=1))
    # transposed-B entry point gives the same matrix
    acc_t = ops.igemm_s8(At, Bt.t().contiguous(), True).cpu().numpy()
    assert np.array_equal(acc_t, acc)


@pytest.mark.parametrize("M,N,K", [(2100, 4112, 1040), (4096, 2048, 128), (2304, 4096, 16)])
def test_qgemm_s8_large_b_as_k_by_n(ops, M, N, K):
    """B [K,N] on the large-tile kernel (operand transposed by the LDS read): ragged M and N tiles,
    a K tail, a single K step; sampled rows against the oracle and the transposed-B entry point."""
    from sofie_amd import lib as L
    r = rng(77 + M + N + K)
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (K, N)).astype(np.int8)
    scale = (r.uniform(20.0, 60.0, N) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-2000, 2000, N).astype(np.int32)
    At, Bt = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    acc = ops.igemm_s8(At, Bt).cpu().numpy()
    rows = np.concatenate([np.arange(0, 40), r.integers(0, M, 40), np.arange(M - 40, M)])
    assert np.array_equal(acc[rows], oracle.igemm_s8(A[rows], B))
    assert np.array_equal(acc, ops.igemm_s8(At, Bt.t().contiguous(), True).cpu().numpy())
    y = ops.qgemm_s8(At, Bt, torch.from_numpy(scale).cuda(), torch.from_numpy(bias).cuda(), zpy=3, relu=True).cpu().numpy()
    assert np.array_equal(y[rows], oracle.qgemm_s8(A[rows], B, scale, bias, zpy=3, relu=True))


def test_qgemm_rounding_ties_and_saturation(ops):
    """Scale 0.5 (and 0.25, 1.5) makes every odd accumulator an exact tie; the byte-packing epilogues must round
    them half to even like the oracle, for the zero-point -128 path (conversion instruction does the rounding)
    and for a general zero-point, and saturate at both ends."""
    M, N, K = 256, 256, 64
    A = np.zeros((M, K), np.int8)
    A[:, 0] = (np.arange(M) - 128).clip(-128, 127)
    A[:, 1] = 1
    B = np.zeros((K, N), np.int8)
    B[0, :] = 1
    B[1, :] = (np.arange(N) % 7) - 3                 # acc[m,n] = (m - 128) + (n % 7 - 3)
    B[2:, :] = 5                                      # multiplied by zeros of A
    for sval in (0.5, 0.25, 1.5, 2.5):
        scale = np.full(N, sval, np.float32)
        bias = (np.arange(N) % 3).astype(np.int32)
        for zpy, relu in ((-128, False), (-128, True), (3, False), (-5, True)):
            ref = oracle.qgemm_s8(A, B, scale, bias, False, zpy=zpy, relu=relu)
            assert np.array_equal(ops.qgemm_s8(A, B, scale, bias, zpy=zpy, relu=relu), ref), (sval, zpy, relu)
            Bt = np.ascontiguousarray(B.T)
            assert np.array_equal(ops.qgemm_s8(A, Bt, scale, bias, transB=True, zpy=zpy, relu=relu), ref)
    # the accumulators really contain ties
    acc = oracle.igemm_s8(A, B)
    assert np.any((acc % 2) != 0)


@pytest.mark.parametrize("cfg", [
    dict(N=2, C=6, H=7, W=6, OC=8, k=(3, 3), p=(1, 1), s=(1, 1), g=2),
    dict(N=1, C=1, H=40, W=40, OC=32, k=(3, 3), p=(1, 1), s=(1, 1), g=1),
    dict(N=2, C=32, H=20, W=20, OC=64, k=(3, 3), p=(1, 1), s=(1, 1), g=1),
    dict(N=2, C=64, H=10, W=10, OC=128, k=(3, 3), p=(1, 1), s=(1, 1), g=1),
    dict(N=1, C=16, H=9, W=11, OC=24, k=(1, 1), p=(0, 0), s=(2, 2), g=1),
    dict(N=1, C=64, H=56, W=56, OC=128, k=(3, 3), p=(1, 1), s=(1, 1), g=1),
    dict(N=2, C=6, H=7, W=6, OC=8, k=(4, 2), p=(1, 0, 2, 1), s=(1, 1), g=2),      # begin != end pads, plain kernel
    dict(N=1, C=1, H=40, W=40, OC=32, k=(3, 3), p=(1, 1, 0, 1), s=(1, 1), g=1),   # not the first-layer kernel's shape
])
def test_qconv2d_s8(ops, cfg):
    from sofie_amd import lib as L
    r = rng(400 + cfg["C"] + cfg["OC"])
    x = r.integers(-128, 128, (cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.int8)
    w = r.integers(-127, 128, (cfg["OC"], cfg["C"] // cfg["g"]) + cfg["k"]).astype(np.int8)
    K = cfg["C"] // cfg["g"] * cfg["k"][0] * cfg["k"][1]
    scale = (r.uniform(20, 60, cfg["OC"]) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-3000, 3000, cfg["OC"]).astype(np.int32)
    zpx = -128
    ref_acc = oracle.iconv2d_s8(x, w, cfg["p"], cfg["s"], cfg["g"], zpx)
    acc = ops.iconv2d_s8(x, w, cfg["p"], cfg["s"], cfg["g"], zpx)
    assert np.array_equal(acc, ref_acc)
    ref = oracle.qconv2d_s8(x, w, scale, bias, cfg["p"], cfg["s"], cfg["g"], zpx, -128, True)
    y = ops.qconv2d_s8(x, w, scale, bias, cfg["p"], cfg["s"], cfg["g"], zpx, -128, True)
    assert np.array_equal(y, ref)
    xh = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    yh = ops.qconv2d_s8(xh, w, scale, bias, cfg["p"], cfg["s"], cfg["g"], zpx, -128, True,
                        x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(yh.transpose(0, 3, 1, 2), ref)
    y0 = ops.qconv2d_s8(x, w, scale, None, cfg["p"], cfg["s"], cfg["g"], 0, 7, False)
    assert np.array_equal(y0, oracle.qconv2d_s8(x, w, scale, None, cfg["p"], cfg["s"], cfg["g"], 0, 7, False))


@pytest.mark.parametrize("cfg", [
    # the matrix-core kernel's shapes: bands that cross image boundaries, a partial last tile, strides,
    # 1x1 / 5x5 / non-square kernels, no padding, wide padding, one image smaller than a tile
    dict(N=3, C=32, H=20, W=20, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=7, C=64, H=10, W=10, OC=128, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=2, C=64, H=56, W=56, OC=128, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=5, C=32, H=9, W=13, OC=64, k=(3, 3), p=(0, 0), s=(1, 1)),
    dict(N=4, C=64, H=15, W=17, OC=192, k=(3, 3), p=(1, 1), s=(2, 2)),
    dict(N=9, C=96, H=6, W=5, OC=64, k=(1, 1), p=(0, 0), s=(1, 1)),
    dict(N=2, C=32, H=12, W=12, OC=128, k=(5, 5), p=(2, 2), s=(1, 1)),
    dict(N=3, C=32, H=11, W=8, OC=64, k=(3, 1), p=(1, 0), s=(2, 1)),
    dict(N=1, C=32, H=4, W=4, OC=64, k=(3, 3), p=(2, 2), s=(1, 1)),
    dict(N=300, C=32, H=3, W=3, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
    # begin != end pads (top, left, bottom, right): bands of H + top + bottom rows, windows placed by the begin pads
    dict(N=5, C=32, H=12, W=12, OC=64, k=(4, 4), p=(1, 1, 2, 2), s=(1, 1)),
    dict(N=5, C=32, H=12, W=12, OC=64, k=(4, 4), p=(2, 2, 1, 1), s=(1, 1)),
    dict(N=3, C=64, H=16, W=14, OC=128, k=(3, 3), p=(0, 0, 1, 1), s=(2, 2)),
    dict(N=4, C=32, H=9, W=10, OC=64, k=(3, 3), p=(2, 0, 0, 1), s=(1, 1)),
    # 3x3 stride 1 on 32 / 64 channels and rows of 32 to 64 padded columns, fetched straight into LDS: the widest row it takes and
    # one column more (the register-staged kernel), enough pixels for several tiles per workgroup (the window of rows
    # slides through many images), a run of pixels per workgroup that ends inside a tile
    dict(N=2, C=64, H=9, W=62, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=2, C=32, H=9, W=63, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=600, C=32, H=21, W=33, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=11, C=64, H=50, W=47, OC=128, k=(3, 3), p=(0, 1, 1, 0), s=(1, 1)),
])
def test_qconv2d_s8_matrix_core_path(ops, cfg):
    """NHWC activations and [OC,KH,KW,C] weights straight into the MFMA kernel; NCHW operands of the same
    shape reach it through the layout conversion. Both must equal the oracle bit for bit."""
    from sofie_amd import lib as L
    r = rng(500 + cfg["C"] + cfg["OC"] + cfg["H"])
    x = r.integers(-128, 128, (cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.int8)
    w = r.integers(-127, 128, (cfg["OC"], cfg["C"]) + cfg["k"]).astype(np.int8)
    K = cfg["C"] * cfg["k"][0] * cfg["k"][1]
    scale = (r.uniform(20, 60, cfg["OC"]) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-3000, 3000, cfg["OC"]).astype(np.int32)
    xh = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    wh = np.ascontiguousarray(w.transpose(0, 2, 3, 1))
    for zpx, zpy, relu in ((-128, -128, True), (3, 11, False)):
        ref = oracle.qconv2d_s8(x, w, scale, bias, cfg["p"], cfg["s"], 1, zpx, zpy, relu)
        yh = ops.qconv2d_s8(xh, wh, scale, bias, cfg["p"], cfg["s"], 1, zpx, zpy, relu, x_layout=L.LAYOUT_NHWC,
                            y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
        assert np.array_equal(yh.transpose(0, 3, 1, 2), ref)
        y = ops.qconv2d_s8(x, w, scale, bias, cfg["p"], cfg["s"], 1, zpx, zpy, relu)
        assert np.array_equal(y, ref)
    acc = ops.qconv2d_s8(xh, wh, None, None, cfg["p"], cfg["s"], 1, 5, x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC,
                         w_layout=L.LAYOUT_NHWC, out=L.OUT_S32)
    assert np.array_equal(acc.transpose(0, 3, 1, 2), oracle.iconv2d_s8(x, w, cfg["p"], cfg["s"], 1, 5))


@pytest.mark.parametrize("cfg", [
    dict(N=3, H=40, W=40, OC=32), dict(N=6, H=7, W=9, OC=16), dict(N=1, H=1, W=1, OC=32), dict(N=5, H=13, W=6, OC=48),
    dict(N=2, H=64, W=50, OC=64), dict(N=9, H=5, W=4, OC=8),
])
def test_first_layer_kernel(ops, cfg):
    """One input channel, 3x3, pad 1: the K = 16 matrix-instruction kernel (OC a multiple of 16; OC = 8 takes the
    plain kernel), with both zero-point conventions, a ReLU clamp, all-positive scales and scales of both signs
    (the pooled variant then picks max or min of the accumulators by the sign), image counts that do not fill
    the last workgroup."""
    from sofie_amd import lib as L
    r = rng(600 + cfg["H"] + cfg["OC"])
    x = r.integers(-128, 128, (cfg["N"], 1, cfg["H"], cfg["W"])).astype(np.int8)
    w = r.integers(-127, 128, (cfg["OC"], 1, 3, 3)).astype(np.int8)
    scale = (r.uniform(20, 60, cfg["OC"]) / (73.3 * 73.3 * 3)).astype(np.float32)
    bias = r.integers(-3000, 3000, cfg["OC"]).astype(np.int32)
    for zpx, zpy, relu, negate in ((-128, -128, True, False), (5, -3, False, True), (-128, -128, False, True)):
        if negate:
            scale = scale.copy()
            scale[::3] *= -1
        ref = oracle.qconv2d_s8(x, w, scale, bias, (1, 1), (1, 1), 1, zpx, zpy, relu)
        y = ops.qconv2d_s8(x, w, scale, bias, (1, 1), (1, 1), 1, zpx, zpy, relu, y_layout=L.LAYOUT_NHWC)
        assert np.array_equal(y.transpose(0, 3, 1, 2), ref)
        if cfg["H"] >= 2 and cfg["W"] >= 2:
            pooled = oracle.maxpool2d(ref, (2, 2), (2, 2))
            yp = ops.qconv2d_pool_s8(x, w, scale, bias, (1, 1), (1, 1), 1, zpx, zpy, relu, y_layout=L.LAYOUT_NHWC)
            assert np.array_equal(yp.transpose(0, 3, 1, 2), pooled)


@pytest.mark.parametrize("n,c,h,w,oc,pool", [(8, 64, 32, 32, 128, None), (9, 64, 32, 32, 128, None), (4, 32, 28, 28, 128, (2, 2)), (24, 32, 28, 28, 128, (2, 2)),
                                               (3, 64, 9, 13, 256, None), (1, 32, 56, 60, 384, None), (5, 64, 6, 62, 128, (2, 2))])
def test_ring_blocks_of_channels_by_pixels(ops, n, c, h, w, oc, pool):
    """64 output channels per workgroup where pixels are few, 128 beyond, on both sides of the line: the oracle's bytes, scales of both signs."""
    from sofie_amd import lib as L
    r = rng(800 + n + c + oc)
    x = r.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = r.integers(-127, 128, (oc, c, 3, 3)).astype(np.int8)
    scale = (r.uniform(20, 60, oc) / (73.3 * 73.3 * np.sqrt(9 * c))).astype(np.float32)
    scale[::3] *= -1
    bias = r.integers(-3000, 3000, oc).astype(np.int32)
    ref = oracle.qconv2d_s8(x, wt, scale, bias, (1, 1), (1, 1), 1, 5, -3, False)
    if pool:
        ref = oracle.maxpool2d(ref, pool, pool)
    xh, wh = np.ascontiguousarray(x.transpose(0, 2, 3, 1)), np.ascontiguousarray(wt.transpose(0, 2, 3, 1))
    call = ops.qconv2d_pool_s8 if pool else ops.qconv2d_s8
    y = call(xh, wh, scale, bias, (1, 1), (1, 1), 1, 5, -3, False, x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
    assert np.array_equal(y.transpose(0, 3, 1, 2), ref)


@pytest.mark.parametrize("n,h,w,oc", [(1, 180, 160, 16), (100, 40, 40, 32), (128, 9, 12, 16), (129, 9, 12, 16), (300, 16, 16, 64), (85, 23, 31, 48), (1, 2, 3, 16)])
def test_first_layer_images_shared_by_workgroups(ops, n, h, w, oc):
    """Up to half as many images as compute units: workgroups share an image, all of it once, in parts of 128 pixels, one part behind the last whole
    round; beyond, a workgroup to each. From bytes, pooled with scales of both signs, and from floats: the oracle's bytes."""
    from sofie_amd import lib as L
    r = rng(700 + n + h)
    x = r.integers(-128, 128, (n, 1, h, w)).astype(np.int8)
    wt = r.integers(-127, 128, (oc, 1, 3, 3)).astype(np.int8)
    scale = (r.uniform(20, 60, oc) / (73.3 * 73.3 * 3)).astype(np.float32)
    scale[::3] *= -1
    bias = r.integers(-3000, 3000, oc).astype(np.int32)
    ref = oracle.qconv2d_s8(x, wt, scale, bias, (1, 1), (1, 1), 1, 5, -3, False)
    y = ops.qconv2d_s8(x, wt, scale, bias, (1, 1), (1, 1), 1, 5, -3, False, y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(y.transpose(0, 3, 1, 2), ref)
    yp = ops.qconv2d_pool_s8(x, wt, scale, bias, (1, 1), (1, 1), 1, 5, -3, False, y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(yp.transpose(0, 3, 1, 2), oracle.maxpool2d(ref, (2, 2), (2, 2)))
    xf = (x.astype(np.float32) - 5.0) * np.float32(0.125)
    yf = ops.quantize_qconv2d_s8(xf, np.float32(0.125), 5, wt, scale, bias, (1, 1), (1, 1), 1, -3, False, None, (2, 2), y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(yf.transpose(0, 3, 1, 2), ref)


@pytest.mark.parametrize("cfg", [
    dict(N=5, C=1, H=40, W=40, OC=32, k=(3, 3), p=(1, 1), pool=(2, 2)),    # first-layer kernel, dword fill
    dict(N=3, C=1, H=9, W=7, OC=16, k=(3, 3), p=(1, 1), pool=None),        # first-layer kernel, byte fill
    dict(N=2, C=1, H=12, W=12, OC=8, k=(3, 3), p=(1, 1), pool=(2, 2)),     # plain kernels through scratch memory
    dict(N=2, C=32, H=8, W=8, OC=64, k=(3, 3), p=(1, 1), pool=None),       # multi-channel float input, MFMA conv
])
def test_quantize_conv_fused_entry_point(ops, cfg):
    """QuantizeLinear -> QLinearConv -> ReLU -> (MaxPool) from a float tensor equals the separate oracle steps,
    including values that saturate and exact .5 ties of x / scale."""
    from sofie_amd import lib as L
    r = rng(900 + cfg["H"] + cfg["OC"])
    shape = (cfg["N"], cfg["C"], cfg["H"], cfg["W"])
    x = r.uniform(-0.2, 1.2, shape).astype(np.float32)
    x.reshape(-1)[::7] = (r.integers(-10, 300, x.reshape(-1)[::7].size) + 0.5) / 255.0
    sx, zpx = np.float32(1 / 255.0), -128
    w = r.integers(-127, 128, (cfg["OC"], cfg["C"]) + cfg["k"]).astype(np.int8)
    K = cfg["C"] * 9
    scale = (r.uniform(20, 60, cfg["OC"]) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-3000, 3000, cfg["OC"]).astype(np.int32)
    xq = oracle.quantize_f32_s8(x, sx, zpx)
    ref = oracle.qconv2d_s8(xq, w, scale, bias, cfg["p"], (1, 1), 1, zpx, -128, True)
    if cfg["pool"]:
        ref = oracle.maxpool2d(ref, cfg["pool"], (2, 2))
    y = ops.quantize_qconv2d_s8(x, sx, zpx, w, scale, bias, cfg["p"], (1, 1), 1, -128, True, cfg["pool"], (2, 2),
                                y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(y.transpose(0, 3, 1, 2), ref)


@pytest.mark.parametrize("sx_bits,zpx", [(0x3c7fffff, -128), (0x3d17f4a8, 7), (0x2b000001, -128), (0x3b808081, 0),
                                          (0x3c000000, -20)])
def test_quantize_conv_fused_division_is_exact(ops, sx_bits, zpx):
    """The first-layer kernel divides by the activation scale with a reciprocal and two fused corrections; the
    result must equal the true float division for any scale (all-ones mantissa, a power of two, outside the range of
    the short sequence), for exact ties, and for values far outside the int8 range."""
    from sofie_amd import lib as L
    r = rng(950 + zpx)
    sx = np.array([sx_bits], np.uint32).view(np.float32)[0]
    N, H, W, OC = 6, 16, 24, 32
    x = (r.uniform(-140, 140, (N, 1, H, W)) * float(sx)).astype(np.float32)
    flat = x.reshape(-1)
    ties = ((r.integers(-200, 200, flat[::5].size) + 0.5) * float(sx)).astype(np.float32)
    flat[::5] = ties
    flat[1::5] = np.nextafter(ties, np.float32(0))[: flat[1::5].size]
    flat[2::97] = np.float32(1e30)
    flat[3::97] = np.float32(-1e30)
    flat[4::97] = np.float32(1e-30)
    w = r.integers(-127, 128, (OC, 1, 3, 3)).astype(np.int8)
    scale = (r.uniform(20, 60, OC) / (73.3 * 73.3 * 3)).astype(np.float32)
    bias = r.integers(-3000, 3000, OC).astype(np.int32)
    xq = oracle.quantize_f32_s8(x, sx, zpx)
    ref = oracle.maxpool2d(oracle.qconv2d_s8(xq, w, scale, bias, (1, 1), (1, 1), 1, zpx, -128, True), (2, 2), (2, 2))
    y = ops.quantize_qconv2d_s8(x, sx, zpx, w, scale, bias, (1, 1), (1, 1), 1, -128, True, (2, 2), (2, 2),
                                y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(y.transpose(0, 3, 1, 2), ref)
    # and the quantizer on its own agrees with the oracle on the same input
    assert np.array_equal(ops.quantize_f32_s8(x, sx, zpx), xq)


@pytest.mark.parametrize("cfg", [
    dict(N=2, C=32, H=20, W=20, OC=64, k=(3, 3), p=(1, 1), pool=(2, 2), ps=(2, 2)),
    dict(N=2, C=6, H=9, W=8, OC=10, k=(3, 3), p=(0, 0), pool=(3, 2), ps=(2, 1)),
    dict(N=1, C=64, H=11, W=11, OC=128, k=(3, 3), p=(1, 1), pool=(2, 2), ps=(2, 2)),
])
def test_conv_pool_entry_point(ops, cfg):
    """The fused entry point on shapes without a fused kernel: convolution into scratch memory, then pooling,
    in both layouts."""
    from sofie_amd import lib as L
    r = rng(700 + cfg["C"])
    x = r.integers(-128, 128, (cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.int8)
    w = r.integers(-127, 128, (cfg["OC"], cfg["C"]) + cfg["k"]).astype(np.int8)
    K = cfg["C"] * cfg["k"][0] * cfg["k"][1]
    scale = (r.uniform(20, 60, cfg["OC"]) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    bias = r.integers(-3000, 3000, cfg["OC"]).astype(np.int32)
    ref = oracle.maxpool2d(oracle.qconv2d_s8(x, w, scale, bias, cfg["p"], (1, 1), 1, -128, -128, True), cfg["pool"], cfg["ps"])
    y = ops.qconv2d_pool_s8(x, w, scale, bias, cfg["p"], (1, 1), 1, -128, -128, True, cfg["pool"], cfg["ps"])
    assert np.array_equal(y, ref)
    xh = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    yh = ops.qconv2d_pool_s8(xh, w, scale, bias, cfg["p"], (1, 1), 1, -128, -128, True, cfg["pool"], cfg["ps"],
                             x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC)
    assert np.array_equal(yh.transpose(0, 3, 1, 2), ref)


@pytest.mark.parametrize("cfg", [
    dict(N=5, C=32, H=20, W=20, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),      # the CNN's second layer
    dict(N=3, C=64, H=11, W=13, OC=128, k=(3, 3), p=(1, 1), s=(1, 1)),     # odd output size: last row / column dropped
    dict(N=70, C=32, H=4, W=6, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),       # many small images per tile
    dict(N=2, C=32, H=17, W=9, OC=192, k=(1, 1), p=(0, 0), s=(1, 1)),
    dict(N=2, C=64, H=21, W=21, OC=64, k=(3, 3), p=(0, 0), s=(2, 2)),      # strided convolution before the pool
    dict(N=1, C=32, H=2, W=2, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),        # a single pooled pixel
    dict(N=4, C=32, H=12, W=10, OC=64, k=(4, 4), p=(1, 1, 2, 2), s=(1, 1)),  # begin != end pads under the pooling
    dict(N=3, C=64, H=9, W=11, OC=128, k=(3, 3), p=(2, 1, 0, 1), s=(1, 1)),
    # rows fetched straight into LDS under the pooling: the widest row, a plane per instruction (4 x 22 slots > 64),
    # and enough images for several tiles per workgroup
    dict(N=2, C=64, H=7, W=62, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=9, C=64, H=20, W=20, OC=128, k=(3, 3), p=(1, 1), s=(1, 1)),
    dict(N=1200, C=32, H=20, W=20, OC=64, k=(3, 3), p=(1, 1), s=(1, 1)),
])
def test_conv_pool_fused_matrix_core_kernel(ops, cfg):
    """Channels-last operands with a 2x2 stride-2 pooling: one kernel whose wavefronts pool on the accumulators.
    Scales of both signs (maximum / minimum of the accumulators), both zero-point conventions."""
    from sofie_amd import lib as L
    r = rng(800 + cfg["C"] + cfg["H"])
    x = r.integers(-128, 128, (cfg["N"], cfg["C"], cfg["H"], cfg["W"])).astype(np.int8)
    w = r.integers(-127, 128, (cfg["OC"], cfg["C"]) + cfg["k"]).astype(np.int8)
    K = cfg["C"] * cfg["k"][0] * cfg["k"][1]
    scale = (r.uniform(20, 60, cfg["OC"]) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    scale[1::5] *= -1
    bias = r.integers(-3000, 3000, cfg["OC"]).astype(np.int32)
    xh = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    wh = np.ascontiguousarray(w.transpose(0, 2, 3, 1))
    for zpx, zpy, relu in ((-128, -128, True), (7, -20, False), (0, 5, True)):
        ref = oracle.maxpool2d(oracle.qconv2d_s8(x, w, scale, bias, cfg["p"], cfg["s"], 1, zpx, zpy, relu), (2, 2), (2, 2))
        y = ops.qconv2d_pool_s8(xh, wh, scale, bias, cfg["p"], cfg["s"], 1, zpx, zpy, relu, x_layout=L.LAYOUT_NHWC,
                                y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
        assert np.array_equal(y.transpose(0, 3, 1, 2), ref), (zpx, zpy, relu)


def _chain_layers(r, shapes, signs=False):
    """Random weights, scales and biases for a chain of 3x3 pad-1 layers; shapes = [(C, OC, pooled), ...]."""
    layers, host = [], []
    for C, OC, pooled in shapes:
        w = r.integers(-127, 128, (OC, C, 3, 3)).astype(np.int8)
        scale = (r.uniform(20, 60, OC) / (73.3 * 73.3 * np.sqrt(9 * C))).astype(np.float32)
        if signs:
            scale[2::7] *= -1
        bias = r.integers(-3000, 3000, OC).astype(np.int32)
        host.append((w, scale, bias, pooled))
        layers.append(dict(w=np.ascontiguousarray(w.transpose(0, 2, 3, 1)), w_layout=1, scale=scale, bias=bias, pads=(1, 1),
                           zpx=-128, zpy=-128, relu=True, pool=(2, 2) if pooled else None, y_layout=1))
    return layers, host


def _chain_reference(x_nchw, host):
    h = x_nchw
    outs = []
    for w, scale, bias, pooled in host:
        h = oracle.qconv2d_s8(h, w, scale, bias, (1, 1), (1, 1), 1, -128, -128, True)
        if pooled:
            h = oracle.maxpool2d(h, (2, 2), (2, 2))
        outs.append(h)
    return outs


@pytest.mark.parametrize("N,H,shapes", [
    (6, 20, [(32, 64, True), (64, 128, False)]),                   # the CNN's second and third layer, layer by layer at this batch
    (3, 12, [(32, 64, False), (64, 64, True), (64, 128, False)]),  # three layers, the pooled one in the middle
    (2, 9, [(16, 24, True)]),                                      # a single layer outside every matrix-core kernel
])
def test_qconv_chain_small(ops, N, H, shapes):
    """sofie_hip_qconv2d_s8_chain on batches where the layers run one after the other: every layer's output equals the
    oracle's, scales of both signs."""
    r = rng(900 + N + H)
    x = r.integers(-128, 128, (N, shapes[0][0], H, H)).astype(np.int8)
    layers, host = _chain_layers(r, shapes, signs=True)
    got = ops.qconv2d_s8_chain(np.ascontiguousarray(x.transpose(0, 2, 3, 1)), layers)
    for y, ref in zip(got, _chain_reference(x, host)):
        assert np.array_equal(y.transpose(0, 3, 1, 2), ref)


def test_qconv_chain_two_layers_in_one_launch(ops):
    """Batch 4096 of 20x20 images, conv 32 -> 64 + ReLU + 2x2 pooling, conv 64 -> 128 + ReLU: every workgroup owns 16
    whole images in both layers, so the chain is one launch in which a workgroup reads back what it wrote. Both outputs
    equal those of the two separate calls byte for byte, and 64 images spread over the batch equal the oracle."""
    from sofie_amd import lib as L
    r = rng(77)
    N = 4096
    x = r.integers(-128, 128, (N, 20, 20, 32)).astype(np.int8)
    layers, host = _chain_layers(r, [(32, 64, True), (64, 128, False)])
    ctx = ops.default_context()
    buf = __import__("ctypes").create_string_buffer(1024)
    n = __import__("ctypes").c_int(0)
    assert ctx.lib.sofie_hip_trace_begin(ctx.h) == 0
    p2, c3 = ops.qconv2d_s8_chain(x, layers)
    assert ctx.lib.sofie_hip_trace_end(ctx.h, buf, 1024, __import__("ctypes").byref(n)) == 0
    assert n.value == 1 and buf.value.decode().split()[0] == "k_qconv_ring_pair"       # one launch for both layers
    a, b = layers
    s2 = ops.qconv2d_pool_s8(x, a["w"], a["scale"], a["bias"], (1, 1), (1, 1), 1, -128, -128, True, x_layout=L.LAYOUT_NHWC,
                             y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
    s3 = ops.qconv2d_s8(s2, b["w"], b["scale"], b["bias"], (1, 1), (1, 1), 1, -128, -128, True, x_layout=L.LAYOUT_NHWC,
                        y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
    assert np.array_equal(p2, s2) and np.array_equal(c3, s3)
    pick = np.arange(0, N, 64) + (np.arange(64) % 16)            # every position inside a workgroup's 16 images
    ref2, ref3 = _chain_reference(np.ascontiguousarray(x[pick].transpose(0, 3, 1, 2)), host)
    assert np.array_equal(p2[pick].transpose(0, 3, 1, 2), ref2)
    assert np.array_equal(c3[pick].transpose(0, 3, 1, 2), ref3)
    # a second call right behind the first (the tensors of the first are rewritten): the same bytes
    p2b, c3b = ops.qconv2d_s8_chain(x, layers)
    assert np.array_equal(p2b, p2) and np.array_equal(c3b, c3)


def test_empty_and_degenerate_inputs(ops):
    """Zero-sized problems return success without touching the output; K = 0 leaves the bias (the accumulators are an
    empty sum); a 1x1 image, a single row and a single column go through the general kernels."""
    from sofie_amd import lib as L
    ctx = ops.default_context()
    lib, h, p = ctx.lib, ctx.h, ctx.ptr
    y = ctx.dev(np.full((4, 4), 7, np.int8))
    A = ctx.dev(np.zeros((4, 16), np.int8))
    sc = ctx.dev(np.ones(4, np.float32))
    # M = 0 and N = 0: nothing is launched, y keeps its bytes; null operands are fine then
    assert lib.sofie_hip_qgemm_s8(h, 1, 0, 4, 16, None, 16, None, 16, None, None, 0, 0, None, 4, L.OUT_S8) == 0
    assert lib.sofie_hip_qgemm_s8(h, 1, 4, 0, 16, p(A), 16, p(A), 16, p(sc), None, 0, 0, p(y), 4, L.OUT_S8) == 0
    assert lib.sofie_hip_gemm_f32(h, 0, 0, 0, 5, 3, 1.0, None, 3, None, 5, 0.0, None, 0, None, 5, 0) == 0
    assert lib.sofie_hip_conv2d_f32(h, None, None, None, None, 0, 3, 5, 5, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0) == 0
    assert lib.sofie_hip_conv_transpose2d_f32(h, None, None, None, None, 0, 3, 5, 5, 4, 3, 3, 0, 0, 1, 1, 1, 1, 1, 7, 7, 0) == 0
    assert lib.sofie_hip_batchnorm_f32(h, None, None, None, None, None, 0, 3, 5, 0) == 0
    assert lib.sofie_hip_relu_f32(h, None, None, 0) == 0
    ctx.sync()
    assert np.all(y.cpu().numpy() == 7)
    # K = 0: int32 output equals the bias row
    bias = np.array([5, -6, 7, 100000], np.int32)
    acc = ctx.empty((3, 4), torch.int32)
    assert lib.sofie_hip_qgemm_s8(h, 1, 3, 4, 0, p(A), 0, p(A), 0, None, p(ctx.dev(bias)), 0, 0, p(acc), 4, L.OUT_S32) == 0
    ctx.sync()
    assert np.array_equal(acc.cpu().numpy(), np.tile(bias, (3, 1)))
    r = rng(99)
    a1 = r.standard_normal((1, 7)).astype(np.float32)
    b1 = r.standard_normal((7, 1)).astype(np.float32)
    assert rel_err(ops.gemm_f32(a1, b1, beta=0.0), oracle.gemm_f32(a1, b1, beta=0.0)) <= FP32_TOL
    x1 = r.standard_normal((1, 1, 1, 1)).astype(np.float32)
    w1 = r.standard_normal((1, 1, 3, 3)).astype(np.float32)
    assert rel_err(ops.conv2d_f32(x1, w1, None, (1, 1)), oracle.conv2d_f32(x1, w1, None, (1, 1))) <= FP32_TOL
    q1 = r.integers(-128, 128, (1, 1, 1, 1)).astype(np.int8)
    wq = r.integers(-127, 128, (1, 1, 1, 1)).astype(np.int8)
    s1 = np.array([0.01], np.float32)
    assert np.array_equal(ops.qconv2d_s8(q1, wq, s1, None, (0, 0)), oracle.qconv2d_s8(q1, wq, s1, None, (0, 0), (1, 1), 1, 0, 0, False))


def test_error_codes_of_the_quantized_entry_points(ops):
    """Bad arguments come back as SOFIE_HIP_EINVAL with a message and launch nothing; the context stays usable."""
    from sofie_amd import lib as L
    ctx = ops.default_context()
    x = ctx.dev(np.zeros((1, 4, 4, 32), np.int8))
    w = ctx.dev(np.zeros((64, 3, 3, 32), np.int8))
    sc = ctx.dev(np.ones(64, np.float32))
    y = ctx.empty((1, 4, 4, 64), torch.int8)
    lib, h, p = ctx.lib, ctx.h, ctx.ptr

    def conv(**kw):
        a = dict(x=p(x), xl=L.LAYOUT_NHWC, w=p(w), wl=L.LAYOUT_NHWC, s=p(sc), y=p(y), groups=1, zpx=0, act=L.ACT_NONE,
                 out=L.OUT_S8, ph=1)
        a.update(kw)
        return lib.sofie_hip_qconv2d_s8(h, a["x"], a["xl"], a["w"], a["wl"], None, a["s"], a["y"], L.LAYOUT_NHWC, 1, 32, 4, 4,
                                        64, 3, 3, a["ph"], 1, 1, 1, 1, 1, a["groups"], a["zpx"], 0, a["act"], a["out"])
    assert conv() == 0
    for bad, text in ((dict(x=None), "null operand"), (dict(groups=3), "groups"), (dict(zpx=300), "zero-point"),
                      (dict(act=7), "activation"), (dict(xl=5), "layout"), (dict(out=L.OUT_BF16), "output kind"),
                      (dict(s=None), "scale is required"), (dict(ph=-1), "pads")):
        assert conv(**bad) == L.EINVAL, bad
        assert text in lib.sofie_hip_last_error(h).decode(), (bad, lib.sofie_hip_last_error(h))
    assert lib.sofie_hip_qconv2d_pool_s8(h, p(x), 1, p(w), 1, None, p(sc), p(y), 1, 1, 32, 4, 4, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 0, 0,
                                         0, 9, 9, 1, 1) == L.EINVAL
    assert "pooling window" in lib.sofie_hip_last_error(h).decode()
    assert lib.sofie_hip_quantize_qconv2d_s8(h, p(ctx.dev(np.zeros((1, 32, 4, 4), np.float32))), -1.0, 0, p(w), 1, None, p(sc),
                                             p(y), 1, 1, 32, 4, 4, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 0) == L.EINVAL
    A = ctx.dev(np.zeros((16, 16), np.int8))
    Y = ctx.empty((16, 16), torch.int8)
    assert lib.sofie_hip_qgemm_s8(h, 1, 16, 16, 16, p(A), 8, p(A), 16, p(ctx.dev(np.ones(16, np.float32))), None, 0, 0, p(Y), 16,
                                  L.OUT_S8) == L.EINVAL
    assert "leading dimension" in lib.sofie_hip_last_error(h).decode()
    assert conv() == 0      # still works
    ctx.sync()


# --------------------------------------------------------------------------- fp8
def fp8_operands(r, M, N, K, transB):
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((N, K) if transB else (K, N)).astype(np.float32)
    sa, sb = np.float32(np.abs(a).max() / 448), np.float32(np.abs(b).max() / 448)
    A = torch.from_numpy(np.clip(a / sa, -448, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    B = torch.from_numpy(np.clip(b / sb, -448, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    return A, B, sa, sb


def test_quantize_e4m3_matches_cast(ops):
    r = rng(14)
    x = np.concatenate([r.standard_normal(6000).astype(np.float32) * 40,
                        r.uniform(-2e-2, 2e-2, 3000).astype(np.float32),
                        np.array([0.0, 448.0, -448.0, 1000.0, -1e9, 464.0, 463.9, 2 ** -10, 2 ** -9 * 1.5,
                                  2 ** -9 * 2.5, 2 ** -7, 0.0146484375], np.float32)])
    q = ops.quantize_f32_e4m3(x, 1.0)
    want = oracle.e4m3_encode(x)
    assert np.array_equal(oracle.e4m3_decode(q), oracle.e4m3_decode(want))


@pytest.mark.parametrize("M,N,K,transB", [
    (64, 64, 64, True), (100, 72, 128, False), (300, 520, 320, True), (512, 1024, 512, False),
    (777, 1028, 1040, True), (33, 47, 50, False)])
def test_gemm_fp8(ops, M, N, K, transB):
    """Tolerance: against the fp64-accumulated product of the same quantised operands,
    |d| <= 2^-8 |ref| (one bf16 rounding) + 7 * 2^-13 * sa*sb*sum_k|a_k b_k|. The second term is
    the accumulation slack of the FP8 matrix instruction, which adds the products of eight consecutive k
    with what lies 2^-14 or more below the largest of them dropped
    (test_fp8_matrix_instruction_sums_groups_of_eight pins that and derives the factor), so the bound is set
    on the magnitude sum, not on the result. On normal operands the error is far inside it: about 2^-17 of
    sum|a_k b_k| as a rule, 2^-14.2 the largest seen in a million outputs."""
    from sofie_amd import lib as L
    r = rng(500 + M + N + K)
    A, B, sa, sb = fp8_operands(r, M, N, K, transB)
    bias = r.standard_normal(N).astype(np.float32)
    yb = ops.gemm_fp8(A, B, sa, sb, bias, transB)
    yf = ops.gemm_fp8(A, B, sa, sb, bias, transB, out=L.OUT_F32)
    _, truth = oracle.gemm_fp8(A, B, sa, sb, bias, transB, acc64=True)
    da = np.abs(oracle.e4m3_decode(A)).astype(np.float64)
    db = np.abs(oracle.e4m3_decode(B)).astype(np.float64)
    mag = (da @ (db.T if transB else db)) * float(sa) * float(sb)
    slack = FP8_SUM_SLACK * mag + 1e-30
    assert np.all(np.abs(yf.astype(np.float64) - truth) <= slack + 2.0 ** -22 * np.abs(truth))
    got = oracle.bf16_decode(yb).astype(np.float64)
    assert np.all(np.abs(got - truth) <= 2.0 ** -8 * np.abs(truth) + slack)
    # the bf16 output is exactly the RNE rounding of the fp32 output of the same kernel
    assert np.array_equal(yb, oracle.bf16_encode(yf))


def test_fp8_matrix_instruction_sums_groups_of_eight(ops):
    """Where the FP8 tolerance comes from. v_mfma_scale_f32_32x32x64_f8f6f4 adds the 64 products of a block in groups
    of eight consecutive k: inside a group the products are aligned to the largest one and what lies 2^-14 or more
    below it is cut off (toward zero); the groups' sums are then added exactly as far as fp32 holds them. A product
    vanishes when it shares its group with one 2^14 times its size and survives anywhere else, so the error of a dot
    product is below 7 * 2^-13 * (sum over the groups of the group's largest |a_k b_k|) <= 7 * 2^-13 * sum|a_k b_k|:
    FP8_SUM_SLACK. Pinned on constructed operands (all values exact in e4m3, scales 1, fp32 output)."""
    from sofie_amd import lib as L
    K = 64

    def product(a, b):
        A, B = oracle.e4m3_encode(a), oracle.e4m3_encode(b)
        assert np.array_equal(oracle.e4m3_decode(A), a) and np.array_equal(oracle.e4m3_decode(B), b)
        return ops.gemm_fp8(A, B, np.float32(1), np.float32(1), None, False, out=L.OUT_F32)[:, 0].astype(np.float64)

    # one product 2^(16 - e) beside 2^16 at k = 0: in the same group of eight (k = 1) it survives down to 2^-13 of the
    # large one and is gone from 2^-14 on; in another group (k = 8) it survives as long as fp32 can hold the sum
    es = list(range(8, 24))
    for k_small in (1, 8):
        a = np.zeros((len(es), K), np.float32)
        b = np.zeros((K, 4), np.float32)
        b[0], b[k_small] = 256.0, 1.0
        a[:, 0] = 256.0
        a[:, k_small] = [2.0 ** (16 - e) for e in es]
        y = product(a, b)
        want = [65536.0 + (2.0 ** (16 - e) if (k_small == 8 or e <= 13) else 0.0) for e in es]
        assert np.array_equal(y, np.array(want)), (k_small, y - 65536.0)
    # which k share the fate: a product of 1.75 beside 65536 at k = 37 is lost at k = 32..39 and nowhere else
    a = np.zeros((K, K), np.float32)
    b = np.full((K, 4), 1.75 * 2.0 ** -6, np.float32)
    b[37] = 256.0
    for k in range(K):
        if k != 37:
            a[k, 37], a[k, k] = 256.0, 64.0
    y = product(a, b)
    assert [k for k in range(K) if k != 37 and y[k] == 65536.0] == [32, 33, 34, 35, 36, 38, 39]
    assert all(y[k] == 65537.75 for k in range(K) if k != 37 and not 32 <= k <= 39)
    # the bound is nearly reached: 63 products of 1.75 * 2^-14 of the large one lose the seven of its group, whole
    a = np.zeros((1, K), np.float32)
    b = np.zeros((K, 4), np.float32)
    a[0, 0], b[0] = 256.0, 256.0
    a[0, 1:], b[1:] = 2.0 ** 8, 1.75 * 2.0 ** -6
    y = product(a, b)[0]
    exact, mag = 65536.0 + 63 * 7.0, 65536.0 + 63 * 7.0
    assert y == 65536.0 + 56 * 7.0
    assert 0.8 * FP8_SUM_SLACK * mag <= exact - y <= FP8_SUM_SLACK * mag
    # signs: the cut is toward zero
    a[0, 1:] = -2.0 ** 8
    assert product(a, b)[0] == 65536.0 - 56 * 7.0


def test_gemm_fp8_large_b_as_k_by_n(ops):
    """B [K,N] on the large-tile FP8 kernel: small integers make every sum exact, so the result must
    equal the integer product, ragged tiles and K tail included."""
    from sofie_amd import lib as L
    r = rng(16)
    M, N, K = 2100, 4112, 1040
    a = r.integers(-4, 5, (M, K)).astype(np.float32)
    b = r.integers(-4, 5, (K, N)).astype(np.float32)
    A, B = oracle.e4m3_encode(a), oracle.e4m3_encode(b)
    y = ops.gemm_fp8(A, B, 1.0, 1.0, None, False, out=L.OUT_F32)
    assert np.array_equal(y, a @ b)


def test_gemm_fp8_exact_for_small_integers(ops):
    """Operands that are small integers in e4m3 make every partial sum exact in fp32."""
    from sofie_amd import lib as L
    r = rng(15)
    M, N, K = 256, 384, 512
    a = r.integers(-4, 5, (M, K)).astype(np.float32)
    b = r.integers(-4, 5, (K, N)).astype(np.float32)
    A, B = oracle.e4m3_encode(a), oracle.e4m3_encode(b)
    y = ops.gemm_fp8(A, B, 1.0, 1.0, None, False, out=L.OUT_F32)
    assert np.array_equal(y, a @ b)


# --------------------------------------------------------------------------- Einsum
EINSUM_GENERAL = [
    ("ik,kj->ji", [(40, 50), (50, 60)]), ("abc,abd->ad", [(7, 9, 33), (7, 9, 65)]), ("i,i->", [(1000,), (1000,)]),
    ("ii->i", [(37, 37)]), ("ij->ji", [(130, 70)]), ("i,j->ij", [(300,), (129,)]), ("ab,bc,cd->ad", [(13, 14), (14, 15), (15, 12)]),
    ("zy,y->z", [(500, 80), (80,)]), ("ijk->", [(5, 6, 7)]), ("abcd,efcd,ae,bf->ab", [(3, 4, 5, 6), (2, 3, 5, 6), (3, 2), (4, 3)]),
]
EINSUM_PRODUCTS = [
    ("ik,kj->ij", [(70, 130), (130, 90)]), ("ki,kj->ij", [(50, 64), (50, 33)]), ("bik,bjk->bij", [(3, 40, 50), (3, 60, 50)]),
    ("ki,jk->ij", [(48, 20), (36, 48)]), ("abik,bkj->abij", [(2, 3, 17, 20), (3, 20, 9)]),
]


@pytest.mark.parametrize("eq,shapes", EINSUM_GENERAL)
def test_einsum_general_kernel_is_the_reference_loop_nest(ops, eq, shapes):
    """Equations that are not matrix products: the kernel sums in the order of the reference's emitted loops with
    separately rounded products and sums, so the result is the oracle's bit for bit."""
    r = rng(sum(map(ord, eq)))
    xs = [r.standard_normal(s).astype(np.float32) for s in shapes]
    y = ops.einsum_f32(eq, xs)
    ref = oracle.einsum_f32(eq, xs)
    assert y.shape == ref.shape
    assert np.array_equal(y, ref)


@pytest.mark.parametrize("eq,shapes", EINSUM_PRODUCTS)
def test_einsum_matrix_products_through_the_gemm_kernel(ops, eq, shapes):
    """(Stacked) matrix products run on the Gemm kernel, whose sums associate differently: 1e-5 relative, and exact on
    small integers."""
    r = rng(sum(map(ord, eq)))
    xs = [r.standard_normal(s).astype(np.float32) for s in shapes]
    y = ops.einsum_f32(eq, xs)
    ref = oracle.einsum_f32(eq, xs)
    assert y.shape == ref.shape
    assert rel_err(y, ref) <= FP32_TOL
    xi = [r.integers(-4, 5, s).astype(np.float32) for s in shapes]
    assert np.array_equal(ops.einsum_f32(eq, xi), oracle.einsum_f32(eq, xi))


# --------------------------------------------------------------------------- 3-D convolution
@pytest.mark.parametrize("cfg", [
    # N, C, D, H, W, OC, k, pads, strides, dilations, groups
    (2, 3, 5, 6, 7, 4, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1),
    (1, 4, 8, 9, 33, 6, (2, 3, 1), (0, 1, 0), (2, 1, 3), (1, 2, 1), 2),
    (3, 8, 4, 4, 70, 8, (1, 1, 5), (0, 0, 2), (1, 1, 1), (1, 1, 3), 8),
    (1, 1, 1, 1, 1, 1, (1, 1, 1), (0, 0, 0), (1, 1, 1), (1, 1, 1), 1),
])
def test_conv3d_f32_matches_the_column_matrix_order(ops, cfg):
    N, C, D, H, W, OC, k, pads, strides, dil, groups = cfg
    r = rng(900 + C + W)
    x = r.standard_normal((N, C, D, H, W)).astype(np.float32)
    w = r.standard_normal((OC, C // groups) + k).astype(np.float32)
    b = r.standard_normal(OC).astype(np.float32)
    for bias, relu in ((b, True), (None, False)):
        y = ops.conv3d_f32(x, w, bias, pads, strides, dil, groups, relu=relu)
        ref = oracle.conv3d_f32(x, w, bias, pads, strides, dil, groups, relu=relu)
        assert y.shape == ref.shape
        assert np.array_equal(y, ref)


# --------------------------------------------------------------------------- the benchmark's full sizes
def _window_sums(xs, k, p, OH, OW):
    """S[n, c, kh, kw] = sum over the output positions of the (zero-padded) input cell that tap (kh, kw) reads."""
    N, C, H, W = xs.shape
    xp = np.zeros((N, C, H + 2 * p, W + 2 * p), np.int64)
    xp[:, :, p:p + H, p:p + W] = xs
    S = np.empty((N, C, k, k), np.int64)
    for kh in range(k):
        for kw in range(k):
            S[:, :, kh, kw] = xp[:, :, kh:kh + OH, kw:kw + OW].sum(axis=(2, 3))
    return S


def test_qconv2d_s8_full_size_layer(ops):
    """The benchmark's layer (batch 256, 64 -> 128 channels, 56x56, 3x3, pad 1, ReLU), int8: three images against
    the oracle bit for bit, every image equal to the same image convolved on its own (the tiles of the batched launch
    cross image borders), and the int32 accumulators of all 102.8 M outputs through one checksum per (image,
    channel): sum over the pixels of acc = sum over the taps of w * (window sum of the input), exact in int64."""
    from sofie_amd import lib as L
    r = rng(77)
    N, C, H, OC = 256, 64, 56, 128
    x = r.integers(-128, 128, (N, H, H, C)).astype(np.int8)                     # channels-last, as between quantized layers
    w = r.integers(-127, 128, (OC, 3, 3, C)).astype(np.int8)
    scale = (r.uniform(20, 60, OC) / (73.3 * 73.3 * np.sqrt(576.0))).astype(np.float32)
    bias = r.integers(-3000, 3000, OC).astype(np.int32)
    y = ops.qconv2d_s8(x, w, scale, bias, (1, 1), (1, 1), 1, -128, -128, True, x_layout=L.LAYOUT_NHWC,
                       y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
    wn = np.ascontiguousarray(w.transpose(0, 3, 1, 2))
    for n in (0, 129, 255):
        xn = np.ascontiguousarray(x[n:n + 1].transpose(0, 3, 1, 2))
        ref = oracle.qconv2d_s8(xn, wn, scale, bias, (1, 1), (1, 1), 1, -128, -128, True)
        assert np.array_equal(y[n].transpose(2, 0, 1), ref[0]), n
    for n in (1, 77, 254):
        alone = ops.qconv2d_s8(x[n:n + 1], w, scale, bias, (1, 1), (1, 1), 1, -128, -128, True, x_layout=L.LAYOUT_NHWC,
                               y_layout=L.LAYOUT_NHWC, w_layout=L.LAYOUT_NHWC)
        assert np.array_equal(alone[0], y[n]), n
    assert 0.05 < np.mean(y == -128) < 0.95 and np.mean(y == 127) < 0.2            # the scales spread the outputs
    acc = ops.qconv2d_s8(x, w, None, None, (1, 1), (1, 1), 1, -128, x_layout=L.LAYOUT_NHWC, y_layout=L.LAYOUT_NHWC,
                         w_layout=L.LAYOUT_NHWC, out=L.OUT_S32)
    got = acc.sum(axis=(1, 2), dtype=np.int64)                                      # [N, OC]
    S = _window_sums(x.transpose(0, 3, 1, 2).astype(np.int64) + 128, 3, 1, H, H)    # x - zp_x, zero outside the image
    want = np.einsum("ockl,nckl->no", wn.astype(np.int64), S)
    assert np.array_equal(got, want)
    # Every int8 output is the requantisation of its accumulator (the int8 launch and the accumulator launch
    # are different kernels). The vectorised formula is tied to the oracle's on a sample first.
    def requant_all(v):
        q = np.rint((v + bias).astype(np.float32) * scale) - 128.0
        return np.clip(q, -128, 127).astype(np.int8)
    sample = acc[17, 23].reshape(-1, OC)[:40]
    for row in sample:
        for c in range(0, OC, 9):
            assert requant_all(row)[c] == oracle.requant_one(int(row[c]) + int(bias[c]), float(scale[c]), -128, True)
    for n0 in range(0, N, 32):
        assert np.array_equal(requant_all(acc[n0:n0 + 32]), y[n0:n0 + 32]), n0


def test_conv2d_f32_full_size_layer(ops):
    """The same layer in fp32 on integer-valued data (every partial sum exact in fp32): two images against the oracle,
    exactly, with bias and ReLU; all outputs of the batch through one checksum per (image, channel)."""
    r = rng(78)
    N, C, H, OC = 256, 64, 56, 128
    x = r.integers(-3, 4, (N, C, H, H)).astype(np.float32)
    w = r.integers(-3, 4, (OC, C, 3, 3)).astype(np.float32)
    b = r.integers(-20, 21, OC).astype(np.float32)
    y = ops.conv2d_f32(x, w, b, (1, 1), (1, 1), (1, 1), 1, True)
    for n in (0, 255):
        ref = oracle.conv2d_f32(x[n:n + 1], w, b, (1, 1), (1, 1), (1, 1), 1, True)
        assert np.array_equal(y[n], ref[0]), n
    del y
    lin = ops.conv2d_f32(x, w, None, (1, 1), (1, 1), (1, 1), 1, False)
    got = lin.sum(axis=(2, 3), dtype=np.float64)
    S = _window_sums(x.astype(np.int64), 3, 1, H, H)
    want = np.einsum("ockl,nckl->no", w.astype(np.int64), S)
    assert np.array_equal(got, want.astype(np.float64))


def test_gemm_fp8_full_size(ops):
    """M = N = 8192, K = 4096 (the benchmark's FP8 GEMM) on small integers in e4m3, which make every sum exact: 256
    rows against the integer product, all 67 M outputs through their row sums and column sums, and the bf16 output
    (with the bias epilogue) equal to the rounding of the fp32 output of the same kernel."""
    from sofie_amd import lib as L
    r = rng(79)
    M, N, K = 8192, 8192, 4096
    a = r.integers(-4, 5, (M, K)).astype(np.float32)
    b = r.integers(-4, 5, (K, N)).astype(np.float32)
    codes = oracle.e4m3_encode(np.arange(-4, 5, dtype=np.float32))              # the nine values' codes, by table
    A, B = codes[a.astype(np.int64) + 4], codes[b.astype(np.int64) + 4]
    y = ops.gemm_fp8(A, B, 1.0, 1.0, None, False, out=L.OUT_F32)
    rows = r.choice(M, 256, replace=False)
    assert np.array_equal(y[rows], a[rows] @ b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.array_equal(y.sum(axis=1, dtype=np.float64), a64 @ b64.sum(axis=1))
    assert np.array_equal(y.sum(axis=0, dtype=np.float64), a64.sum(axis=0) @ b64)
    bias = r.integers(-8, 9, N).astype(np.float32)
    Bt = np.ascontiguousarray(B.T)
    yf = ops.gemm_fp8(A, Bt, 0.5, 0.25, bias, True, out=L.OUT_F32)
    assert np.array_equal(yf, y * np.float32(0.125) + bias)                     # power-of-two scales keep it exact
    yb = ops.gemm_fp8(A, Bt, 0.5, 0.25, bias, True)
    import torch
    assert np.array_equal(yb, torch.from_numpy(yf).bfloat16().view(torch.int16).numpy().view(np.uint16))   # torch rounds RNE
    assert np.array_equal(yb[rows[0]], oracle.bf16_encode(yf[rows[0]]))


@pytest.mark.parametrize("transB", [True, False])
def test_gemm_fp8_more_tiles_than_compute_units(ops, transB):
    """306 tiles of 256 x 256 on 256 compute units, ragged in M and N: the launch in which a workgroup walks over
    several tiles and requests the next tile's operands before it converts the present one. Small integers and
    power-of-two scales make every sum exact, so the bf16 output must be the rounding of the exact result."""
    from sofie_amd import lib as L
    r = rng(81 + int(transB))
    M, N, K = 4100, 4356, 512
    a = r.integers(-4, 5, (M, K)).astype(np.float32)
    b = r.integers(-4, 5, (K, N)).astype(np.float32)
    codes = oracle.e4m3_encode(np.arange(-4, 5, dtype=np.float32))
    A, B = codes[a.astype(np.int64) + 4], codes[b.astype(np.int64) + 4]
    if transB:
        B = np.ascontiguousarray(B.T)
    bias = r.integers(-8, 9, N).astype(np.float32)
    exact = (a @ b) * np.float32(0.125) + bias
    yb = ops.gemm_fp8(A, B, 0.5, 0.25, bias, transB)
    assert np.array_equal(yb, torch.from_numpy(exact).bfloat16().view(torch.int16).numpy().view(np.uint16))
    yn = ops.gemm_fp8(A, B, 0.5, 0.25, None, transB)      # no bias: the tile's parameter block stays zero
    assert np.array_equal(yn, torch.from_numpy((a @ b) * np.float32(0.125)).bfloat16().view(torch.int16).numpy().view(np.uint16))
    yf = ops.gemm_fp8(A, B, 0.5, 0.25, bias, transB, out=L.OUT_F32)
    assert np.array_equal(yf, exact)


@pytest.mark.parametrize("transB", [False, True])
def test_gemm_fp8_benchmark_operands_at_full_depth(ops, transB):
    """The benchmark's own FP8 GEMM (8192 x 8192 x 4096, N(0,1) operands cast to e4m3 at amax/448, bias, bf16 out):
    a band of 512 rows against the fp64-accumulated product of the same e4m3 operands, with the tolerance of
    test_gemm_fp8 (2^-8 |ref| + 7 * 2^-13 sa sb sum|a_k b_k|) at the full K = 4096; the error is printed in bf16 ulps."""
    r = rng(83)
    M = N = 8192
    K = 4096
    A, B, sa, sb = fp8_operands(r, M, N, K, transB)
    bias = r.standard_normal(N).astype(np.float32)
    yb = ops.gemm_fp8(A, B, sa, sb, bias, transB)
    rows = np.sort(r.choice(M, 512, replace=False))
    da = oracle.e4m3_decode(A[rows]).astype(np.float64)
    db = oracle.e4m3_decode(B).astype(np.float64)
    db = db.T if transB else db
    truth = (da @ db) * (float(sa) * float(sb)) + bias.astype(np.float64)
    mag = (np.abs(da) @ np.abs(db)) * (float(sa) * float(sb))
    got = oracle.bf16_decode(yb[rows]).astype(np.float64)
    err = np.abs(got - truth)
    tol = 2.0 ** -8 * np.abs(truth) + FP8_SUM_SLACK * mag + 1e-30
    assert np.all(err <= tol)
    # in bf16 ulps of the true value, over the outputs that are not results of cancellation (|truth| at least a tenth
    # of sum|a_k b_k|'s typical size would be arbitrary: the output's own root mean square is the yardstick)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(truth), 1e-30))) - 7)
    big = np.abs(truth) >= np.sqrt(np.mean(truth ** 2))
    print("fp8 gemm K=4096 %s: bf16 ulp of the error max %.3f mean %.3f over the %d outputs of at least rms size; "
          "largest error / tolerance %.3f" % ("[N,K]" if transB else "[K,N]", (err / ulp)[big].max(), (err / ulp)[big].mean(),
                                              int(big.sum()), (err / tol).max()))


def test_trace_times_every_launch(ops):
    """sofie_hip_trace_begin / _end: one line per launch between the two calls, in launch order, with the name of the
    kernel and a positive time; opening a second trace, ending one that is not open, or recording a graph while a trace is
    open is refused."""
    import ctypes as C
    from sofie_amd import lib as L
    ctx = ops.default_context()
    lib = ctx.lib
    x = ctx.dev(rng(5).standard_normal(1 << 16).astype(np.float32))
    y = ctx.empty((1 << 16,), torch.float32)
    a = ctx.dev(rng(6).integers(-127, 128, (64, 64)).astype(np.int8))
    s1 = ctx.dev(np.full(64, 1e-3, np.float32))
    yq = ctx.empty((64, 64), torch.int8)
    buf = C.create_string_buffer(4096)
    n = C.c_int(-1)
    assert lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)) == L.EINVAL
    assert lib.sofie_hip_trace_begin(ctx.h) == 0
    assert lib.sofie_hip_trace_begin(ctx.h) == L.EINVAL
    assert lib.sofie_hip_capture_begin(ctx.h) == L.EINVAL
    for _ in range(3):
        ctx.check(lib.sofie_hip_relu_f32(ctx.h, ctx.ptr(x), ctx.ptr(y), x.numel()))
    ctx.check(lib.sofie_hip_qgemm_s8(ctx.h, 1, 64, 64, 64, ctx.ptr(a), 64, ctx.ptr(a), 64, ctx.ptr(s1), None, 0, 0, ctx.ptr(yq), 64, L.OUT_S8))
    assert lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)) == 0
    lines = buf.value.decode().splitlines()
    assert n.value == 4 and len(lines) == 4
    assert [l.split()[0] for l in lines[:3]] == ["k_relu_f32"] * 3 and lines[3].split()[0].startswith("k_")
    assert all(float(l.split()[1]) > 0 for l in lines)
    # a buffer too small for the text: whole lines only, NUL-terminated, the count still complete
    assert lib.sofie_hip_trace_begin(ctx.h) == 0
    for _ in range(3):
        ctx.check(lib.sofie_hip_relu_f32(ctx.h, ctx.ptr(x), ctx.ptr(y), x.numel()))
    small = C.create_string_buffer(24)
    assert lib.sofie_hip_trace_end(ctx.h, small, 24, C.byref(n)) == 0
    assert n.value == 3 and 1 <= len(small.value.decode().splitlines()) < 3 and small.value.decode().endswith("\n")
    ctx.sync()
    assert torch.equal(y, torch.relu(x))


# --------------------------------------------------------------------------- graph recording rules
def test_capture_rules_are_enforced():
    """Between capture_begin and capture_end the calls that would wait on, or record a memset node into, the
    capturing stream return EINVAL and leave the recording intact; a recorded graph pins the context's scratch
    buffer: a later call that would have to grow (free) it is refused until the graph is destroyed. Every kernel
    that runs here exits normally; the refused calls never reach the device."""
    import ctypes as C
    from sofie_amd import lib as L
    from sofie_amd import ops as o
    ctx = o.Context(0, guard=False)          # a context of its own: the recorded graph pins its scratch buffer
    lib, h, p = ctx.lib, ctx.h, ctx.ptr
    r = rng(7)
    M, N, K = 256, 256, 8192                 # long K, few tiles: the split-K path, partial sums in the scratch buffer
    A = r.integers(-127, 128, (M, K)).astype(np.int8)
    B = r.integers(-127, 128, (N, K)).astype(np.int8)
    scale = (r.uniform(20, 60, N) / (73.3 * 73.3 * np.sqrt(K))).astype(np.float32)
    dA, dB, dS = ctx.dev(A), ctx.dev(B), ctx.dev(scale)
    y = ctx.empty((M, N), torch.int8)
    host = np.zeros(16, np.uint8)

    def call(m=M):
        return lib.sofie_hip_qgemm_s8(h, 1, m, N, K, p(dA), K, p(dB), K, p(dS), None, 0, 0, p(y), N, L.OUT_S8)

    assert call() == 0                        # eager once: the scratch buffer gets its size
    ctx.sync()
    want = y.cpu().numpy().copy()
    assert np.array_equal(want, oracle.qgemm_s8(A, B, scale, transB=True))
    assert lib.sofie_hip_capture_begin(h) == 0
    try:
        ms = C.c_float()
        dp = C.c_void_p()
        assert lib.sofie_hip_memset(h, p(y), 0, 16) == L.EINVAL
        assert lib.sofie_hip_upload(h, p(y), host.ctypes.data_as(C.c_void_p), 16) == L.EINVAL
        assert lib.sofie_hip_download(h, host.ctypes.data_as(C.c_void_p), p(y), 16) == L.EINVAL
        assert lib.sofie_hip_sync(h) == L.EINVAL
        assert lib.sofie_hip_malloc(h, C.byref(dp), 1024) == L.EINVAL and not dp.value
        assert lib.sofie_hip_free(h, p(y)) == L.EINVAL
        assert lib.sofie_hip_timer_start(h) == L.EINVAL
        assert lib.sofie_hip_timer_stop(h, C.byref(ms)) == L.EINVAL
        assert b"capture" in lib.sofie_hip_last_error(h)
        assert call() == 0                    # recorded, not run
    except BaseException:
        lib.sofie_hip_capture_end(h, None)
        raise
    g = C.c_void_p()
    assert lib.sofie_hip_capture_end(h, C.byref(g)) == 0 and g.value
    for _ in range(3):                        # replays with eager work and waits in between
        y.zero_()
        torch.cuda.synchronize()
        assert lib.sofie_hip_graph_launch(h, g) == 0
        ctx.sync()
        assert np.array_equal(y.cpu().numpy(), want)
    # a call that needs a larger scratch buffer is refused while the graph lives ...
    A2 = ctx.dev(np.zeros((4 * M, K), np.int8))
    y2 = ctx.empty((4 * M, N), torch.int8)
    big = lambda: lib.sofie_hip_qgemm_s8(h, 1, 4 * M, N, K, p(A2), K, p(dB), K, p(dS), None, 0, 0, p(y2), N, L.OUT_S8)
    assert big() == L.EINVAL
    assert b"graph" in lib.sofie_hip_last_error(h)
    assert lib.sofie_hip_graph_launch(h, g) == 0          # ... and the graph still replays on the buffer it recorded
    ctx.sync()
    assert np.array_equal(y.cpu().numpy(), want)
    # ... and goes through once it is destroyed
    assert lib.sofie_hip_graph_destroy(h, g) == 0
    assert big() == 0
    ctx.sync()
    assert not y2.cpu().numpy().any()
    ctx.close()


# --------------------------------------------------------------------------- stacked matrix products
@pytest.mark.parametrize("sa,sb,tA,tB,relu", [
    ((2, 1, 4, 5), (3, 5, 6), 0, 0, False),          # both operands broadcast over a leading dimension
    ((2, 3, 4, 6), (6, 2), 0, 0, True),              # one matrix against a stack
    ((5, 7, 33), (5, 33, 70), 0, 0, False),
    ((3, 2, 40, 17), (3, 1, 9, 40), 1, 1, False),    # both stored transposed
    ((1, 130, 65), (4, 2, 65, 131), 0, 0, True),     # tiles of 128 x 128, ragged
])
def test_gemm_f32_stacked_is_numpy_matmul(sa, sb, tA, tB, relu):
    """sofie_hip_gemm_f32_stacked against numpy.matmul in float64 (every product reads its own matrices, broadcast
    dimensions repeat) and against the single-product entry point, which it must equal bit for bit."""
    import ctypes as C
    from sofie_amd import lib as L
    from sofie_amd import ops as o
    ctx = o.default_context()
    r = rng(900 + sum(sa) + sum(sb))
    A = r.standard_normal(sa).astype(np.float32)
    B = r.standard_normal(sb).astype(np.float32)
    a64 = np.swapaxes(A, -1, -2).astype(np.float64) if tA else A.astype(np.float64)
    b64 = np.swapaxes(B, -1, -2).astype(np.float64) if tB else B.astype(np.float64)
    truth = np.matmul(a64, b64)
    if relu:
        truth = np.maximum(truth, 0)
    lead = truth.shape[:-2]
    M, N = truth.shape[-2:]
    K = a64.shape[-1]
    la = (1,) * (len(lead) - (A.ndim - 2)) + A.shape[:-2]
    lb = (1,) * (len(lead) - (B.ndim - 2)) + B.shape[:-2]

    def strides(l, mat):
        out, s = [0] * len(l), mat
        for i in reversed(range(len(l))):
            out[i] = s if l[i] != 1 else 0
            s *= l[i]
        return out
    st_a, st_b = strides(la, A.shape[-2] * A.shape[-1]), strides(lb, B.shape[-2] * B.shape[-1])
    dA, dB = ctx.dev(A), ctx.dev(B)
    y = ctx.empty(truth.shape, torch.float32)
    n = len(lead)
    ctx.check(ctx.lib.sofie_hip_gemm_f32_stacked(ctx.h, tA, tB, M, N, K, 1.0, ctx.ptr(dA), A.shape[-1], ctx.ptr(dB), B.shape[-1],
                                                 ctx.ptr(y), N, n, (C.c_int * n)(*lead), (C.c_longlong * n)(*st_a),
                                                 (C.c_longlong * n)(*st_b), L.ACT_RELU if relu else L.ACT_NONE))
    got = ctx.ret(y, A)
    assert rel_err(got, truth) <= FP32_TOL
    # the same products one at a time
    Af = np.broadcast_to(A.reshape(la + A.shape[-2:]), lead + A.shape[-2:]).reshape((-1,) + A.shape[-2:])
    Bf = np.broadcast_to(B.reshape(lb + B.shape[-2:]), lead + B.shape[-2:]).reshape((-1,) + B.shape[-2:])
    for i in range(0, Af.shape[0], max(1, Af.shape[0] // 3)):
        one = o.gemm_f32(np.ascontiguousarray(Af[i]), np.ascontiguousarray(Bf[i]), None, 1.0, 0.0, bool(tA), bool(tB), relu)
        assert np.array_equal(one, got.reshape((-1, M, N))[i])


# --------------------------------------------------------------------------- fp32 average pooling
@pytest.mark.parametrize("cfg", [
    dict(shape=(2, 3, 9, 8), k=(3, 2), s=(2, 1), p=(0, 0, 0, 0)),
    dict(shape=(1, 4, 7, 7), k=(3, 3), s=(1, 1), p=(1, 1, 1, 1)),
    dict(shape=(2, 2, 10, 11), k=(2, 4), s=(2, 3), p=(1, 2, 1, 0)),
    dict(shape=(3, 130, 6, 6), k=(6, 6), s=(1, 1), p=(0, 0, 0, 0)),      # the global average of many planes
    dict(shape=(1, 1, 40, 300), k=(5, 7), s=(3, 4), p=(2, 3, 2, 3)),
])
def test_avgpool2d_f32(ops, cfg):
    """Same order of additions and one division as the oracle's restatement of the reference's loops: identical bits."""
    r = rng(1000 + cfg["shape"][1])
    x = r.standard_normal(cfg["shape"]).astype(np.float32)
    for include in (False, True):
        y = ops.avgpool2d(x, cfg["k"], cfg["s"], cfg["p"], include)
        assert np.array_equal(y, oracle.avgpool2d(x, cfg["k"], cfg["s"], cfg["p"], include))
