"""The one-launch chain of fully connected layers at the edges of its tiles: 16 rows and 16 columns of an output tile, pieces of 64
rows of a weight matrix, parts of K, and the rows per workgroup (16, 32, 64 by the number of rows and the widths)."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from sofie_amd import ops as o
    return o


def exact_and_bound(x, Ws, bs, relus):
    """The float64 result, and a bound on what fp32 sums of K products and a bias in any order are away from it, carried through
    the layers (ReLU passes an error on or takes it away)."""
    h, err = x.astype(np.float64), np.zeros_like(x, dtype=np.float64)
    for W, b, relu in zip(Ws, bs, relus):
        W, b = W.astype(np.float64), 0.0 if b is None else b.astype(np.float64)
        mag = (np.abs(h) + err) @ np.abs(W) + np.abs(b)
        err = err @ np.abs(W) + (W.shape[0] + 1) * 2.0 ** -24 * 1.01 * mag
        h = h @ W + b
        if relu:
            h = np.maximum(h, 0.0)
    return h, err


@pytest.mark.parametrize("M,dims", [(1, [1, 1]), (15, [16, 16]), (17, [17, 15, 1]), (16, [64, 16, 64]), (33, [65, 63, 127, 5]),
                                    (256, [64, 128, 64, 8]), (5, [1024, 1024, 1024]), (3, [129, 33, 257]), (40, [20] * 17),
                                    (4097, [60, 33, 9]), (4097, [512, 500, 7]), (4111, [700, 601, 3]), (16385, [50, 129, 66, 8]),
                                    (16400, [300, 257])])
def test_mlp_f32_edges(ops, M, dims):
    r = np.random.default_rng(M + sum(dims))
    n = len(dims) - 1
    x = r.standard_normal((M, dims[0])).astype(np.float32)
    Ws = [(r.standard_normal((a, b)) / np.sqrt(a)).astype(np.float32) for a, b in zip(dims, dims[1:])]
    bs = [r.standard_normal(b).astype(np.float32) if i % 3 != 1 else None for i, b in enumerate(dims[1:])]
    relus = [i + 1 < n for i in range(n)]
    h, err = exact_and_bound(x, Ws, bs, relus)
    got = ops.mlp_f32(x, Ws, bs, relus).astype(np.float64)
    assert got.shape == h.shape
    assert np.all(np.abs(got - h) <= err), (M, dims, np.max(np.abs(got - h) / err))


@pytest.mark.parametrize("M,dims", [(5, [1024, 1024, 1024]), (70, [300, 257, 300, 10])])
def test_mlp_f32_recorded_without_scratch_memory(ops, M, dims):
    """Wide layers take a launch each, with scratch memory between them; a recording on a context that has none takes one launch
    for all of them, and every replay gives the same result."""
    ctx = ops.Context(0, stream=torch.cuda.Stream())
    r = np.random.default_rng(7)
    n = len(dims) - 1
    Ws = [(r.standard_normal((a, b)) / np.sqrt(a)).astype(np.float32) for a, b in zip(dims, dims[1:])]
    bs = [r.standard_normal(b).astype(np.float32) for b in dims[1:]]
    x = r.standard_normal((M, dims[0])).astype(np.float32)
    h, err = exact_and_bound(x, Ws, bs, [True] * n)
    xd, wd, bd = ctx.dev(x, torch.float32), [ctx.dev(w, torch.float32) for w in Ws], [ctx.dev(b, torch.float32) for b in bs]
    y = torch.zeros((M, dims[-1]), device="cuda")
    args = (n, (C.c_int * (n + 1))(*dims), (C.c_void_p * n)(*[t.data_ptr() for t in wd]), (C.c_void_p * n)(*[t.data_ptr() for t in bd]),
            (C.c_int * n)(*[1] * n), C.c_void_p(xd.data_ptr()), dims[0], C.c_void_p(y.data_ptr()), dims[-1], M)
    torch.cuda.synchronize()
    graph = C.c_void_p()
    ctx.check(ctx.lib.sofie_hip_capture_begin(ctx.h))
    ctx.check(ctx.lib.sofie_hip_mlp_f32(ctx.h, *args))
    ctx.check(ctx.lib.sofie_hip_capture_end(ctx.h, C.byref(graph)))
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        ctx.check(ctx.lib.sofie_hip_graph_launch(ctx.h, graph))
        ctx.check(ctx.lib.sofie_hip_sync(ctx.h))
        assert np.all(np.abs(y.cpu().numpy() - h) <= err)
    ctx.check(ctx.lib.sofie_hip_graph_destroy(ctx.h, graph))
    y.zero_()
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_mlp_f32(ctx.h, *args))      # the scratch buffer may grow now
    ctx.check(ctx.lib.sofie_hip_sync(ctx.h))
    assert np.all(np.abs(y.cpu().numpy() - h) <= err)
    ctx.close()


@pytest.mark.parametrize("M,dims", [(3, [40, 40]), (700, [40, 24]), (5000, [300, 300]), (40000, [500, 500]), (300, [64, 100, 64]), (300, [600, 700, 600])])
def test_mlp_f32_over_its_own_input(ops, M, dims):
    """y is x: every row is taken in before anything of it is written, whatever the number of layers and the kernel."""
    r = np.random.default_rng(M)
    n, ld = len(dims) - 1, dims[0]
    Ws = [(r.standard_normal((a, b)) / np.sqrt(a)).astype(np.float32) for a, b in zip(dims, dims[1:])]
    bs = [r.standard_normal(b).astype(np.float32) for b in dims[1:]]
    x = r.standard_normal((M, ld)).astype(np.float32)
    h, err = exact_and_bound(x, Ws, bs, [True] * n)
    ctx = ops.default_context()
    xd, wd, bd = ctx.dev(x.copy()), [ctx.dev(w) for w in Ws], [ctx.dev(b) for b in bs]
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_mlp_f32(ctx.h, n, (C.c_int * (n + 1))(*dims), (C.c_void_p * n)(*[t.data_ptr() for t in wd]),
                                        (C.c_void_p * n)(*[t.data_ptr() for t in bd]), (C.c_int * n)(*[1] * n), C.c_void_p(xd.data_ptr()), ld,
                                        C.c_void_p(xd.data_ptr()), ld, M))
    ctx.sync()
    got = xd.cpu().numpy()
    assert np.all(np.abs(got[:, :dims[-1]] - h) <= err)
    assert np.array_equal(got[:, dims[-1]:], x[:, dims[-1]:])


def test_mlp_f32_rows_of_several_launches(ops):
    """2^26 rows of 16 per workgroup of 1024 threads: as many threads as a launch does not hold any more."""
    M, dims = (1 << 26) + 3, [1, 600, 600, 1]
    r = np.random.default_rng(26)
    Ws = [(r.standard_normal((a, b)) / np.sqrt(a)).astype(np.float32) for a, b in zip(dims, dims[1:])]
    bs = [r.standard_normal(b).astype(np.float32) for b in dims[1:]]
    ctx = ops.default_context()
    xd, y = torch.linspace(-3.0, 3.0, M, device="cuda"), torch.zeros(M, device="cuda")
    wd, bd = [ctx.dev(w) for w in Ws], [ctx.dev(b) for b in bs]
    torch.cuda.synchronize()
    ctx.check(ctx.lib.sofie_hip_mlp_f32(ctx.h, 3, (C.c_int * 4)(*dims), (C.c_void_p * 3)(*[t.data_ptr() for t in wd]),
                                        (C.c_void_p * 3)(*[t.data_ptr() for t in bd]), (C.c_int * 3)(1, 1, 0), C.c_void_p(xd.data_ptr()), 1,
                                        C.c_void_p(y.data_ptr()), 1, M))
    ctx.sync()
    rows = np.concatenate([np.arange(20), r.integers(0, M, 50), np.arange((1 << 25) - 20, (1 << 25) + 20), np.arange(M - 20, M)])
    pick = torch.from_numpy(rows).cuda()
    h, err = exact_and_bound(xd[pick].cpu().numpy()[:, None], Ws, bs, [True, True, False])
    assert np.all(np.abs(y[pick].cpu().numpy()[:, None] - h) <= err)


@pytest.mark.parametrize("N", [5, 17, 100])
def test_mlp_f32_infinite_weight_stays_in_its_column(ops, N):
    """Lanes behind a layer's last column hold weights of the next row; nothing of theirs reaches a result."""
    r = np.random.default_rng(N)
    x = r.uniform(0.5, 1.0, (20, 37)).astype(np.float32)
    W = r.standard_normal((37, N)).astype(np.float32)
    ref = ops.mlp_f32(x, [W], [None], [False])
    W[:, 0] = np.inf
    got = ops.mlp_f32(x, [W], [None], [False])
    assert np.all(got[:, 0] == np.inf) and np.array_equal(got[:, 1:], ref[:, 1:])


@pytest.mark.parametrize("M,N1,N2,kernel", [(20, 5, 17, "k_mlp_f32"), (600, 17, 5, "k_mlp_f32"), (5000, 100, 30, "k_mlp_f32"),
                                            (9000, 33, 9, "k_mlp_f32"), (17500, 30, 12, "k_mlp_f32"), (20, 30, 17, "k_mlp_f32_row"),
                                            (500, 100, 9, "k_mlp_f32_row"), (8, 16, 768, "k_mlp_f32_row")])
def test_mlp_f32_chain_keeps_infinite_weights_in_their_columns(ops, M, N1, N2, kernel):
    """The same inside the chain kernels, on 16, 32 and 64 rows per workgroup and on one: an infinite column of the last layer (the
    lanes behind its last column hold it too) is its column of the result, a column of minus infinity of the first layer is
    a zero behind the ReLU."""
    r = np.random.default_rng(M + N1)
    dims = [37, N1, N2]
    x = r.uniform(0.5, 1.0, (M, 37)).astype(np.float32)
    Ws = [r.uniform(0.1, 1.0, (a, b)).astype(np.float32) for a, b in zip(dims, dims[1:])]
    Ws[0][:, 0], Ws[1][0, :] = -1.0, 0.0
    ctx = ops.default_context()

    def run():
        buf, n = C.create_string_buffer(4096), C.c_int(-1)
        assert ctx.lib.sofie_hip_trace_begin(ctx.h) == 0
        try:
            y = ops.mlp_f32(x, Ws, [None, None], [True, False])
        finally:
            assert ctx.lib.sofie_hip_trace_end(ctx.h, buf, 4096, C.byref(n)) == 0
        assert [l.split()[0] for l in buf.value.decode().splitlines()] == [kernel]
        return y

    ref = run()
    assert np.all(np.isfinite(ref))
    Ws[1][1:, 0] = np.inf
    got = run()
    assert np.all(got[:, 0] == np.inf) and np.array_equal(got[:, 1:], ref[:, 1:])
    Ws[0][:, 0] = -np.inf
    again = run()
    assert np.array_equal(again, got)
