"""2x2 fp32 max pooling of stride 2 on k_maxpool2d_f32_pairs: two and four outputs per thread, odd heights, a last column or row without a
window, and the rows it leaves to k_maxpool2d, bit for bit against the oracle's order of comparisons (zeros of both signs, NaN)."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,h,w", [(1, 2, 4), (3, 5, 8), (7, 13, 12), (50, 40, 40), (33, 21, 20), (5, 9, 6), (5, 8, 9), (2, 3, 516)])
def test_maxpool_pairs(nc, h, w):
    from sofie_amd import ops
    r = np.random.default_rng(h * w)
    x = r.integers(-2, 3, (1, nc, h, w)).astype(np.float32)
    x[r.random(x.shape) < 0.2] = -0.0
    x[r.random(x.shape) < 0.05] = -np.inf
    got, ref = ops.maxpool2d(x, (2, 2), (2, 2)), oracle.maxpool2d(x, (2, 2), (2, 2))
    assert np.array_equal(got.view(np.int32), ref.view(np.int32))
    # NaN never wins; where there is nothing else the lowest value does
    x[r.random(x.shape) < 0.5] = np.nan
    q = x[:, :, :h // 2 * 2, :w // 2 * 2].reshape(1, nc, h // 2, 2, w // 2, 2)
    assert np.array_equal(ops.maxpool2d(x, (2, 2), (2, 2)), np.where(np.isnan(q), -np.inf, q).max(axis=(3, 5)))


@pytest.mark.parametrize("pads", [(0, 0, 1, 0), (0, 0, 0, 1), (0, 0, 1, 1), (0, 0, 2, 0), (0, 0, 0, 4), (0, 0, 3, 5), (1, 0, 0, 0), (0, 1, 0, 1)])
@pytest.mark.parametrize("nc,h,w", [(1, 7, 8), (5, 7, 8), (5, 8, 8), (3, 41, 40), (2, 2, 4), (1, 3, 4), (9, 6, 20)])
def test_windows_that_reach_over_the_planes_end(nc, h, w, pads):
    """Pads behind the plane (and in front of it): cells that are not there are left out, not the next plane's or those behind the tensor.
    Every value lies below every value of the plane behind it, so that one cell of that would be seen."""
    from sofie_amd import ops
    r = np.random.default_rng(h * w + sum(pads))
    x = (r.integers(-2, 3, (1, nc, h, w)) + 10 * np.arange(nc)[None, :, None, None]).astype(np.float32)
    x[r.random(x.shape) < 0.1] = -np.inf
    got, ref = ops.maxpool2d(x, (2, 2), (2, 2), pads), oracle.maxpool2d(x, (2, 2), (2, 2), pads)
    assert got.shape == ref.shape and np.array_equal(got.view(np.int32), ref.view(np.int32))
