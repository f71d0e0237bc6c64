"""Matrices of a batch times a vector each, the transposed product and the rank-one update (an attention over a batch), at the
edges of the streaming kernels' loads, against fp64."""
import numpy as np
import pytest

from tests.util import f32

pytestmark = pytest.mark.gpu


def _check(got, subscripts, a, b, y0):
    """Every term and every partial sum is rounded once, by at most 2^-24 of the sum of the terms' magnitudes."""
    a, b, y0 = (x.astype(np.float64) for x in (a, b, y0))
    exact = np.einsum(subscripts, a, b) + y0
    terms = a.shape[1] if subscripts != "imk,ik->im" else a.shape[2]
    bound = (terms + 2) * 2.0 ** -24 * (np.einsum(subscripts, np.abs(a), np.abs(b)) + np.abs(y0))
    assert np.all(np.abs(got - exact) <= bound)


# M columns of A an item (pairs to a wavefront, eight to a block), K deep (256 a lane's four loads), enough items for the
# one-column kernel (M * items >= 2048) and one fewer
@pytest.mark.parametrize("M,K,items,pad", [(35, 1024, 64, 0), (1, 256, 2048, 0), (1, 260, 2047, 0), (2, 1020, 1024, 8),
                                           (9, 1028, 228, 4), (33, 2052, 70, 0), (8, 508, 300, 0),
                                           (64, 1024, 128, 0), (64, 1028, 128, 0), (160, 512, 128, 0)])  # 32 MB of A, and more
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_transposed_matrix_times_vector_of_a_batch(dev, M, K, items, pad, beta):
    rng = np.random.default_rng(M * K)
    a = f32(rng.standard_normal((items, M * K + pad)))
    v, y0 = f32(rng.standard_normal((items, K))), f32(rng.standard_normal((items, M)))
    y = dev.tensor(y0)
    dev.gemm_strided_batched(1, 0, M, 1, K, dev.tensor(a), M * K + pad, dev.tensor(v), K, beta, y, M, items)
    _check(y.numpy(), "imk,ik->im", a[:, :M * K].reshape(items, M, K), v, beta * y0)


@pytest.mark.parametrize("K", [256, 1020, 1024, 1028])
def test_transposed_matrix_of_a_batch_with_infinities(dev, K):
    """An infinity in the last rows stays one: what a lane fetches past the end is not multiplied."""
    M, items = 40, 64
    rng = np.random.default_rng(K)
    a, v = f32(rng.standard_normal((items, M, K))), f32(rng.standard_normal((items, K)))
    v[:, -4:] = 0.5
    a[1, 3, -1], a[2, 5, -4], a[3, 7, -2] = np.inf, -np.inf, np.nan
    y = dev.empty((items, M))
    dev.gemm_strided_batched(1, 0, M, 1, K, dev.tensor(a), M * K, dev.tensor(v), K, 0.0, y, M, items)
    got = y.numpy()
    assert got[1, 3] == np.inf and got[2, 5] == -np.inf and np.isnan(got[3, 7])
    got[1, 3] = got[2, 5] = got[3, 7] = 0.0
    assert np.all(np.isfinite(got))


@pytest.mark.parametrize("K", [1, 32, 33, 35, 48, 49, 64, 65])  # depths in one round of loads a wavefront, and one more
@pytest.mark.parametrize("M,items", [(256, 3), (260, 20), (1024, 8)])
def test_matrix_times_vector_of_a_batch(dev, M, K, items):
    rng = np.random.default_rng(M + K)
    a, v, y0 = (f32(rng.standard_normal(s)) for s in ((items, K, M), (items, K), (items, M)))
    y = dev.tensor(y0)
    dev.gemm_strided_batched(0, 0, M, 1, K, dev.tensor(a), M * K, dev.tensor(v), K, 1.0, y, M, items)
    _check(y.numpy(), "ikm,ik->im", a, v, y0)


@pytest.mark.parametrize("M,N,items", [(256, 1, 2), (260, 9, 30), (1024, 35, 16)])
@pytest.mark.parametrize("K", [1, 2])
def test_rank_one_update_of_a_batch(dev, M, N, K, items):
    rng = np.random.default_rng(M + N)
    l, r, y0 = (f32(rng.standard_normal(s)) for s in ((items, K, M), (items, K, N), (items, N, M)))
    y = dev.tensor(y0)
    dev.gemm_strided_batched(0, 1, M, N, K, dev.tensor(l), M * K, dev.tensor(r), N * K, 1.0, y, M * N, items)
    _check(y.numpy(), "ikm,ikn->inm", l, r, y0)
