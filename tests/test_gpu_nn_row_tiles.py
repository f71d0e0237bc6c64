"""Products with a narrow right operand over rows that are no multiple of 32: row tiles in consecutive runs, one to an XCD, with
tiles past the last one; against fp64."""
import numpy as np
import pytest

from tests.util import f32

pytestmark = pytest.mark.gpu


# one and two row tiles of 32 a block, the depth in one block and over several; a last tile of one row; tiles padded to a
# multiple of eight, none to pad, and where padding would cost a round of the CUs (85 x 3 of 256)
@pytest.mark.parametrize("M,N,K", [(33, 32, 64), (257, 40, 128), (1000, 32, 256), (2600, 20, 1300), (2599, 64, 1300),
                                   (5001, 33, 96), (10000, 17, 64), (2700, 96, 128), (2705, 70, 520), (16417, 32, 64),
                                   (10001, 64, 256), (2500, 32, 1024)])
def test_narrow_products_over_ragged_rows(dev, M, N, K):
    rng = np.random.default_rng(M + N)
    W, x, b = f32(rng.standard_normal((K, M))), f32(rng.standard_normal((N, K))), f32(rng.standard_normal(M))
    fx, dx = dev.empty((N, M)), dev.tensor(f32(np.ones((N, M))))
    dev.affine_forward(M, N, K, dev.tensor(b), dev.tensor(W), dev.tensor(x), fx)
    dev.gemm_nn(M, N, K, dev.tensor(W), dev.tensor(x), 1.0, dx)
    exact, size = x.astype(np.float64) @ W, np.abs(x).astype(np.float64) @ np.abs(W)
    # every product and every partial sum is rounded once, by at most 2^-24 of the sum of the terms' magnitudes
    assert np.all(np.abs(fx.numpy() - (exact + b)) <= (K + 4) * 2.0 ** -24 * (size + np.abs(b)))
    assert np.all(np.abs(dx.numpy() - (exact + 1)) <= (K + 4) * 2.0 ** -24 * (size + 1))
