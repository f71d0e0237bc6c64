"""Indices that come from host memory: in the launch's argument block (64 or 960 of them), in two pieces, by a copy beyond."""
import numpy as np
import pytest

from dynet_amd import DyhipError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 65, 960, 961, 1920, 1921])
@pytest.mark.parametrize("dim,mult", [(1, 1.0), (20, 0.5), (67, 1.0), (256, 2.0), (1028, 1.0)])
def test_lookup_of_host_indices(dev, n, dim, mult):
    rng = np.random.default_rng(n + dim)
    table = rng.standard_normal((50, dim)).astype(np.float32)
    ids = rng.integers(0, 50, n).astype(np.uint32)
    tt, idd, fx = dev.tensor(table), dev.empty((n,), np.uint32), dev.empty((n, dim))
    want = ids.copy()
    dev.lookup_forward(ids, idd, dim, 50, tt, fx, mult)
    ids[:] = 0  # the caller's memory is its own again
    np.testing.assert_array_equal(fx.numpy(), table[want] * np.float32(mult))
    np.testing.assert_array_equal(idd.numpy(), want)


@pytest.mark.parametrize("n", [1, 64, 65, 960, 961, 1920, 1921])
def test_pnls_of_host_labels(dev, n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 33)).astype(np.float32)
    labels = rng.integers(0, 33, n).astype(np.uint32)
    xt, aux, fx = dev.tensor(x), dev.empty((3 * n,)), dev.empty((n,))
    want = labels.copy()
    dev.pnls_forward(33, n, xt, labels, aux, fx)
    labels[:] = 0
    x64 = x.astype(np.float64)
    exact = np.log(np.exp(x64).sum(1)) - x64[np.arange(n), want]
    # logarithm and difference of values below 8, each rounded once; 33 terms summed
    assert np.max(np.abs(fx.numpy() - exact)) <= 8 * 2.0 ** -23 + 33 * 2.0 ** -24


@pytest.mark.parametrize("rows,n", [(r, n) for r in (1, 64, 65, 512, 513, 4099) for n in (1, 64, 65, 960)]
                         + [(65536, 1), (70001, 64), (65537, 65)])
def test_pnls_of_host_labels_over_every_kernel_of_the_columns(dev, rows, n):
    """The labels reach the loss and, through the auxiliary memory, the gradient; up to 64 columns of 65 536 rows are cut."""
    rng = np.random.default_rng(n + rows)
    x = rng.standard_normal((n, rows)).astype(np.float32)
    labels = rng.integers(0, rows, n).astype(np.uint32)
    xt, aux, fx = dev.tensor(x), dev.empty((3 * n,)), dev.empty((n,))
    dy, dx = dev.tensor(np.ones(n, np.float32)), dev.tensor(np.zeros((n, rows), np.float32))
    dev.pnls_forward(rows, n, xt, labels, aux, fx)
    dev.pnls_backward(rows, n, xt, aux, dy, dx)
    x64, at = x.astype(np.float64), np.arange(n)
    z = np.log(np.exp(x64).sum(1))
    # logarithm and difference of values below 16, each rounded once; a term of the sum goes through up to 32 sums and merges
    bound = 16 * 2.0 ** -23 + 64 * 2.0 ** -24
    assert np.max(np.abs(fx.numpy() - (z - x64[at, labels]))) <= bound
    want = np.exp(x64 - z[:, None])
    want[at, labels] -= 1.0
    # z as above and x - z rounded below 16, under an exponential of at most one
    assert np.max(np.abs(dx.numpy() - want)) <= 2 * bound


def test_host_indices_are_not_recorded_into_a_graph(dev):
    tt, idd, fx = dev.tensor(np.ones((4, 8), np.float32)), dev.empty((3,), np.uint32), dev.empty((3, 8))
    aux, loss = dev.empty((9,)), dev.empty((3,))
    ids = np.array([1, 2, 3], np.uint32)
    dev.sync()
    dev.graph_begin()
    try:
        with pytest.raises(DyhipError, match="graph"):
            dev.lookup_forward(ids, idd, 8, 4, tt, fx)
        with pytest.raises(DyhipError, match="graph"):
            dev.pnls_forward(8, 3, fx, ids, aux, loss)
    finally:
        dev.graph_end().destroy()
