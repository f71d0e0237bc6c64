"""argmax of long columns at the edges of the block kernel's 128-bit loads, against numpy."""
import numpy as np
import pytest

from dynet_amd import DevTensor
from oracle import cpu_oracle as orc
from tests.util import f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 2, 3])  # of the first column, in floats
@pytest.mark.parametrize("rows", [2049, 4099, 8192, 8193, 10000, 16385, 20002])  # block sizes; one round of loads and more
def test_first_maximum_of_a_column(dev, rows, offset):
    cols = 24
    x = f32(np.random.default_rng(rows + offset).standard_normal((cols, rows)))
    places = [0, 1, 2, 3, 4, 5, rows // 2, rows - 5, rows - 4, rows - 3, rows - 2, rows - 1]
    for c, r in enumerate(places):
        x[c, r] = 9.0
        x[c, min(r + 1031, rows - 1)] = 9.0  # the first of two
    x[12] = -np.inf
    x[13] = np.inf
    x[14] = 2.0
    x[15, :] = -np.inf
    x[15, rows - 2] = -1e38
    x[16, 0] = np.nan                     # nothing is greater than it
    x[17, 7] = x[17, rows // 3] = np.nan  # passed over
    x[18, 1:] = np.nan
    whole = dev.tensor(np.concatenate([np.zeros(offset, np.float32), x.ravel()]))
    idx = dev.empty(cols, np.int64)
    dev.argmax_cols(rows, cols, DevTensor(dev, whole.ptr + 4 * offset, (cols, rows), np.float32), idx)
    want = np.where(np.isnan(x), -np.inf, x).argmax(axis=1)
    want[16] = 0
    assert np.array_equal(idx.numpy(), want)


# a thread, a wavefront, a block and chunks of a column
@pytest.mark.parametrize("rows,cols", [(1, 20), (5, 20), (32, 20), (33, 20), (64, 20), (100, 20), (2048, 20), (2049, 20), (8193, 20),
                                       (65536, 20), (70001, 20), (65536, 80)])
def test_not_a_number_is_passed_over_at_every_length(dev, rows, cols):
    rng = np.random.default_rng(rows)
    x = f32(rng.standard_normal((cols, rows)))
    x[0, 0] = np.nan
    x[1, 1:] = np.nan
    x[2, :-1] = np.nan
    x[3] = np.nan
    x[4] = -np.inf
    x[5] = -np.inf
    x[5, rows // 2:] = np.nan
    x[6] = -np.inf
    x[6, rows - 1] = -3e38
    for c in range(7, 14):
        x[c, rng.random(rows) < 0.5] = np.nan
    x[14, : rows // 2] = -np.inf
    x[15, 1:: 64] = np.nan  # what one lane of a wavefront reads first
    x[16, 1: 64] = np.nan
    x[17] = np.inf
    x[17, 0] = -np.inf
    idx, fx = dev.empty(cols, np.int64), dev.empty((cols, rows))
    dev.argmax_cols(rows, cols, dev.tensor(x), idx)
    assert np.array_equal(idx.numpy(), orc.argmax_cols(rows, cols, x))
    dev.argmax_onehot_forward(rows, cols, dev.tensor(x), idx, fx)
    assert np.array_equal(fx.numpy().argmax(axis=1), orc.argmax_cols(rows, cols, x))
