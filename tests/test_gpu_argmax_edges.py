"""argmax of long columns at the edges of the block kernel's 128-bit loads, against numpy."""
import numpy as np
import pytest

from dynet_amd import DevTensor
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
