"""Row argmax at the edges of its vector loads, against numpy.

Rows that start on each 4-byte phase of a 16-byte boundary (odd lengths), rows
shorter than one 16-byte load, the sizes around one and two rounds of a
block's loads (1024 threads x 4 x 16 bytes), ties across rounds, infinities
and NaN (which never wins; a row of nothing else gives 0).
"""
import numpy as np
import pytest

from hummingflight_amd import capi

pytestmark = pytest.mark.gpu


def rows_argmax(x):
    T, n = x.shape
    xd, bd = capi.DeviceBuffer.of(x), capi.DeviceBuffer(4 * T)
    capi.call("hfmoe_argmax_rows", xd.ptr, T, n, bd.ptr, None)
    capi.call("hfmoe_synchronize")
    got = bd.download(np.int32, T)
    xd.free()
    bd.free()
    return got


@pytest.mark.parametrize("n", [1, 3, 5, 4095, 4097, 16383, 16384, 16387, 32771, 154880])
def test_row_argmax_edges(hf, n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((9, n)).astype(np.float32)
    x[1, -1] = 9.0  # the last element
    x[2, 0] = 9.0
    x[3, n // 2:] = 9.0  # ties from the middle on
    x[4, :] = -np.inf  # the first of equals, at the lowest value there is
    x[5, :] = np.nan
    x[6, rng.integers(0, n, max(1, n // 3))] = np.nan
    x[7, n // 3] = np.inf
    x[7, 2 * n // 3] = np.inf
    want = [0 if np.isnan(r).all() else int(np.nanargmax(r)) for r in x]
    assert rows_argmax(x).tolist() == want
