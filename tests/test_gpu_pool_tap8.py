"""Pooling with tap indexes of a byte and of an int: the same values, at the line between them and on both
the staged kernels and the ones for rows too long to stage."""
import numpy as np
import pytest

from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray

pytestmark = pytest.mark.gpu


# n, c, h, w, kernel, stride, padding, dilation
@pytest.mark.parametrize('case', [(2, 3, 19, 17, (16, 16), (1, 2), (3, 0), (1, 1)), (2, 3, 21, 18, (3, 3), (2, 2), (1, 1), (1, 1)),
                                  (1, 2, 9, 4100, (2, 3), (2, 3), (0, 1), (1, 2)), (1, 1, 5, 300, (1, 256), (1, 1), (0, 0), (1, 1))])
def test_byte_and_int_taps_agree(case):
    n, c, h, w, ks, st, pd, dl = case
    rng = np.random.default_rng(sum(ks))
    x = rng.integers(-3, 4, (n, c, h, w)).astype(np.float32)          # ties
    x.flat[:5] = [np.nan, np.inf, -np.inf, np.nan, 0]
    out = tuple((v + 2 * p - d * (k - 1) - 1) // s + 1 for v, p, d, k, s in zip((h, w), pd, dl, ks, st))
    xd = hiparray(x)
    y, tap = ops.maxpool2d_fwd(xd, out, ks, st, pd, dl)
    assert tap.dtype == np.uint8
    y4, tap4 = hiparray.empty(y.shape), hiparray.empty(y.shape, np.int32)
    geometry = (n * c, h, w, *out, *ks, *st, *pd, *dl)
    _hip.call('tt_maxpool2d_fwd_f32', xd.ptr, y4.ptr, tap4.ptr, *geometry)
    np.testing.assert_array_equal(y.get(), y4.get())
    np.testing.assert_array_equal(tap.get(), tap4.get())
    dy = hiparray(rng.standard_normal(y.shape).astype(np.float32))
    np.testing.assert_array_equal(ops.maxpool2d_bwd(dy, tap, (h, w), ks, st, pd, dl).get(),
                                  ops.maxpool2d_bwd(dy, tap4, (h, w), ks, st, pd, dl).get())


def test_more_taps_than_a_byte_counts_take_ints():
    x = hiparray(np.random.default_rng(0).standard_normal((1, 2, 20, 20)).astype(np.float32))
    y, tap = ops.maxpool2d_fwd(x, (4, 4), (17, 17), (1, 1), (0, 0), (1, 1))
    assert tap.dtype == np.int32
    assert ops.maxpool2d_bwd(y, tap, (20, 20), (17, 17), (1, 1), (0, 0), (1, 1)).shape == (1, 2, 20, 20)
    with pytest.raises(RuntimeError, match='do not fit a byte'):
        _hip.call('tt_maxpool2d_fwd_tap8_f32', x.ptr, y.ptr, tap.ptr, 2, 20, 20, 4, 4, 17, 17, 1, 1, 0, 0, 1, 1)
