"""Operations whose launch waits for a successor, on the device: errors come from the call that is wrong."""
import numpy as np
import pytest

import pytortto_amd as tt
from pytortto_amd import _hip
from pytortto_amd.xparray import hiparray

pytestmark = pytest.mark.gpu
F = tt.nn.functional


def _tensor(*shape, seed=0):
    return tt.Tensor(hiparray(np.random.default_rng(seed).standard_normal(shape).astype(np.float32)))


# x, weight, arguments of conv2d
REFUSED = [((1, 8, 8, 8), (6, 2, 3, 3), dict(groups=4)), ((1, 2, 8, 8), (2, 2, 3, 3), dict(dilation=(0, 1))),
           ((1, 2, 8, 8), (2, 2, 3, 3), dict(padding=(-1, 0))), ((1, 65536, 1, 1), (65536, 1, 1, 1), dict(groups=65536)),
           ((1, 1, 16384, 1), (1, 1, 1, 1), {}), ((0, 2, 8, 8), (2, 2, 3, 3), {})]


@pytest.mark.parametrize('x,w,kw', REFUSED, ids=lambda v: str(v))
def test_a_refused_convolution_raises_with_and_without_gradients(x, w, kw):
    x, w = tt.Tensor(hiparray.zeros(x)), tt.Tensor(hiparray.zeros(w))
    x.requires_grad = True
    with pytest.raises(RuntimeError) as first:
        F.conv2d(x, w, **kw)
    with tt.no_grad():
        for _ in range(2):
            with pytest.raises(RuntimeError) as second:
                F.conv2d(x, w, **kw)
            assert str(second.value) == str(first.value)
    assert _hip.pending() is None


@pytest.mark.parametrize('behind_conv', [True, False])
def test_a_refused_evaluation_batch_norm_raises_with_and_without_gradients(behind_conv):
    x, w, stats = _tensor(2, 8, 5, 5), _tensor(8, 8, 1, 1), [tt.zeros(8), tt.ones(8)]      # statistics left on the host
    gamma = _tensor(8)
    gamma.requires_grad = True
    for exc in (True, False):
        h = F.conv2d(x, w) if behind_conv else x
        with pytest.raises(AttributeError):
            if exc:
                F.batch_norm(h, *stats, weight=gamma)
            else:
                with tt.no_grad():
                    F.batch_norm(h, *stats, weight=gamma)
    with tt.no_grad():
        h = F.conv2d(x, w)
        with pytest.raises(AttributeError):
            F.batch_norm(h, *stats)
        np.testing.assert_allclose(h.data.get(), np.einsum('nchw,kc->nkhw', x.data.get(), w.data.get()[:, :, 0, 0]),
                                   rtol=1e-4, atol=1e-5)
        wide = tt.Tensor(hiparray.zeros((1, 65536, 1, 2)))
        flat = tt.Tensor(hiparray.zeros(65536))
        with pytest.raises(RuntimeError, match='65535 channels'):
            F.batch_norm(wide, flat, flat)
        with pytest.raises(RuntimeError, match='must be positive'):
            F.batch_norm(tt.Tensor(hiparray.zeros((0, 8, 2, 2))), _tensor(8), _tensor(8))
