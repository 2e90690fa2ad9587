"""Operations whose launch waits for a successor, on the device: errors come from the call that is wrong, and every
value that is held has the bits of the separate launches."""
import itertools

import numpy as np
import pytest

import pytortto_amd as tt
from pytortto_amd import _hip, ops
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


@pytest.fixture(params=['f32', 'bf16', 'bf16x3', 'channel-last'])
def math(request):
    _hip.set_conv_math('bf16' if request.param == 'channel-last' else request.param)
    _hip.call('tt_conv2d_bf16_first_enable', 3 if request.param == 'channel-last' else 1)
    try:
        yield request.param
    finally:
        _hip.call('tt_conv2d_bf16_first_enable', 1)
        _hip.set_conv_math('f32')


@pytest.mark.parametrize('norm,add,relu', [v for v in itertools.product((0, 1), (0, 1), (0, 1, 2)) if any(v)])
def test_values_held_between_are_those_of_separate_launches(norm, add, relu, math):
    """Each set of values in between that a caller can hold; relu 2: in place."""
    n, c, k = 2, 6, 20
    x, w, residual, beta, mean, gamma = (_tensor(*s, seed=i) for i, s in
                                         enumerate(((n, c, 9, 7), (k, c, 3, 3), (n, k, 9, 7), (k,), (k,), (k,))))
    var = tt.Tensor(hiparray(np.random.default_rng(9).uniform(0.1, 2, k).astype(np.float32)))
    want = [ops.conv2d_fwd(x.data, w.data, None, (1, 1), (1, 1), (1, 1), 1)]
    if norm:
        want.append(ops.bn_fwd_eval(want[-1], gamma.data, beta.data, mean.data, var.data, 1e-5)[0])
    if add:
        want.append(ops.add(want[-1], residual.data))
    if relu == 1:
        want.append(ops.relu_fwd(want[-1]))
    elif relu:
        want[-1] = ops.relu_fwd(want[-1])
    steps = ([lambda v: F.batch_norm(v, mean, var, gamma, beta)] if norm else []) + ([lambda v: v + residual] if add else []) + \
        ([lambda v: F.relu(v, inplace=relu == 2)] if relu else [])
    with tt.no_grad():
        for held in itertools.product((False, True), repeat=len(steps)):
            values = []
            h = F.conv2d(x, w, padding=(1, 1))
            for step, keep in zip(steps, held):
                values.append(h if keep else None)
                h = step(h)
            values = values[:len(want) - 1] + [h]
            x_was = x.data.get()            # a call into the library: the launch happens here
            for got, ref in zip(values, want):
                if got is not None:
                    np.testing.assert_array_equal(got.data.get(), ref.get())
            assert x_was.any()
