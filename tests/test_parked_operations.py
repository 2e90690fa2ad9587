"""What happens to an operation that waits for its successor (``_hip.defer``), on the host: the library is a
stand-in that records the calls and fails them on demand, so nothing here touches a GPU."""
import gc

import numpy as np
import pytest

import pytortto_amd as tt
from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray

F = tt.nn.functional


class _Library:
    def __init__(self):
        self.calls, self.fail = [], set()

    def __getattr__(self, name):
        def function(*args):
            if name == 'tt_malloc':
                args[0]._obj.value = 4096 * (1 + len(self.calls))
            self.calls.append(name)
            return int(name in self.fail)
        return function

    def tt_last_error(self):
        return b'refused by the library'

    def launched(self):
        """The calls since the last look, but for memory and transfers."""
        names = [n for n in self.calls if n not in ('tt_malloc', 'tt_free', 'tt_memcpy_h2d')]
        self.calls.clear()
        return names


@pytest.fixture
def library(monkeypatch):
    stand_in = _Library()
    monkeypatch.setattr(_hip, '_lib', stand_in)
    monkeypatch.setattr(_hip, '_ready', True)
    monkeypatch.setattr(_hip, '_pending', None)
    monkeypatch.setattr(_hip, '_earlier', None)
    ops._conv2d_fwd_accepts.cache_clear()
    yield stand_in
    ops._conv2d_fwd_accepts.cache_clear()
    _hip.take_pending()
    gc.collect()                # device arrays give their blocks back to the stand-in


def _tensor(*shape, dtype=np.float32):
    return tt.Tensor(hiparray(np.ones(shape, dtype)), dtype=dtype)


def _on_device(module):
    module.cuda()
    return module


CONV, NORM = 'tt_conv2d_fwd_f32', 'tt_bn_act_fwd_train_f32'
CONV_WITH, EVAL, EVAL_RELU = 'tt_conv2d_norm_act_fwd_f32', 'tt_bn_fwd_eval_f32', 'tt_bn_relu_fwd_eval_f32'
ADD, ADD_RELU, RELU = 'tt_add_f32', 'tt_add_relu_f32', 'tt_relu_fwd_f32'


def test_a_refused_add_leaves_the_batch_norm_in_front_of_it_parked(library):
    bn = _on_device(tt.nn.BatchNorm2d(4))
    whole = _tensor(2, 4, 3, 3, dtype=np.int64)
    y = bn(_tensor(2, 4, 3, 3))
    library.launched()
    for operands in ((y, whole), (whole, y)):
        with pytest.raises(TypeError, match='float32 only'):
            operands[0] + operands[1]
    assert _hip.pending().__class__ is ops.DeferredBatchNorm
    y.data.ptr, bn.running_mean.data.ptr, bn.running_var.data.ptr
    assert library.launched() == [NORM]


def test_a_refused_add_or_batch_norm_leaves_the_convolution_in_front_of_it_parked(library):
    conv, bn = _on_device(tt.nn.Conv2d(4, 4, 1)), _on_device(tt.nn.BatchNorm2d(4))
    bn.eval()
    bn.running_var.data = hiparray(np.ones(4))              # float64
    whole = _tensor(2, 4, 3, 3, dtype=np.int64)
    with tt.no_grad():
        y = conv(_tensor(2, 4, 3, 3))
        library.launched()
        with pytest.raises(TypeError, match='float32 only'):
            y + whole
        with pytest.raises(TypeError, match='float32 only'):
            bn(y)
        assert _hip.pending().__class__ is ops.DeferredConv
        y.data.ptr
    assert library.launched() == [CONV]


@pytest.mark.parametrize('training', [True, False])
def test_arrays_of_a_launch_that_fails_after_joining_raise(library, training):
    conv, bn = _on_device(tt.nn.Conv2d(4, 4, 1)), _on_device(tt.nn.BatchNorm2d(4))
    bn.train(training)
    with tt.no_grad():
        y = bn(conv(_tensor(2, 4, 3, 3)))
        library.fail = {NORM, 'tt_conv2d_norm_act_fwd_f32'}
        with pytest.raises(RuntimeError, match='refused by the library'):
            F.relu(y).data.ptr
    library.fail = set()
    for array in (y.data,) + ((bn.running_mean.data, bn.running_var.data) if training else ()):
        with pytest.raises(RuntimeError, match='refused by the library'):
            array.ptr


def test_an_operation_behind_one_that_fails_is_marked_too(library):
    bn = _on_device(tt.nn.BatchNorm2d(4))
    y = bn(_tensor(2, 4, 3, 3))
    library.fail = {NORM}
    op = object.__new__(ops.DeferredAdd)
    op.out = hiparray.lazy((2, 2))
    with pytest.raises(RuntimeError, match='refused by the library'):
        _hip.defer(op)
    assert _hip.pending() is None
    for array in (y.data, op.out):
        with pytest.raises(RuntimeError, match='refused by the library'):
            array.ptr


def test_an_in_place_relu_that_is_refused_leaves_its_input_parked(library):
    x = _tensor(2, 4, 3, 3)
    t = x + _tensor(2, 4, 3, 3)
    t.requires_grad = True                                  # a leaf that asks for a gradient
    library.launched()
    with pytest.raises(RuntimeError, match='in-place operation'):
        F.relu(t, inplace=True)
    t.data.ptr
    assert library.launched() == ['tt_add_f32']


def test_what_the_library_refuses_is_raised_by_the_call(library):
    conv = _on_device(tt.nn.Conv2d(4, 4, 1))
    x = _tensor(2, 4, 3, 3)
    with tt.no_grad():
        assert conv(x) is not None and _hip.pending() is not None
        _hip.flush()
        library.fail = {'tt_workspace_size_conv2d_fwd_f32', CONV}
        with pytest.raises(RuntimeError, match='refused by the library'):
            conv(_tensor(2, 4, 3, 5))
        assert _hip.pending() is None


def _nothing_held(conv, bn, x):
    return F.relu(bn(conv(x)) + x)


def _rebound(conv, bn, x):
    h = conv(x)
    h = bn(h)
    h = h + x
    return F.relu(h)


def _rebound_in_place(conv, bn, x):
    h = conv(x)
    h = bn(h)
    return F.relu(h, inplace=True)


def _rebound_late(conv, bn, x):
    h = conv(x)
    h = conv(F.relu(bn(h)))             # the name still holds the first value when the second convolution is called
    return F.relu(bn(h))


def _three_in_a_row(conv, bn, x):
    return conv(F.relu(conv(bn(conv(x)))))


def _shortcut_around_the_norm(conv, bn, x):
    a = conv(x)
    return conv(F.relu(bn(a))) + a


def _residual_is_the_input_of_the_norm(conv, bn, x):
    a = conv(x)
    return F.relu(bn(a) + a)


def _norm_held(conv, bn, x):
    n = bn(conv(x))
    return F.relu(n + x) + n


def _sum_held(conv, bn, x):
    s = bn(conv(x)) + x
    return F.relu(s) + s


def _relu_input_held(conv, bn, x):
    a = conv(x)
    return F.relu(a) + a


def _all_held(conv, bn, x):
    a = conv(x)
    n = bn(a)
    s = n + x
    return a, n, s, F.relu(s)


def _two_relus(conv, bn, x):
    return F.relu(F.relu(conv(x)))


@pytest.mark.parametrize('network,launches', [
    (_nothing_held, [CONV_WITH]), (_rebound, [CONV_WITH]), (_rebound_in_place, [CONV_WITH]), (_two_relus, [CONV_WITH, RELU]),
    (_rebound_late, [CONV_WITH, CONV_WITH]), (_three_in_a_row, [CONV_WITH, CONV_WITH, CONV]),
    (_shortcut_around_the_norm, [CONV, EVAL_RELU, CONV_WITH]), (_residual_is_the_input_of_the_norm, [CONV, EVAL, ADD_RELU]),
    (_norm_held, [CONV_WITH, ADD_RELU, ADD]), (_sum_held, [CONV_WITH, RELU, ADD]), (_relu_input_held, [CONV, RELU, ADD]),
    (_all_held, [CONV, EVAL, ADD, RELU])], ids=lambda v: getattr(v, '__name__', ''))
def test_a_convolution_is_launched_once(library, network, launches):
    """What joined the convolution is one launch with it, unless a value in between is still held when the launch
    comes: that one is stored, and nothing is computed again to read it."""
    conv, bn, x = _on_device(tt.nn.Conv2d(4, 4, 1)), _on_device(tt.nn.BatchNorm2d(4)), _tensor(2, 4, 3, 3)
    bn.eval()
    with tt.no_grad():
        conv(x), _hip.flush(), library.launched()
        y = network(conv, bn, x)
        for t in y if isinstance(y, tuple) else (y,):
            t.data.ptr
    assert library.launched() == launches


def test_a_failing_convolution_leaves_the_one_behind_it_parked(library):
    """Two convolutions are parked; the first fails when a third comes: its own arrays and the third's raise, the
    second is launched as it would have been."""
    conv, x = _on_device(tt.nn.Conv2d(4, 4, 1)), _tensor(2, 4, 3, 3)
    with tt.no_grad():
        first, second = conv(x), conv(x)
        library.launched()
        library.fail = {CONV}
        with pytest.raises(RuntimeError, match='refused by the library'):
            conv(x)
        library.fail = set()
    with pytest.raises(RuntimeError, match='refused by the library'):
        first.data.ptr
    library.launched()
    second.data.ptr
    assert library.launched() == [CONV] and _hip.pending() is None


def test_taking_the_last_operation_runs_the_one_in_front_of_it(library):
    conv, x = _on_device(tt.nn.Conv2d(4, 4, 1)), _tensor(2, 4, 3, 3)
    with tt.no_grad():
        first, second = conv(x), conv(x)
        library.launched()
        assert _hip.take_pending().out is second.data and library.launched() == [CONV]
        assert first.data._buf._ptr and not second.data._buf._ptr
