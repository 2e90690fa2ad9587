"""What follows a convolution in an evaluation pass, applied to its accumulators before they are
stored: BatchNorm with given statistics, residual add, ReLU -- the same bits as the separate launches."""
import numpy as np
import pytest

import pytortto_amd as tt
from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray

pytestmark = pytest.mark.gpu
F = tt.nn.functional

# n, c, h, w, k, r, stride, pad, groups, bias: rows that are not whole groups of eight, one pixel, partial
# tiles, shared reductions (few tiles, many channels), 64-row tiles, groups, 7x7 taps, 1x1 at whole chunks
CASES = [(1, 3, 5, 5, 5, 3, 1, 1, 1, True), (2, 64, 9, 7, 130, 3, 1, 1, 1, False), (2, 256, 7, 7, 512, 3, 1, 1, 1, False),
         (3, 64, 14, 14, 64, 1, 1, 0, 1, False), (2, 128, 8, 8, 257, 1, 1, 0, 1, True), (4, 32, 13, 13, 48, 3, 2, 1, 2, True),
         (2, 3, 33, 33, 64, 7, 2, 3, 1, False), (1, 2048, 7, 7, 512, 1, 1, 0, 1, False), (16, 64, 28, 28, 256, 1, 1, 0, 1, False)]


def _host(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize('math', ['f32', 'bf16', 'bf16x3'])
@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(map(str, c)))
def test_same_bits_as_separate_launches(case, math):
    n, c, h, w, k, r, st, pad, groups, with_bias = case
    rng = np.random.default_rng(sum(case))
    x, wt = hiparray(_host(rng, n, c, h, w)), hiparray(_host(rng, k, c // groups, r, r) * 0.1)
    bias = hiparray(_host(rng, k)) if with_bias else None
    gamma, beta, mean, var = (hiparray(v) for v in (_host(rng, k), _host(rng, k), _host(rng, k),
                                                    rng.uniform(0.1, 2, k).astype(np.float32)))
    geometry = ((st, st), (pad, pad), (1, 1), groups)
    _hip.set_conv_math(math)
    try:
        y = ops.conv2d_fwd(x, wt, bias, *geometry)
        residual = hiparray(_host(rng, *y.shape))
        bn = ops.bn_fwd_eval(y, gamma, beta, mean, var, 1e-5)[0]
        plain = ops.bn_fwd_eval(y, None, None, mean, var, 1e-5)[0]
        for norm, res, relu in ((1, 0, 0), (1, 0, 1), (1, 1, 1), (1, 1, 0), (0, 1, 0), (0, 0, 1), (2, 0, 1)):
            want = {0: y, 1: bn, 2: plain}[norm]
            want = ops.add(want, residual) if res else want
            want = ops.relu_fwd(want) if relu else want
            op = ops.DeferredConv(x, wt, bias, *ops._conv2d_geometry(x, wt, bias, *geometry))
            if norm:
                op.absorb_norm(mean, var, gamma if norm == 1 else None, beta if norm == 1 else None, 1e-5)
                assert _hip.take_pending() is op
            if res:
                op.absorb_add(residual)
                assert _hip.take_pending() is op
            if relu:
                got = op.run_with_relu(hiparray.empty(y.shape))
            else:
                op.run()
                got = op.out
            np.testing.assert_array_equal(got.get(), want.get())
    finally:
        _hip.set_conv_math('f32')


def test_evaluation_pass_joins_the_convolution_and_keeps_every_value_readable():
    tt.manual_seed(0)
    conv, bn, short = tt.nn.Conv2d(16, 24, 3, padding=1), tt.nn.BatchNorm2d(24), tt.nn.Conv2d(16, 24, 1, bias=False)
    bn.running_mean.copy_(np.random.randn(24)), bn.running_var.copy_(np.random.rand(24) + 0.5)
    for m in (conv, bn, short):
        m.cuda()
        m.eval()
    x = tt.randn(3, 16, 9, 9).cuda()

    def forward():
        a = conv(x)
        b = bn(a)
        s = short(x)
        c = s + b
        return a, b, s, c, F.relu(c), F.relu(bn(conv(x))), F.relu(bn(a))

    want = [t.data.get() for t in forward()]            # gradients on: every launch on its own
    with tt.no_grad():
        b = bn(conv(x))
        assert _hip.pending().__class__ is ops.DeferredConv and _hip.pending().norm is not None
        c = b + short(x)
        assert _hip.pending().__class__ is ops.DeferredConv and _hip.pending().residual is not None
        F.relu(c)
        got = forward()
        x_was = x.data.get()
        conv.weight.data.fill(0.0)                      # in place: what is still to be produced comes first
        x.data.fill(0.0)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g.data.get(), w)
    assert x_was.any()
