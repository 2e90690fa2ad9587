"""What a residual block puts around its convolutions and BatchNorms, inside their kernels: the residual
add and ReLU behind a training BatchNorm, the ReLU's mask formed from x in its backward, and the
accumulation of a second gradient and the ReLU's mask in the kernels that write an input gradient --
the same bits as the separate launches."""
import numpy as np
import pytest

import pytortto_amd as tt
from pytortto_amd import _hip, ops
from pytortto_amd.autograd import grad_nn
from pytortto_amd.xparray import hiparray

pytestmark = pytest.mark.gpu
F = tt.nn.functional

# every kernel variant of the BatchNorm passes (planes, flat float4, flat scalar, single-kernel
# passes of both block sizes), each with a ragged end
SHAPES = [(4, 3, 5, 5), (16, 5, 4, 4), (8, 64, 14, 14), (5, 7, 24, 20), (64, 64, 28, 28), (96, 12, 28, 28),
          (4, 128, 7, 7), (16, 130, 9, 7), (32, 256, 14, 14), (24, 576, 14, 14), (2, 3, 1, 1)]
# n, c, h, w, k, r, pad, dil, groups of stride-1 input gradients: rows that are not whole groups of eight,
# partial tiles, shared reductions (few tiles, many channels), 64-row tiles, 1x1 in place and plain,
# a single dy pixel (spread over the kernel), 7x7 taps
CONVS = [(1, 5, 5, 5, 3, 3, 1, 1, 1), (2, 130, 9, 7, 64, 3, 1, 1, 1), (2, 512, 7, 7, 256, 3, 1, 1, 1),
         (3, 64, 14, 14, 64, 1, 0, 1, 1), (2, 257, 8, 8, 128, 1, 0, 1, 1), (16, 256, 28, 28, 64, 1, 0, 1, 1),
         (4, 48, 13, 13, 32, 3, 2, 2, 2), (3, 24, 4, 4, 100, 4, 0, 1, 1), (2, 64, 20, 20, 8, 7, 3, 1, 1)]


def _host(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


def _same_bits(a, b):
    a, b = a.get(), b.get()
    na, nb = np.isnan(a), np.isnan(b)
    np.testing.assert_array_equal(na, nb)
    np.testing.assert_array_equal(a.view(np.uint32)[~na], b.view(np.uint32)[~nb])


def _ptr(a):
    return None if a is None else a.ptr


@pytest.mark.parametrize('shape', SHAPES, ids=lambda s: 'x'.join(map(str, s)))
@pytest.mark.parametrize('affine', [True, False])
def test_batch_norm_with_residual_relu_and_accumulation(shape, affine):
    rng = np.random.default_rng(sum(shape))
    n, c = shape[:2]
    dims = (n, c, int(np.prod(shape[2:])))
    x = hiparray(0.5 + 2 * _host(rng, *shape))
    gamma, beta = (hiparray(_host(rng, c)), hiparray(_host(rng, c))) if affine else (None, None)
    res, other, dy_host = hiparray(_host(rng, *shape)), hiparray(_host(rng, *shape)), _host(rng, *shape)
    dy_host.flat[:4] = [np.inf, -np.inf, np.nan, -1.0]
    dy = hiparray(dy_host)

    def forward(residual, relu, coef):
        y, st = hiparray.empty(shape), [hiparray.empty((c,)) for _ in range(3)]
        _hip.call('tt_bn_act_fwd_train_f32', x.ptr, _ptr(gamma), _ptr(beta), _ptr(residual), y.ptr, st[0].ptr, st[1].ptr,
                  st[2].ptr, _ptr(coef), None, None, None, None, None, 0.0, 1e-5, relu, *dims)
        return y, st

    plain, _, _, _, _, _ = ops.bn_fwd_train(x, gamma, beta, None, None, 0.0, 1e-5)
    total, act = ops.add(plain, res), ops.relu_fwd(plain)
    coef = hiparray.empty((2 * c,))
    _same_bits(forward(res, 0, None)[0], total)
    _same_bits(forward(res, 1, None)[0], ops.relu_fwd(total))
    y, st = forward(None, 1, coef)
    _same_bits(y, act)

    for masked in (False, True):
        want = ops.bn_bwd(x, ops.relu_bwd(dy, act) if masked else dy, gamma, *st)
        got = ops.bn_bwd(x, dy, gamma, *st, coef=coef if masked else None, add=other)
        _same_bits(got[0], ops.add(want[0], other))
        _same_bits(got[1], want[1])
        _same_bits(got[2], want[2])


@pytest.mark.parametrize('math', ['f32', 'bf16', 'bf16x3'])
@pytest.mark.parametrize('case', CONVS, ids=lambda c: '-'.join(map(str, c)))
def test_input_gradient_with_accumulation_and_mask(case, math):
    n, c, h, w, k, r, pad, dil, groups = case
    rng = np.random.default_rng(sum(case))
    wt, other = hiparray(_host(rng, k, c // groups, r, r)), _host(rng, n, c, h, w)
    y = hiparray(_host(rng, n, c, h, w))
    p, q = (v + 2 * pad - dil * (r - 1) for v in (h, w))
    dy = hiparray(_host(rng, n, k, p, q))
    other.flat[:3] = [np.inf, -np.inf, np.nan]
    other = hiparray(other)
    geometry = ((h, w), (1, 1), (pad, pad), (dil, dil), groups)
    _hip.set_conv_math(math)
    try:
        dx = ops.conv2d_dgrad(dy, wt, None, *geometry)
        total = ops.add(other, dx)
        _same_bits(ops.conv2d_dgrad(dy, wt, None, *geometry, add=other), total)
        _same_bits(ops.conv2d_dgrad(dy, wt, None, *geometry, relu_y=y), ops.relu_bwd(dx, y))
        _same_bits(ops.conv2d_dgrad(dy, wt, None, *geometry, add=other, relu_y=y), ops.relu_bwd(total, y))
    finally:
        _hip.set_conv_math('f32')
    with pytest.raises(RuntimeError, match='stride 2 x 2'):
        ops.conv2d_dgrad(dy, wt, None, (h, w), (2, 2), (pad, pad), (dil, dil), groups, add=other)


def _blocks():
    """Post- and pre-activation residual blocks, ReLUs with one and two other consumers, and one that also
    feeds the result directly."""
    tt.manual_seed(3)
    nn = tt.nn
    convs = [nn.Conv2d(16, 16, s, padding=s // 2, bias=False) for s in (3, 1, 3, 1, 3)]
    norms = [nn.BatchNorm2d(16) for _ in range(4)]
    for m in convs + norms:
        m.cuda()

    def forward(x):
        a = F.relu(norms[0](convs[0](x)) + x)
        b = F.relu(norms[1](convs[1](a)) + a)
        c = F.relu(b + convs[2](b))
        d = convs[3](F.relu(norms[2](c))) + c
        e = F.relu(norms[3](d) + d)
        return a + (convs[4](e) + e)
    return convs + norms, forward


def test_residual_blocks_give_the_gradients_of_separate_launches(monkeypatch):
    rng = np.random.default_rng(5)
    xh, gh = _host(rng, 3, 16, 12, 12), _host(rng, 3, 16, 12, 12)

    def run():
        modules, forward = _blocks()
        x = tt.Tensor(hiparray(xh), requires_grad=True)
        y = forward(x)
        y.backward(tt.Tensor(hiparray(gh)))
        return [y.data, x.grad] + [p.grad for m in modules for p in m.parameters() if p.grad is not None] + \
            [m.running_var.data for m in modules if hasattr(m, 'running_var')]

    got = run()
    monkeypatch.setattr(grad_nn, 'take_arrived', lambda *a: None)
    monkeypatch.setattr(grad_nn, '_relu_waiting_for', lambda *a: (None, None))
    monkeypatch.setattr(ops.DeferredBatchNorm, 'run_with_relu',
                        lambda self, out=None, keep_coef=False: _separate_relu(self, out))
    want = run()
    assert len(got) == len(want) == 2 + 5 + 8 + 4
    for a, b in zip(got, want):
        _same_bits(a, b)


def _separate_relu(op, out):
    op.run()
    op.coef = None
    return ops.relu_fwd(op.out, out=op.out if out is None else out)


def test_values_between_stay_readable():
    rng = np.random.default_rng(6)
    x, s = tt.Tensor(hiparray(_host(rng, 4, 8, 6, 6))), tt.Tensor(hiparray(_host(rng, 4, 8, 6, 6)))
    bn = tt.nn.BatchNorm2d(8)
    bn.cuda()
    n = bn(x)
    t = s + n
    assert _hip.pending().__class__ is ops.DeferredBatchNorm and _hip.pending().residual is s.data
    y = F.relu(t)
    assert bn.num_batches_tracked.item() == 1.0
    plain = ops.bn_fwd_train(x.data, bn.weight.data, bn.bias.data, None, None, 0.0, 1e-5)[0]
    total = ops.add(plain, s.data)
    s.data.fill(0.0)                                    # in place: what is still to be produced comes first
    x.data.fill(0.0)
    _same_bits(n.data, plain)
    _same_bits(t.data, total)
    _same_bits(y.data, ops.relu_fwd(total))
    assert bn.num_batches_tracked.item() == 1.0


def test_errors_name_the_entry_point_that_was_called():
    dy, wt, other = hiparray.zeros((1, 6, 8, 8)), hiparray.zeros((6, 2, 3, 3)), hiparray.zeros((1, 8, 8, 8))
    for add, name in ((None, 'tt_conv2d_dgrad_f32'), (other, 'tt_conv2d_dgrad_acc_f32')):
        with pytest.raises(RuntimeError, match=f'^{name}: channels'):
            ops.conv2d_dgrad(dy, wt, None, (8, 8), (1, 1), (1, 1), (1, 1), 4, add=add)
