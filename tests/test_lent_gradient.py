"""The gradient that ``backward`` is given is read in place: what a node keeps or writes of it must be a copy,
and what its owner does with it afterwards must not be seen."""
import numpy as np
import pytest

import pytortto_amd as tt
from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray

from .test_parked_operations import library  # noqa: F401  (a recording stand-in for the device library)

F = tt.nn.functional


def _device(*shape):
    return hiparray(np.ones(shape, np.float32))


def test_a_loan_costs_nothing_until_somebody_writes(library):  # noqa: F811
    g = _device(3, 4)
    block = g.ptr
    first, second = g.lent(), g.lent()
    assert first.ptr == block and second.ptr == block and library.launched() == []
    second.fill(2.0)                                    # the holder writes: its own copy
    assert library.launched() == ['tt_memcpy_d2d', 'tt_fill_f32']
    g.fill(3.0)                                         # the owner writes: whoever still holds a loan copies first
    assert g.ptr == block and library.launched() == ['tt_memcpy_d2d', 'tt_fill_f32']
    g.fill(3.0)                                         # ... once
    third = g.lent()
    del third
    g.fill(4.0)                                         # nobody holds one any more
    assert library.launched() == ['tt_fill_f32'] * 2


@pytest.fixture
def memory(library, monkeypatch):  # noqa: F811
    """Replays what the library is asked to do: {block: name of the values it holds} and, by kernel, the values
    of the blocks that it was given when it was launched (None: nobody has written them)."""
    holds, seen = {}, {}
    original = _hip.call
    blocks = iter(range(1 << 20, 1 << 30, 1 << 12))

    def call(name, *args):
        if _hip._pending is not None:
            _hip.flush()
        if name == 'tt_malloc':
            args[0]._obj.value = next(blocks)
        elif name == 'tt_memcpy_d2d':
            holds[args[0]] = holds.get(args[1])
        elif name == 'tt_memcpy_h2d':
            holds[args[0]] = 'host'
        else:
            original(name, *args)
            seen.setdefault(name, []).append([holds.get(a) for a in args if isinstance(a, int) and a >= 1 << 20])
            if name == 'tt_fill_f32':
                holds[args[0]] = 'filled'
    monkeypatch.setattr(_hip, 'call', call)
    yield holds, seen
    _hip.flush()


def test_a_parked_operation_that_reads_a_loan_sees_its_values_when_the_owner_writes(memory):
    holds, seen = memory
    g, y = _device(3, 4), _device(3, 4)
    holds[g.ptr] = 'gradient'
    loan = g.lent()
    dx = ops.relu_bwd_deferred(loan, y, None)
    assert 'tt_relu_bwd_f32' not in seen                    # parked
    g.fill(7.0)
    assert seen['tt_relu_bwd_f32'][0][0] == 'gradient'      # dy: the owner's block, or one that holds its values
    assert holds[g.ptr] == 'filled' and holds[loan.ptr] == 'gradient' and dx.ptr != loan.ptr


def test_a_block_is_not_published_before_it_holds_the_values(memory, monkeypatch):
    holds, seen = memory
    g = _device(3, 4)
    holds[g.ptr] = 'gradient'
    loan, source, replay = g.lent(), g.ptr, _hip.call

    def call(name, *args):
        if name == 'tt_memcpy_d2d':                         # what another thread would find at this moment
            assert loan.ptr == source
        replay(name, *args)
    monkeypatch.setattr(_hip, 'call', call)
    g.fill(7.0)
    assert loan.ptr != source and holds[loan.ptr] == 'gradient'


def test_the_gradient_of_an_earlier_pass_lent_to_a_graph_that_adds_to_it(memory):
    """``z.grad`` is given to backward and added to by it while the ReLU's backward that reads it is still parked."""
    holds, seen = memory
    bn = tt.nn.BatchNorm2d(4)
    bn.cuda()
    x, z = (tt.Tensor(_device(2, 4, 3, 3), requires_grad=True) for _ in range(2))
    z.grad = _device(2, 4, 3, 3)
    holds[z.grad.ptr] = 'gradient'
    b = bn(x)
    r = F.relu(b)
    ((x + b) + (z + r)).backward(tt.Tensor(z.grad, copy=False))
    _hip.flush()
    dy = [call[1] if name == 'tt_bn_act_bwd_f32' else call[0]
          for name in ('tt_relu_bwd_f32', 'tt_bn_act_bwd_f32') for call in seen.get(name, ())]
    assert dy and 'gradient' in dy
    for call in seen.get('tt_relu_bwd_f32', ()):
        assert call[0] == 'gradient'


@pytest.mark.gpu
def test_backward_gives_what_a_copied_gradient_gives():
    rng = np.random.default_rng(3)
    shape = (4, 6, 10, 12)
    x0, g0 = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))

    def leaf():
        x = tt.Tensor(hiparray(x0))
        x.requires_grad = True
        return x
    # a leaf keeps what it is handed: views and sums of the gradient itself, and a function that scales it in place
    for name, f, slope in (('view', lambda x: x.view(4, 6, 120).view(*shape), None), ('add', lambda x: x + x, None),
                           ('leaky', lambda x: F.leaky_relu(x, 0.25), 0.25)):
        x, g = leaf(), tt.Tensor(hiparray(g0))
        f(x).backward(g)
        want = g0 * np.where(x0 < 0, np.float32(slope), np.float32(1)) if slope else g0 * (2 if name == 'add' else 1)
        np.testing.assert_array_equal(g.data.get(), g0, err_msg=name)
        np.testing.assert_array_equal(x.grad.get(), want, err_msg=name)
        g.data.fill(7.0)                                # the owner's next step
        np.testing.assert_array_equal(x.grad.get(), want, err_msg=name)
    # the gradient of an earlier pass as the next one's: it is added to while it is still being read
    x = leaf()
    (x + x).backward(tt.Tensor(hiparray(g0)))
    (x + F.leaky_relu(x, 0.25)).backward(tt.Tensor(x.grad))
    scale = np.where(x0 < 0, np.float32(1.25), np.float32(2))
    np.testing.assert_allclose(x.grad.get(), 2 * g0 + 2 * g0 * scale, rtol=1e-6, atol=0)
