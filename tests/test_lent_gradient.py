"""The gradient that ``backward`` is given is read in place: what a node keeps or writes of it must be a copy,
and what its owner does with it afterwards must not be seen."""
import numpy as np
import pytest

import pytortto_amd as tt
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
