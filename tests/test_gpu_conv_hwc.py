"""The channel-last convolution kernels (bf16 arithmetic) at the sizes where they can go wrong: channels and rows that fill no chunk or tile, images smaller than a tile, split reductions
of even and ragged share, reversed taps with more padding than the kernel reaches, 2 and 31 taps."""
import ctypes

import numpy as np
import pytest

import oracle
from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray
from tests.brute import bf16_round
from tests.test_gpu_conv_bf16 import _forward_and_input_gradient

pytestmark = pytest.mark.gpu

# n, c, h, w, k, r, s, stride, pad, dilation, groups
CASES = [(1, 3, 6, 5, 5, 3, 3, (1, 1), (1, 1), (1, 1), 1),        # one chunk mostly padding, one ragged tile
         (2, 64, 9, 7, 64, 3, 3, (1, 1), (1, 1), (1, 1), 1),      # whole chunks, 64-row tiles
         (2, 65, 9, 7, 65, 3, 3, (1, 1), (1, 1), (1, 1), 1),      # one past them
         (2, 160, 9, 7, 190, 3, 3, (1, 1), (1, 1), (1, 1), 1),    # 64-row tiles where 128 pad more
         (3, 130, 7, 7, 40, 1, 1, (1, 1), (0, 0), (1, 1), 1),     # one tap, pixels no multiple of four
         (9, 16, 4, 4, 130, 3, 3, (1, 1), (1, 1), (1, 1), 1),     # eight images in a tile
         (3, 512, 5, 5, 96, 3, 3, (1, 1), (1, 1), (1, 1), 1),     # split reduction, ragged last share
         (2, 256, 8, 8, 256, 3, 3, (2, 2), (1, 1), (1, 1), 1),    # stride 2 (forward), split
         (2, 40, 13, 11, 72, 1, 2, (1, 1), (0, 1), (1, 1), 1),    # two taps
         (1, 33, 40, 9, 31, 31, 1, (1, 1), (15, 0), (1, 1), 1),   # 31 taps
         (2, 48, 12, 10, 80, 5, 3, (1, 1), (4, 2), (2, 1), 1),    # dilation
         (2, 32, 6, 6, 32, 2, 2, (1, 1), (1, 1), (1, 1), 1),      # more rows out than in
         (2, 32, 8, 8, 48, 3, 3, (1, 3), (0, 0), (1, 1), 1),      # unequal strides
         (5, 128, 16, 16, 128, 3, 3, (1, 1), (1, 1), (1, 1), 1)]


CHANNEL_LAST = -2       # what the launch plan says of these kernels (-1: the bf16-first ones)


def _plan():
    plan = (ctypes.c_int * 8)()
    _hip.call('tt_conv2d_last_launch', plan)
    return plan


@pytest.fixture
def math():
    """Every launch the kernels support is sent to them, whatever its size."""
    _hip.set_conv_math('bf16')
    _hip.call('tt_conv2d_bf16_first_enable', 3)
    try:
        yield
    finally:
        _hip.call('tt_conv2d_bf16_first_enable', 1)
        _hip.set_conv_math('f32')


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(map(str, c[:7])))
def test_forward_and_input_gradient(case, math):
    _forward_and_input_gradient(case)
    n, c, h, w, k, r, s, st, pd, dl, g = case
    rng = np.random.default_rng(2)
    x, wt = (hiparray(rng.standard_normal(v).astype(np.float32)) for v in ((n, c, h, w), (k, c, r, s)))
    y = ops.conv2d_fwd(x, wt, None, st, pd, dl, g)
    assert _plan()[4] == CHANNEL_LAST and _plan()[7] >> 8 == 1
    # the same product in the kernels that gather in place: another order of summation
    dx = ops.conv2d_dgrad(y, wt, None, (h, w), st, pd, dl, g)
    assert (_plan()[4] == CHANNEL_LAST) == (st == (1, 1))
    _hip.call('tt_conv2d_bf16_first_enable', 0)
    for got, other in ((y, ops.conv2d_fwd(x, wt, None, st, pd, dl, g)), (dx, ops.conv2d_dgrad(y, wt, None, (h, w), st, pd, dl, g))):
        assert _plan()[4] >= 0
        np.testing.assert_allclose(got.get(), other.get(), rtol=1e-4, atol=1e-5 * float(np.abs(other.get()).max()))


@pytest.mark.parametrize('split', [False, True])
def test_values_next_to_the_image_are_not_touched(split, math):
    """Non-finite values in the images before and after one: nothing of theirs reaches it, and its own reach
    exactly the outputs whose window covers them."""
    n, c, h, k = 3, 256 if split else 16, 6, 40
    rng = np.random.default_rng(4)
    x = rng.standard_normal((n, c, h, h)).astype(np.float32)
    wt = hiparray(rng.standard_normal((k, c, 3, 3)).astype(np.float32))
    clean = ops.conv2d_fwd(hiparray(x), wt, None, (1, 1), (1, 1), (1, 1), 1).get()
    x[0], x[2] = np.nan, np.inf
    x[1, 5, 0, 0] = np.nan
    y = ops.conv2d_fwd(hiparray(x), wt, None, (1, 1), (1, 1), (1, 1), 1).get()
    assert _plan()[4] == CHANNEL_LAST
    hit = np.zeros((h, h), bool)
    hit[:2, :2] = True
    assert np.isnan(y[1][:, hit]).all()
    np.testing.assert_array_equal(y[1][:, ~hit], clean[1][:, ~hit])


@pytest.mark.parametrize('dims,taken', [((8, 64, 14, 14, 64, 3, 3), False),        # little work
                                        ((16, 64, 56, 56, 64, 3, 3), False),       # few channels, tiles enough
                                        ((64, 128, 28, 28, 128, 3, 3), True),      # the same with more channels
                                        ((16, 256, 14, 14, 256, 3, 3), True),      # few tiles, long reduction
                                        ((16, 160, 45, 37, 192, 3, 3), False),     # padded channels
                                        ((16, 2048, 7, 7, 512, 1, 1), True),       # 1x1 on 49 pixels
                                        ((16, 512, 8, 8, 2048, 1, 1), False)])     # plain matrix product
def test_size_rule_and_workspace(dims, taken, math):
    """Which calls go there by default; the workspace query says what a call asks for."""
    _hip.call('tt_conv2d_bf16_first_enable', 1)
    n, c, h, w, k, r, s = dims
    geometry = (1, 1, r // 2, s // 2, 1, 1, 1)
    x, wt = hiparray.zeros((n, c, h, w)), hiparray.zeros((k, c, r, s))
    ops.conv2d_fwd(x, wt, None, (1, 1), (r // 2, s // 2), (1, 1), 1)
    nbytes = ctypes.c_size_t()
    _hip.call('tt_workspace_size_conv2d_fwd_f32', ctypes.byref(nbytes), *dims, *geometry)
    assert (_plan()[4] == CHANNEL_LAST) == taken
    # the layouts of x and of the weights, with the channels padded to 64 and the rows to whole tiles; the others
    # ask for repacked weights and for every sharing block's partial tile
    padded = -(-c // 64) * 64
    layouts = 2 * (n * h * w + -(-k // _plan()[0]) * _plan()[0] * r * s) * padded
    partials = 3 * _hip.device_info()['compute_units'] * 128 * 128 * 4
    if taken:
        assert _plan()[:2] == [128, 128]
        splits = (nbytes.value - layouts) // (4 * n * k * h * w)
        assert splits in (0, 2, 3, 4, 5, 6, 7, 8) and 0 <= nbytes.value - layouts - 4 * splits * n * k * h * w < 3 * 256
    else:
        assert nbytes.value >= partials and nbytes.value - partials < 8 * (k + 128) * (c + 64) * r * s


@pytest.mark.parametrize('dims', [(8, 128, 28, 28, 128, 3, 3), (3, 372, 25, 9, 137, 3, 3), (2, 1024, 7, 7, 64, 1, 1)])
def test_sums_are_as_accurate_as_in_the_other_kernels(dims, math):
    """Against float64 sums of the rounded operands, the root mean square error is no larger than that of the
    kernels that gather in place (5 % for what one draw of the values can differ by), forward and backward."""
    n, c, h, w, k, r, s = dims
    rng = np.random.default_rng(12)
    x, wt = (rng.standard_normal(v).astype(np.float32) for v in ((n, c, h, w), (k, c, r, s)))
    pad = (r // 2, s // 2)
    gy = rng.standard_normal((n, k, h, w)).astype(np.float32)
    xr, wr, gyr = (bf16_round(a).astype(np.float64) for a in (x, wt, gy))
    want = (oracle.convolution_forward(xr, wr, None, (1, 1), pad, (1, 1), 1)[0],
            oracle.conv2d_backward_x(gyr, wr, (1, 1), pad, (1, 1), 1, x_hw=(h, w)))
    xd, wd, gyd = hiparray(x), hiparray(wt), hiparray(gy)

    def errors():
        got = (ops.conv2d_fwd(xd, wd, None, (1, 1), pad, (1, 1), 1), ops.conv2d_dgrad(gyd, wd, None, (h, w), (1, 1), pad, (1, 1), 1))
        return [np.sqrt(np.mean((a.get() - b) ** 2)) for a, b in zip(got, want)]

    here = errors()
    assert _plan()[4] == CHANNEL_LAST
    _hip.call('tt_conv2d_bf16_first_enable', 0)
    there = errors()
    assert _plan()[4] >= 0
    assert all(a <= 1.05 * b for a, b in zip(here, there)), (here, there)


def _same_bits(a, b):
    a, b = a.get(), b.get()
    nan = np.isnan(a)
    np.testing.assert_array_equal(nan, np.isnan(b))
    np.testing.assert_array_equal(a.view(np.uint32)[~nan], b.view(np.uint32)[~nan])


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(map(str, c[:7])))
def test_what_follows_in_an_evaluation_pass(case, math):
    """BatchNorm, residual and ReLU applied to the accumulators, or to the split reduction's sums: the bits of the
    launches they stand in for, with non-finite values in the residual."""
    n, c, h, w, k, r, s, st, pd, dl, g = case
    rng = np.random.default_rng(3)
    x, wt = (hiparray(rng.standard_normal(v).astype(np.float32)) for v in ((n, c, h, w), (k, c, r, s)))
    bias, gamma, beta, mean = (hiparray(rng.standard_normal(k).astype(np.float32)) for _ in range(4))
    var = hiparray(rng.uniform(0.1, 2, k).astype(np.float32))
    geometry = (st, pd, dl, g)
    for b in (None, bias):
        y = ops.conv2d_fwd(x, wt, b, *geometry)
        res = rng.standard_normal(y.shape).astype(np.float32)
        res.flat[:4] = [np.inf, -np.inf, np.nan, -0.0]
        res = hiparray(res)
        bn = ops.bn_fwd_eval(y, gamma, beta, mean, var, 1e-5)[0]
        plain = ops.bn_fwd_eval(y, None, None, mean, var, 1e-5)[0]
        for norm, add, relu in ((1, 0, 0), (1, 0, 1), (1, 1, 1), (0, 1, 0), (0, 0, 1), (2, 1, 0)):
            want = {0: y, 1: bn, 2: plain}[norm]
            want = ops.add(want, res) if add else want
            want = ops.relu_fwd(want) if relu else want
            op = ops.DeferredConv(x, wt, b, *ops._conv2d_geometry(x, wt, b, *geometry))
            if norm:
                op.absorb_norm(mean, var, gamma if norm == 1 else None, beta if norm == 1 else None, 1e-5)
            if add:
                op.absorb_add(res)
            if relu:
                op.run_with_relu(hiparray.lazy(y.shape))
            _hip.flush()
            assert _plan()[4] == CHANNEL_LAST
            _same_bits(op.out, want)


@pytest.mark.parametrize('case', [c for c in CASES if c[7] == (1, 1)], ids=lambda c: '-'.join(map(str, c[:7])))
def test_accumulation_and_mask_in_the_input_gradient(case, math):
    n, c, h, w, k, r, s, st, pd, dl, g = case
    rng = np.random.default_rng(6)
    p, q = h + 2 * pd[0] - dl[0] * (r - 1), w + 2 * pd[1] - dl[1] * (s - 1)
    dy, wt, y, other = (rng.standard_normal(v).astype(np.float32) for v in ((n, k, p, q), (k, c, r, s), (n, c, h, w), (n, c, h, w)))
    other.flat[:3] = [np.inf, -np.inf, np.nan]
    dy, wt, y, other = (hiparray(a) for a in (dy, wt, y, other))
    geometry = ((h, w), st, pd, dl, g)
    dx = ops.conv2d_dgrad(dy, wt, None, *geometry)
    total = ops.add(other, dx)
    for add, relu_y, want in ((other, None, total), (None, y, ops.relu_bwd(dx, y)), (other, y, ops.relu_bwd(total, y))):
        _same_bits(ops.conv2d_dgrad(dy, wt, None, *geometry, add=add, relu_y=relu_y), want)
        assert _plan()[4] == CHANNEL_LAST


@pytest.mark.parametrize('c,taken', [(65535 * 64, True), (65535 * 64 + 1, False)])
def test_more_channels_than_a_grid_has_rows(c, taken, math):
    """The layout pass has a row of blocks for every 64 channels.  (Only the plan is asked, through the workspace.)"""
    _hip.call('tt_conv2d_bf16_first_enable', 1)
    nbytes = ctypes.c_size_t()
    _hip.call('tt_workspace_size_conv2d_fwd_f32', ctypes.byref(nbytes), 2, c, 1, 1, 64, 1, 1, 1, 1, 0, 0, 1, 1, 1)
    padded = -(-c // 64) * 64
    assert (nbytes.value - 2 * (2 + 64) * padded < 8 * 4 * 64 * 2 + 3 * 256) == taken
