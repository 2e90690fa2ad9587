"""The kernels for few rows (vector unit), over every geometry they take, and the matrix kernels on the small
cases that these take over from them."""
import ctypes

import numpy as np
import pytest

import oracle
from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray
from tests.brute import bf16_round
from tests.cases import CONV_CASES, CONVT_CASES, random_conv_cases, random_convt_cases, random_large_kernel_cases
from tests.test_gpu_conv import TILE_CASES, _check, _last_launch, _run_conv
from tests.test_gpu_conv_bf16 import _forward_and_input_gradient

pytestmark = pytest.mark.gpu

ALWAYS, WHERE_FASTER, NEVER = 2, 1, 0


@pytest.fixture
def narrow():
    def choose(which):
        _hip.call('tt_conv2d_narrow_enable', which)
    yield choose
    choose(WHERE_FASTER)


# rows of 1, 4 | 5, 8 | 9, 16; channels on either side of four; runs of channels that end inside a fetch and a stage of 128
# steps; more taps than a mask has bits; nine classes, some without a tap; many pixels per thread, ragged
EDGES = [
    (2, 1, 9, 11, 1, 3, 3, (1, 1), (1, 1), (1, 1), 1), (2, 3, 9, 11, 4, 3, 3, (1, 1), (1, 1), (1, 1), 1),
    (2, 4, 9, 11, 5, 3, 3, (2, 1), (1, 0), (1, 1), 1), (1, 5, 12, 7, 8, 5, 5, (1, 1), (2, 2), (1, 2), 1),
    (3, 43, 6, 5, 9, 3, 3, (1, 1), (1, 1), (1, 1), 1), (1, 129, 5, 5, 16, 1, 1, (1, 1), (0, 0), (1, 1), 1),
    (1, 130, 4, 6, 16, 3, 3, (1, 1), (1, 1), (1, 1), 1), (2, 3, 19, 23, 3, 13, 11, (1, 1), (6, 5), (1, 1), 1),
    (2, 6, 20, 17, 6, 2, 2, (3, 3), (0, 1), (1, 1), 3), (2, 16, 10, 12, 16, 3, 3, (2, 2), (1, 1), (1, 1), 16),
    (9, 8, 131, 127, 8, 3, 3, (1, 1), (1, 1), (1, 1), 8), (5, 4, 263, 201, 16, 1, 1, (1, 1), (0, 0), (1, 1), 1),
    (1, 5, 259, 257, 96, 1, 1, (1, 1), (0, 0), (1, 1), 1), (70, 2, 2, 3, 5, 1, 3, (1, 1), (0, 1), (1, 1), 1),
]


@pytest.mark.parametrize('case', EDGES + [c for c in CONV_CASES if c[4] // c[10] <= 16])
@pytest.mark.parametrize('bias', [True, False])
def test_meets_the_float32_bar(case, bias, narrow):
    narrow(ALWAYS)
    _run_conv(case, seed=5, bias=bias)
    # (an input gradient that spreads one pixel over the whole kernel is a matrix product of C*R*S rows)
    assert _last_launch()['persistent_blocks'] == -3 or case[1] // case[10] > 16 or case[2:4] == case[5:7]


@pytest.mark.parametrize('case', random_conv_cases(60, 77) + random_large_kernel_cases(8, 78))
def test_random_geometries(case, narrow):
    narrow(ALWAYS)
    _run_conv(case, seed=6)


@pytest.mark.parametrize('case', EDGES[:11] + random_conv_cases(20, 79))
def test_bf16_operands(case, narrow):
    narrow(ALWAYS)
    _hip.set_conv_math('bf16')
    try:
        _forward_and_input_gradient(case)
    finally:
        _hip.set_conv_math('f32')


@pytest.mark.parametrize('case', CONVT_CASES + random_convt_cases(20, 80))
def test_transposed(case, narrow):
    narrow(ALWAYS)
    n, ci, h, w_, co, r, s, st, pd, op, dl, g = case
    rng = np.random.default_rng(7)
    x = rng.standard_normal((n, ci, h, w_)).astype(np.float32)
    w = (rng.standard_normal((ci, co // g, r, s)) / np.sqrt(ci // g * r * s)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    y32 = oracle.transposed_convolution_forward(x, w, b, st, pd, op, dl, g)
    y64 = oracle.transposed_convolution_forward(*(a.astype(np.float64) for a in (x, w, b)), st, pd, op, dl, g)
    y = ops.conv2d_dgrad(hiparray(x), hiparray(w), hiparray(b), y32.shape[-2:], st, pd, dl, g).get()
    _check('y', y, y32, y64)


@pytest.mark.parametrize('case', [c for c in CONV_CASES + TILE_CASES if min(c[1], c[4]) // c[10] <= 16])
def test_matrix_kernels_on_the_cases_taken_over(case, narrow):
    narrow(NEVER)
    _hip.call('tt_set_conv_dense_cell_min_tiles', 0 if case[7] != (1, 1) else -1)
    try:
        _run_conv(case, seed=8)
    finally:
        _hip.call('tt_set_conv_dense_cell_min_tiles', -1)
    assert _last_launch()['persistent_blocks'] != -3


@pytest.mark.parametrize('dims,forward,gradient,weights', [
    ((128, 4, 64, 64, 16, 3, 2, 1, 3, 2, 3, 1, 2, 2), True, True, True),        # the notebook's groups
    ((32, 32, 56, 56, 32, 3, 3, 1, 1, 1, 1, 1, 1, 32), True, True, True),       # depthwise
    ((8, 64, 28, 28, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), False, False, True),        # a long chain on few pixels
    ((8, 3, 64, 64, 64, 7, 7, 2, 2, 3, 3, 1, 1, 1), False, False, False),       # 49 taps, 1024 steps
    ((4, 64, 28, 28, 64, 1, 1, 1, 1, 0, 0, 1, 1, 1), False, False, False),
    ((64, 3, 224, 224, 64, 7, 7, 2, 2, 3, 3, 1, 1, 1), False, False, False),    # the same on many pixels: 1.3e10 products
    ((128, 3, 64, 64, 64, 4, 4, 2, 2, 1, 1, 1, 1, 1), False, True, False),      # 5.4e8
    ((13, 4, 15, 141, 2, 4, 4, 2, 2, 2, 2, 1, 1, 1), False, True, False)])      # four chunks: weights read in place
def test_rule(dims, forward, gradient, weights):
    n, c, h, w, k, r, s, sh, sw, ph, pw, dh, dw, g = dims
    p, q = (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1
    x, dy, wt = hiparray.zeros((n, c, h, w)), hiparray.zeros((n, k, p, q)), hiparray.zeros((k, c // g, r, s))
    geometry = ((sh, sw), (ph, pw), (dh, dw), g)
    ops.conv2d_fwd(x, wt, None, *geometry)
    assert (_last_launch()['persistent_blocks'] == -3) == forward
    ops.conv2d_dgrad(dy, wt, None, (h, w), *geometry)
    assert (_last_launch()['persistent_blocks'] == -3) == gradient
    ops.conv2d_wgrad(x, dy, wt.shape, *geometry)
    plan = (ctypes.c_int * 4)()
    _hip.call('tt_conv2d_last_wgrad_launch', plan)
    assert (plan[2] == -3) == weights


@pytest.mark.parametrize('dims,f32,bf16', [
    ((2, 4, 32, 16, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, True),         # 36 columns, 1024 pixels: one launch
    ((2, 4, 33, 16, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), False, False),       # 1056
    ((2, 8, 33, 16, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, True),         # 72 columns
    ((8, 4, 32, 32, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, False),        # 8192
    ((16, 4, 32, 32, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, True),        # 16384
    ((1, 4, 8, 16, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), False, False),        # 128
    ((1, 4, 8, 17, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, True),
    ((33, 33, 32, 32, 9, 1, 1, 1, 1, 0, 0, 1, 1, 1), True, False),      # nine rows, 33 columns, 33792
    ((33, 32, 32, 32, 9, 1, 1, 1, 1, 0, 0, 1, 1, 1), True, True),
    ((8, 114, 32, 32, 5, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, False),      # five rows, 1026 columns
    ((8, 114, 32, 32, 4, 3, 3, 1, 1, 1, 1, 1, 1, 1), True, True)])
def test_rule_of_the_weight_gradient(dims, f32, bf16):
    import torch
    n, c, h, w, k, r, s, sh, sw, ph, pw, dh, dw, g = dims
    p, q = (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1
    rng = np.random.default_rng(2)
    x, dy = (rng.standard_normal(a).astype(np.float32) for a in ((n, c, h, w), (n, k, p, q)))
    plan = (ctypes.c_int * 4)()
    try:
        for math, narrow_ones in (('f32', f32), ('bf16', bf16)):
            _hip.set_conv_math(math)
            got = ops.conv2d_wgrad(hiparray(x), hiparray(dy), (k, c // g, r, s), (sh, sw), (ph, pw), (dh, dw), g).get()
            _hip.call('tt_conv2d_last_wgrad_launch', plan)
            assert (plan[2] == -3) == narrow_ones
            a, b = (torch.tensor(v if math == 'f32' else bf16_round(v), dtype=torch.float64) for v in (x, dy))

            def sums(a, b):
                return torch.nn.grad.conv2d_weight(a, (k, c // g, r, s), b, (sh, sw), (ph, pw), (dh, dw), g).numpy()
            # a sum of m rounded products is off by about sqrt(m) roundings of its magnitudes' sum, in whatever order
            assert (np.abs(got - sums(a, b)) <= 2.0 ** -24 * (n * p * q) ** .5 * sums(a.abs(), b.abs())).all()
    finally:
        _hip.set_conv_math('f32')
