"""The kernels that keep a patch of the source in LDS (three bfloat16 terms), over every geometry they
take: the float32 bar of tests/test_gpu_conv.py, and sums no further from float64 ones than those of the kernels
that gather in place."""
import numpy as np
import pytest

from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray
from tests.cases import CONV_CASES, CONVT_CASES, random_conv_cases, random_convt_cases, random_large_kernel_cases
from tests.test_gpu_conv import TILE_CASES, _last_launch, _run_conv
from tests.test_gpu_conv import test_conv_transpose_forward_backward as _conv_transpose_checks

pytestmark = pytest.mark.gpu

ALWAYS, WHERE_FASTER, NEVER = 2, 1, 0


@pytest.fixture
def patch():
    def choose(which, math='bf16x3'):
        _hip.call('tt_conv2d_patch_enable', which)
        _hip.set_conv_math(math)
    yield choose
    choose(WHERE_FASTER)
    _hip.set_conv_math('f32')


# n, c, h, w, k, r, s, stride, pad, dilation, groups: one pixel; images smaller than a tile, many in it, framed by more
# zeros than the taps reach, by fewer, by none; rows wider than a tile; channels and rows on either side of 16, 32, 64,
# 128; one tap; as many as there may be; a single tile with its reduction shared
EDGES = [
    (1, 1, 1, 1, 1, 1, 1, (1, 1), (0, 0), (1, 1), 1), (70, 16, 2, 4, 32, 3, 3, (1, 1), (1, 1), (1, 1), 1),
    (300, 17, 2, 3, 33, 3, 3, (1, 1), (1, 1), (1, 1), 1), (31, 15, 5, 4, 31, 3, 3, (1, 1), (0, 0), (1, 1), 1),
    (9, 24, 7, 7, 64, 3, 3, (1, 1), (4, 3), (1, 1), 1), (3, 40, 9, 13, 65, 5, 5, (1, 1), (2, 2), (1, 1), 1),
    (5, 33, 14, 14, 128, 3, 3, (1, 1), (2, 2), (2, 2), 1), (2, 16, 28, 28, 129, 3, 2, (1, 1), (1, 0), (1, 3), 1),
    (1, 20, 3, 140, 70, 2, 3, (1, 1), (0, 1), (1, 1), 1), (2, 16, 40, 300, 32, 1, 3, (1, 1), (0, 1), (1, 1), 1),
    (4, 64, 12, 11, 96, 1, 1, (1, 1), (0, 0), (1, 1), 1), (2, 8, 12, 40, 8, 1, 31, (1, 1), (0, 15), (1, 1), 1),
    (2, 18, 16, 15, 34, 5, 6, (1, 1), (2, 2), (1, 1), 1), (1, 512, 7, 7, 64, 3, 3, (1, 1), (1, 1), (1, 1), 1),
    (40, 130, 14, 14, 200, 3, 3, (1, 1), (1, 1), (1, 1), 1), (6, 48, 61, 43, 160, 3, 3, (1, 1), (1, 1), (1, 1), 1),
]

# input gradients of two and four classes: of equal and unequal sizes and taps, one tap each, with dilation, rows of dx
# that no tap reaches
STRIDED = [
    (4, 33, 16, 16, 40, 4, 4, (2, 2), (1, 1), (1, 1), 1), (3, 20, 15, 13, 48, 3, 3, (2, 2), (1, 1), (1, 1), 1),
    (2, 64, 9, 8, 30, 2, 2, (2, 2), (0, 0), (1, 1), 1), (5, 24, 11, 20, 65, 3, 4, (1, 2), (1, 1), (1, 1), 1),
    (2, 40, 21, 17, 24, 5, 3, (2, 1), (3, 0), (1, 2), 1), (2, 36, 20, 19, 130, 3, 5, (2, 2), (0, 2), (3, 1), 1),
    (1, 200, 14, 14, 64, 3, 3, (2, 2), (1, 1), (1, 1), 1), (2, 17, 12, 31, 33, 2, 4, (1, 4), (0, 1), (1, 1), 1),
]


@pytest.mark.parametrize('case', EDGES + STRIDED + [c for c in CONV_CASES + TILE_CASES if c[10] == 1])
@pytest.mark.parametrize('bias,math', [(True, 'bf16x3'), (False, 'f32')])
def test_meets_the_float32_bar(case, bias, math, patch):
    patch(ALWAYS, math)
    _run_conv(case, seed=5, bias=bias)
    if case in EDGES + STRIDED:   # the input gradient
        assert _last_launch()['persistent_blocks'] == -4


@pytest.mark.parametrize('case', random_conv_cases(60, 91) + random_large_kernel_cases(8, 92))
def test_random_geometries(case, patch):
    patch(ALWAYS, 'f32')
    _run_conv(case, seed=6)


@pytest.mark.parametrize('case', CONVT_CASES + random_convt_cases(20, 93))
@pytest.mark.parametrize('math', ['bf16x3', 'f32'])
def test_transposed(case, math, patch):
    patch(ALWAYS, math)
    _conv_transpose_checks(case)


@pytest.mark.parametrize('c,r', [(48, 3), (32, 3), (80, 5), (16, 1)])
def test_the_workspace_holds_what_is_read_ahead(c, r, patch):
    """The product fetches weights two taps ahead and runs an odd number of taps as if it were one more: a 128-row
    layer's waves read up to three taps of 3 KB past their last.  (A size query: nothing is launched.)"""
    import ctypes
    patch(ALWAYS, 'f32')
    taps = -(-c // 16) * r * r
    size = ctypes.c_size_t()
    _hip.call('tt_workspace_size_conv2d_fwd_f32', ctypes.byref(size), 64, c, 28, 28, 128, r, r, 1, 1, r // 2, r // 2, 1, 1, 1)
    assert size.value >= 3072 * (4 * taps + 2 + taps % 2)


@pytest.mark.parametrize('dims,bf16x3,f32', [
    ((128, 128, 16, 16, 128, 3, 1), True, True),      # 256 blocks
    ((136, 128, 16, 16, 128, 3, 1), False, True),     # 272: some compute units have two to run
    ((264, 128, 16, 16, 128, 3, 1), True, True),      # 528
    ((24, 36, 7, 28, 363, 4, 2), False, False),       # 264, and below what float32 arithmetic sends here
    ((58, 96, 7, 42, 62, 5, 2), False, True)])        # 268 that share their reductions
def test_rule(dims, bf16x3, f32, patch):
    n, c, h, w, k, r, pad = dims
    x, wt = hiparray.zeros((n, c, h, w)), hiparray.zeros((k, c, r, r))
    for math, expected in (('bf16x3', bf16x3), ('f32', f32)):
        patch(WHERE_FASTER, math)
        ops.conv2d_fwd(x, wt, None, (1, 1), (pad, pad), (1, 1), 1)
        assert (_last_launch()['persistent_blocks'] == -4) == expected, math


@pytest.mark.parametrize('math', ['bf16x3', 'f32'])
@pytest.mark.parametrize('n,c,hw,k', [(9, 64, 14, 96), (2, 256, 7, 70), (40, 32, 28, 64)])   # the second shares its reduction
def test_epilogues(n, c, hw, k, math, patch):
    """The same bits as the entry points they stand in for."""
    patch(ALWAYS, math)
    rng = np.random.default_rng(3)
    x, w, res, mask = (hiparray(rng.standard_normal(s).astype(np.float32))
                       for s in ((n, c, hw, hw), (k, c, 3, 3), (n, k, hw, hw), (n, c, hw, hw)))
    mean, gamma, beta = (hiparray(rng.standard_normal(k).astype(np.float32)) for _ in range(3))
    var = hiparray(rng.random(k).astype(np.float32) + np.float32(.5))
    y = ops.conv2d_fwd(x, w, None, (1, 1), (1, 1), (1, 1), 1)
    out = hiparray.empty(y.shape)
    _hip.call('tt_conv2d_norm_act_fwd_f32', x.ptr, w.ptr, None, out.ptr, mean.ptr, var.ptr, gamma.ptr, beta.ptr, 1e-5,
              res.ptr, 1, n, c, hw, hw, k, 3, 3, 1, 1, 1, 1, 1, 1, 1)
    assert _last_launch()['persistent_blocks'] == -4
    want = np.maximum(ops.bn_fwd_eval(y, gamma, beta, mean, var, 1e-5)[0].get() + res.get(), 0)
    assert np.array_equal(out.get(), want)
    dx = ops.conv2d_dgrad(res, w, None, (hw, hw), (1, 1), (1, 1), (1, 1), 1).get()
    fused = ops.conv2d_dgrad(res, w, None, (hw, hw), (1, 1), (1, 1), (1, 1), 1, add=x, relu_y=mask).get()
    assert _last_launch()['persistent_blocks'] == -4
    assert np.array_equal(fused, (dx + x.get()) * (mask.get() > 0))


@pytest.mark.parametrize('n,c,hw,k', [(9, 64, 14, 96), (2, 256, 7, 70), (3, 17, 28, 33)])
@pytest.mark.parametrize('scale', [1.0, 2.0 ** 120, 2.0 ** -126, 2.0 ** -140])
def test_operands_the_terms_do_not_hold(n, c, hw, k, scale, patch):
    """float32 arithmetic: infinities, NaN, magnitudes that round to a bfloat16 infinity and operands whose last terms
    it cannot hold give what the other kernels give, behind an epilogue as well."""
    rng = np.random.default_rng(4)
    xh, wh = rng.standard_normal((n, c, hw, hw)).astype(np.float32), rng.standard_normal((k, c, 3, 3)).astype(np.float32)
    xh, wh = np.ldexp(xh, int(np.log2(scale))), wh / np.float32(4)
    if scale == 1.0:
        xh[0, 0, 2, 3], xh[0, 1, 2, 5], xh[1, c - 1, 0, 0], xh[1, 3, 5, 5] = np.inf, -np.inf, np.nan, np.float32(3.4e38)
        wh[5, 2, 1, 1] = -np.inf
    x, w = hiparray(xh), hiparray(wh)
    bias = hiparray(rng.standard_normal(k).astype(np.float32) * np.float32(scale))
    add = hiparray((rng.standard_normal((n, c, hw, hw)) * scale).astype(np.float32))
    dy = hiparray(np.resize(xh, (n, k, hw, hw)))
    geometry = ((1, 1), (1, 1), (1, 1), 1)

    def results():
        return (ops.conv2d_fwd(x, w, None, *geometry).get(), ops.conv2d_fwd(x, w, bias, *geometry).get(),
                ops.conv2d_dgrad(dy, w, None, (hw, hw), *geometry).get(),
                ops.conv2d_dgrad(dy, w, None, (hw, hw), *geometry, add=add, relu_y=add).get())
    patch(ALWAYS, 'f32')
    got = results()
    assert _last_launch()['persistent_blocks'] == -4
    patch(NEVER, 'f32')
    for a, b in zip(got, results()):
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(np.isinf(a), np.isinf(b))
        finite = np.isfinite(a) & np.isfinite(b)
        assert finite.mean() > .5
        size = float(np.abs(b[finite], dtype=np.float64).max())
        # float32 instructions round every product and sum to a multiple of 2^-149
        np.testing.assert_allclose(a[finite], b[finite], rtol=1e-5, atol=max(1e-6 * min(size, 1e3 * scale), 2.0 ** -150 * 9 * max(c, k)))


@pytest.mark.parametrize('dims', [(4, 64, 28, 28, 64, 3, 1), (2, 512, 7, 7, 512, 3, 1), (4, 128, 16, 16, 256, 3, 1), (3, 96, 20, 17, 48, 5, 1),
                                  (8, 64, 56, 56, 64, 3, 1), (4, 64, 32, 32, 128, 4, 2), (4, 128, 28, 28, 256, 3, 2)])
def test_sums_are_as_accurate_as_in_the_other_kernels(dims, patch):
    """Against the exact sums of both arithmetics' kernels that gather in place."""
    import torch
    n, c, h, w, k, r, stride = dims
    pad = (r - 1) // 2
    p, q = ((x + 2 * pad - r) // stride + 1 for x in (h, w))
    rng = np.random.default_rng(11)
    xh, wh = rng.standard_normal((n, c, h, w)).astype(np.float32), rng.standard_normal((k, c, r, r)).astype(np.float32)
    dyh = rng.standard_normal((n, k, p, q)).astype(np.float32)
    x64, w64 = torch.tensor(xh, dtype=torch.float64, requires_grad=True), torch.tensor(wh, dtype=torch.float64)
    y64 = torch.nn.functional.conv2d(x64, w64, padding=pad, stride=stride)
    y64.backward(torch.tensor(dyh, dtype=torch.float64))
    want = {'y': y64.detach().numpy(), 'dx': x64.grad.numpy()}
    x, wt, dy = hiparray(xh), hiparray(wh), hiparray(dyh)
    geometry = ((stride, stride), (pad, pad), (1, 1), 1)

    def errors():
        got = {'y': ops.conv2d_fwd(x, wt, None, *geometry).get(), 'dx': ops.conv2d_dgrad(dy, wt, None, (h, w), *geometry).get()}
        return {key: np.linalg.norm(got[key] - want[key]) / np.linalg.norm(want[key]) for key in got}
    patch(ALWAYS)
    new = errors()
    patch(NEVER)
    old = errors()
    patch(NEVER, 'f32')
    f32 = errors()
    for key in want:
        print(dims, key, 'patch %.2e, gathered %.2e, float32 %.2e' % (new[key], old[key], f32[key]))
        assert new[key] <= old[key] and new[key] <= f32[key], key
