"""Float32 launches of the kernels that gather in place on three exact bf16 terms: every addressing mode, tile and way
of storing, the float32 bar of tests/test_gpu_conv.py, sums no further from float64 ones than those of the float32
instructions, and operands that the terms do not hold."""
import numpy as np
import pytest

from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray
from tests.cases import CONV_CASES, random_conv_cases
from tests.test_gpu_conv import TILE_CASES, _last_launch, _run_conv
from tests.test_gpu_conv_patch import EDGES as PATCH_EDGES, STRIDED

pytestmark = pytest.mark.gpu

ALWAYS, WHERE_FASTER, NEVER = 2, 1, 0


@pytest.fixture
def terms():
    def choose(which):
        _hip.call('tt_conv2d_f32_terms_enable', which)
        _hip.call('tt_conv2d_patch_enable', which if which == WHERE_FASTER else NEVER)
        _hip.call('tt_conv2d_narrow_enable', which if which == WHERE_FASTER else NEVER)
    yield choose
    choose(WHERE_FASTER)


def in_terms():
    return _last_launch()['mode'] >> 8 == 3


# n, c, h, w, k, r, s, stride, pad, dilation, groups: whole matrix products; pixels in no whole quads; channels in no
# whole chunks; rows and pixels around a tile's edge; a shared reduction; strided with cells, without; masks of 31, 49
# and more taps; one pixel
EDGES = [
    (4, 64, 12, 12, 96, 1, 1, (1, 1), (0, 0), (1, 1), 1), (3, 48, 7, 7, 129, 1, 1, (1, 1), (0, 0), (1, 1), 1),
    (5, 33, 9, 11, 65, 1, 1, (1, 1), (0, 0), (1, 1), 1), (2, 2048, 7, 7, 64, 1, 1, (1, 1), (0, 0), (1, 1), 1),
    (2, 32, 14, 12, 40, 1, 1, (2, 2), (0, 0), (1, 1), 1), (3, 32, 15, 13, 130, 1, 1, (2, 2), (0, 0), (1, 1), 1),
    (1, 16, 9, 9, 70, 1, 1, (1, 3), (1, 1), (1, 1), 1), (2, 17, 15, 14, 72, 3, 3, (2, 2), (1, 1), (1, 1), 1),
    (2, 3, 30, 30, 64, 7, 7, (2, 2), (3, 3), (1, 1), 1), (1, 5, 20, 20, 66, 9, 8, (1, 1), (4, 4), (1, 1), 1),
    (3, 96, 28, 28, 127, 3, 3, (1, 1), (1, 1), (1, 1), 1), (1, 1, 1, 1, 1, 1, 1, (1, 1), (0, 0), (1, 1), 1),
    (64, 8, 8, 8, 32, 3, 3, (1, 1), (2, 2), (2, 2), 1),
]


@pytest.mark.parametrize('case', EDGES + [c for c in CONV_CASES + TILE_CASES if c[10] == 1] + random_conv_cases(40, 17))
def test_meets_the_float32_bar(case, terms):
    terms(ALWAYS)
    _run_conv(case, seed=5, bias=case in EDGES[::2])


def _arrays(n, c, hw, k, r, stride, rng):
    p = (hw + 2 * (r // 2) - r) // stride + 1
    return (rng.standard_normal(s).astype(np.float32) for s in ((n, c, hw, hw), (k, c, r, r), (n, k, p, p)))


GEOMETRIES = [(9, 64, 14, 96, 1, 1), (2, 512, 7, 70, 1, 1), (8, 256, 28, 256, 1, 1), (3, 64, 28, 128, 1, 2), (3, 17, 28, 33, 3, 2),
              (4, 48, 28, 130, 3, 1)]


@pytest.mark.parametrize('dims', GEOMETRIES)
def test_sums_are_as_accurate_as_in_float32_instructions(dims, terms):
    import torch
    n, c, hw, k, r, stride = dims
    xh, wh, dyh = _arrays(*dims, np.random.default_rng(11))
    x64, w64 = torch.tensor(xh, dtype=torch.float64, requires_grad=True), torch.tensor(wh, dtype=torch.float64)
    y64 = torch.nn.functional.conv2d(x64, w64, padding=r // 2, stride=stride)
    y64.backward(torch.tensor(dyh, dtype=torch.float64))
    x, w, dy = hiparray(xh), hiparray(wh), hiparray(dyh)
    geometry = ((stride, stride), (r // 2, r // 2), (1, 1), 1)
    one_launch = stride == 1 or r == 1   # the classes of other strided gradients share a grid of float32 instructions

    def errors(expected):
        y = ops.conv2d_fwd(x, w, None, *geometry)
        assert in_terms() == expected
        dx = ops.conv2d_dgrad(dy, w, None, (hw, hw), *geometry)
        assert in_terms() == (expected and one_launch)
        return [np.linalg.norm(a.get() - b) / np.linalg.norm(b) for a, b in ((y, y64.detach().numpy()), (dx, x64.grad.numpy()))]
    terms(ALWAYS)
    new = errors(True)
    terms(NEVER)
    old = errors(False)
    print(dims, new, old)
    assert new[0] <= old[0] and new[1] <= old[1]


@pytest.mark.parametrize('dims', GEOMETRIES[:2] + GEOMETRIES[3:])
@pytest.mark.parametrize('scale', [1.0, 2.0 ** 120, 2.0 ** -126, 2.0 ** -140])
def test_operands_the_terms_do_not_hold(dims, scale, terms):
    """Infinities, NaN, magnitudes that round to a bfloat16 infinity and operands whose last terms it cannot hold give
    what the float32 instructions give, behind an epilogue as well."""
    n, c, hw, k, r, stride = dims
    rng = np.random.default_rng(4)
    xh, wh, dyh = _arrays(*dims, rng)
    xh, dyh, wh = np.ldexp(xh, int(np.log2(scale))), np.ldexp(dyh, int(np.log2(scale))), wh / np.float32(4)
    if scale == 1.0:
        for a in (xh, dyh):
            a[0, 0, 2, 2], a[0, 1, 2, 4], a[1, -1, 0, 0], a[1, 3, 4, 4] = np.inf, -np.inf, np.nan, np.float32(3.4e38)
        wh[5, 2, 0, 0] = -np.inf
    x, w, dy = hiparray(xh), hiparray(wh), hiparray(dyh)
    bias = hiparray(rng.standard_normal(k).astype(np.float32) * np.float32(scale))
    add = hiparray((rng.standard_normal((n, c, hw, hw)) * scale).astype(np.float32))
    geometry = ((stride, stride), (r // 2, r // 2), (1, 1), 1)

    def results():
        out = [ops.conv2d_fwd(x, w, None, *geometry).get(), ops.conv2d_fwd(x, w, bias, *geometry).get(),
               ops.conv2d_dgrad(dy, w, None, (hw, hw), *geometry).get()]
        if stride == 1:
            out.append(ops.conv2d_dgrad(dy, w, None, (hw, hw), *geometry, add=add, relu_y=add).get())
        return out
    terms(ALWAYS)
    got = results()
    terms(NEVER)
    for a, b in zip(got, results()):
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(np.isinf(a), np.isinf(b))
        finite = np.isfinite(a) & np.isfinite(b)
        assert finite.mean() > .5
        size = float(np.abs(b[finite], dtype=np.float64).max())
        # float32 instructions round every product and sum to a multiple of 2^-149
        np.testing.assert_allclose(a[finite], b[finite], rtol=1e-5,
                                   atol=max(1e-6 * min(size, 1e3 * scale), 2.0 ** -150 * r * r * max(c, k)))


def _distance(got, want, size):
    """2-norm of the error, beyond the rounding of a result, in units of the sums of magnitudes."""
    return float(np.linalg.norm(np.maximum(np.abs(got - want) - 2.0 ** -150, 0) / size))


@pytest.mark.parametrize('kernels', ['gather', 'patch'])
@pytest.mark.parametrize('dims', [(9, 64, 14, 96, 1, 1), (3, 17, 28, 33, 3, 1), (3, 64, 28, 128, 3, 2)])
@pytest.mark.parametrize('ex,ew', [(-120, 40), (-124, 60), (-126, 60), (-133, 60), (-135, 30), (-140, 100), (60, -126),
                                   (100, -140), (-126, 0), (-140, 0), (-70, -70), (-90, 30), (60, 15), (90, 20)])
def test_operands_of_any_magnitude(dims, ex, ew, kernels, terms):
    """Sums as near to float64 ones as those of the float32 instructions, where the last terms of one operand lie
    below the least bfloat16, where all of them do, and where lifted sums overflow."""
    import torch
    n, c, hw, k, r, stride = dims
    xh, wh, dyh = (np.ldexp(a, e) for a, e in zip(_arrays(*dims, np.random.default_rng(8)), (ex, ew, ex)))
    geometry = ((stride, stride), (r // 2, r // 2), (1, 1), 1)

    def sums(x, w, dy):
        x, w, dy = (torch.tensor(a, dtype=torch.float64) for a in (x, w, dy))
        x.requires_grad = True
        y = torch.nn.functional.conv2d(x, w, padding=r // 2, stride=stride)
        y.backward(dy)
        return y.detach().numpy(), x.grad.numpy()
    want, size = sums(xh, wh, dyh), sums(np.abs(xh), np.abs(wh), np.abs(dyh))
    x, w, dy = hiparray(xh), hiparray(wh), hiparray(dyh)

    def errors():
        got = (ops.conv2d_fwd(x, w, None, *geometry).get(), ops.conv2d_dgrad(dy, w, None, (hw, hw), *geometry).get())
        return [_distance(a.astype(np.float64), b, np.where(s > 0, s, 1)) for a, b, s in zip(got, want, size)]
    terms(NEVER)
    old = errors()
    terms(ALWAYS)
    if kernels == 'patch':
        _hip.call('tt_conv2d_patch_enable', ALWAYS)
    new = errors()
    assert _last_launch()['persistent_blocks'] == -4 or kernels == 'gather'
    print(dims, ex, ew, kernels, new, old)
    assert all(a <= b for a, b in zip(new, old)), (new, old)


@pytest.mark.parametrize('case,kernels', [(c, 'gather') for c in EDGES] + [(c, 'patch') for c in PATCH_EDGES + STRIDED])
def test_sums_formed_again_at_every_geometry(case, kernels, terms):
    """Lifted operands overflow, and every wave falls back on the float32 instructions."""
    import torch
    n, c, h, w, k, r, s, stride, pad, dil, _ = case
    rng = np.random.default_rng(6)
    p, q = ((x + 2 * a - d * (f - 1) - 1) // t + 1 for x, a, d, f, t in zip((h, w), pad, dil, (r, s), stride))
    xh, wh, dyh = (rng.standard_normal(a).astype(np.float32) for a in ((n, c, h, w), (k, c, r, s), (n, k, p, q)))
    xh, dyh = np.ldexp(xh, 110), np.ldexp(dyh, 110)
    x64, w64 = torch.tensor(np.abs(xh), dtype=torch.float64, requires_grad=True), torch.tensor(np.abs(wh), dtype=torch.float64)
    y64 = torch.nn.functional.conv2d(x64, w64, stride=stride, padding=pad, dilation=dil)
    y64.backward(torch.tensor(np.abs(dyh), dtype=torch.float64))
    size = y64.detach().numpy(), x64.grad.numpy()

    def results():
        x, wt, dy = hiparray(xh), hiparray(wh), hiparray(dyh)
        return [a.get() for a in (ops.conv2d_fwd(x, wt, None, stride, pad, dil, 1), ops.conv2d_dgrad(dy, wt, None, (h, w), stride, pad, dil, 1))]
    terms(NEVER)
    want = results()
    terms(ALWAYS)
    if kernels == 'patch':
        _hip.call('tt_conv2d_patch_enable', ALWAYS)
    for a, b, m in zip(results(), want, size):
        assert np.isfinite(b).all()
        # either sum is off by at most a rounding of 2^-24 for each of its products, of what has been added up
        assert (np.abs(a.astype(np.float64) - b) <= 2 * 2.0 ** -24 * r * s * max(c, k) * m).all()


@pytest.mark.parametrize('dims,kernels', [((64, 512, 28, 256, 1, 1), 'gather'), ((128, 128, 16, 128, 3, 1), 'patch')])
def test_sums_formed_again_keep_pace(dims, kernels, terms):
    """A launch whose every sum is formed again takes two to three times as long as on the float32 instructions alone
    (by single lanes it took 140 to 210 times as long)."""
    n, c, hw, k, r, _ = dims
    xh, wh, _ = _arrays(*dims, np.random.default_rng(1))
    xh[:, -1] = np.inf
    x, w = hiparray(xh), hiparray(wh)

    def milliseconds():
        first, last = _hip.Event(), _hip.Event()
        for i in range(4):
            if i == 1:
                first.record()
            y = ops.conv2d_fwd(x, w, None, (1, 1), (r // 2, r // 2), (1, 1), 1)
        last.record()
        _hip.synchronize()
        assert not np.isfinite(y.get()[:, :, 1:-1, 1:-1]).any()
        return first.elapsed_ms(last)
    terms(NEVER)
    alone = milliseconds()
    terms(WHERE_FASTER)
    again = milliseconds()
    assert (_last_launch()['persistent_blocks'] == -4) == (kernels == 'patch') and in_terms()
    print(dims, alone, again)
    assert again < 10 * alone


@pytest.mark.parametrize('c', [1, 3, 4])
def test_short_sums_stay_on_the_more_accurate_instructions(c, terms):
    """However large the launch: three products and fewer are nearer to their float64 sum in float32 instructions."""
    rng = np.random.default_rng(12)
    x, w = hiparray.zeros((550 // c, c, 112, 112)), hiparray.zeros((256, c, 1, 1))      # 3.5e9 products and sums
    terms(WHERE_FASTER)
    ops.conv2d_fwd(x, w, None, (1, 1), (0, 0), (1, 1), 1)
    assert in_terms() == (c >= 4)
    xh, wh = rng.standard_normal((8, c, 56, 56)).astype(np.float32), rng.standard_normal((96, c, 1, 1)).astype(np.float32)
    want = np.einsum('nchw,kc->nkhw', xh.astype(np.float64), wh[:, :, 0, 0].astype(np.float64))
    size = np.einsum('nchw,kc->nkhw', np.abs(xh).astype(np.float64), np.abs(wh[:, :, 0, 0]).astype(np.float64))

    def error(which):
        terms(which)
        return _distance(ops.conv2d_fwd(hiparray(xh), hiparray(wh), None, (1, 1), (0, 0), (1, 1), 1).get().astype(np.float64), want, size)
    if c >= 4:
        assert error(ALWAYS) <= error(NEVER)


@pytest.mark.parametrize('dims', [d for d in GEOMETRIES if d[5] == 1])
def test_epilogues(dims, terms):
    """The same bits as the entry points they stand in for; an epilogue that writes what it reads keeps the float32
    instructions."""
    n, c, hw, k, r, _ = dims
    terms(ALWAYS)
    rng = np.random.default_rng(3)
    x, w, res = (hiparray(a) for a in _arrays(*dims, rng))
    mask = hiparray(rng.standard_normal(x.shape).astype(np.float32))
    mean, gamma, beta = (hiparray(rng.standard_normal(k).astype(np.float32)) for _ in range(3))
    var = hiparray(rng.random(k).astype(np.float32) + np.float32(.5))
    geometry = ((1, 1), (r // 2, r // 2), (1, 1), 1)
    y = ops.conv2d_fwd(x, w, None, *geometry)
    want = np.maximum(ops.bn_fwd_eval(y, gamma, beta, mean, var, 1e-5)[0].get() + res.get(), 0)

    def fused(out, residual):
        _hip.call('tt_conv2d_norm_act_fwd_f32', x.ptr, w.ptr, None, out.ptr, mean.ptr, var.ptr, gamma.ptr, beta.ptr, 1e-5,
                  residual.ptr, 1, n, c, hw, hw, k, r, r, 1, 1, r // 2, r // 2, 1, 1, 1)
        return out.get()
    assert np.array_equal(fused(hiparray.empty(y.shape), res), want) and in_terms()
    dx = ops.conv2d_dgrad(res, w, None, (hw, hw), *geometry).get()
    both = ops.conv2d_dgrad(res, w, None, (hw, hw), *geometry, add=x, relu_y=mask).get()
    assert in_terms() and np.array_equal(both, (dx + x.get()) * (mask.get() > 0))
    got = fused(res, res)
    assert not in_terms()
    np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4 * float(np.abs(want).max()))
