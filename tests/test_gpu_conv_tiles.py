"""The tile rule of the float32 forward and input gradient at its lines: up to 32 rows with tiles enough for
the device, and few tiles with a long reduction, which is shared between blocks where that shortens it."""
import ctypes

import pytest

from pytortto_amd import _hip, ops
from pytortto_amd.xparray import hiparray
from tests.test_gpu_conv import _last_launch, _run_conv

pytestmark = pytest.mark.gpu

# n, c, h, w, k, r, s, stride, pad, dilation, groups; tile of the input gradient (rows, pixels, shared between blocks)
CASES = [((4, 32, 128, 128, 32, 3, 3, (1, 1), (1, 1), (1, 1), 1), (32, 256, False)),     # 256 tiles
         ((4, 31, 128, 127, 32, 3, 3, (1, 1), (1, 1), (1, 1), 1), (64, 64, False)),      # 254
         ((4, 33, 128, 128, 8, 1, 1, (1, 1), (0, 0), (1, 1), 1), (64, 64, False)),       # 33 rows, plain product
         ((2, 6, 182, 182, 10, 3, 2, (1, 1), (1, 1), (1, 1), 2), (32, 256, False)),      # per group
         ((1, 16, 9, 9, 336, 1, 1, (1, 1), (0, 0), (1, 1), 1), (64, 64, True)),          # 21 chunks: eight and the exchange
         ((1, 16, 9, 9, 320, 1, 1, (1, 1), (0, 0), (1, 1), 1), (64, 64, False)),         # 20: not shorter
         ((2, 10, 1, 1, 2048, 1, 1, (1, 1), (0, 0), (1, 1), 1), (64, 64, True))]         # 128


@pytest.mark.parametrize('case,tile', CASES, ids=[str(c[:6]) for c, _ in CASES])
def test_tile_rule(case, tile):
    _run_conv(case)
    plan = _last_launch()
    assert (plan['bm'], plan['bn'], plan['sharing_blocks'] > 0) == tile


@pytest.mark.parametrize('k,c,r', [(192, 24, 3), (129, 160, 3), (190, 7, 3), (320, 33, 1), (193, 16, 3), (130, 3, 7)])
def test_weight_gradient_rows_that_fill_no_128(k, c, r):
    """Rows and columns on either side of the lines between 64- and 128-wide tiles."""
    _run_conv((3, c, 11, 9, k, r, r, (1, 1), (r // 2, r // 2), (1, 1), 1))


@pytest.mark.parametrize('case,sharing', [((1, 16, 9, 9, 336, 1, 1, (1, 1), (0, 0), (1, 1), 1), 5),        # two tiles of 21 steps, eight to a block
                                          ((8, 128, 28, 28, 128, 3, 3, (1, 1), (1, 1), (1, 1), 1), 441)])  # 49
def test_blocks_without_a_share_are_not_launched(case, sharing):
    _run_conv(case)
    plan = _last_launch()
    assert plan['whole_tiles'] == 0 and plan['persistent_blocks'] == plan['sharing_blocks'] == sharing


@pytest.mark.parametrize('case,sharing', [((1, 150, 9, 9, 100, 1, 1, (1, 1), (0, 0), (1, 1), 1), 0),       # 10 steps
                                          ((1, 241, 9, 9, 100, 1, 1, (1, 1), (0, 0), (1, 1), 1), 8),       # 16, four tiles
                                          ((8, 138, 20, 20, 128, 1, 1, (1, 1), (0, 0), (1, 1), 1), 0)])    # 9, a hundred tiles
def test_split_rule_in_bf16_arithmetic(case, sharing):
    n, c, h, w, k, r, s, stride, pad, dil, groups = case
    x, wt = hiparray.zeros((n, c, h, w)), hiparray.zeros((k, c, r, s))
    _hip.set_conv_math('bf16')
    try:
        ops.conv2d_fwd(x, wt, None, stride, pad, dil, groups)
        plan = _last_launch()
    finally:
        _hip.set_conv_math('f32')
    assert plan['persistent_blocks'] == plan['sharing_blocks'] == sharing


@pytest.mark.parametrize('dims,tiles', [((24, 160, 45, 37, 192, 3, 3, 1, 1, 1, 1, 1, 1, 1), 3 * 12),      # 64 x 128
                                        ((67, 64, 38, 8, 134, 3, 3, 2, 2, 1, 1, 1, 1, 1), 2 * 9),         # few chunks: 128 x 64
                                        ((130, 404, 17, 12, 2164, 1, 1, 2, 2, 0, 0, 1, 1, 4), 4 * 5 * 2)])
def test_weight_gradient_tile_rule(dims, tiles):
    n, c, h, w, k, r, s, sh, sw, ph, pw, dh, dw, g = dims
    p, q = ((h + 2 * ph - r) // sh + 1, (w + 2 * pw - s) // sw + 1)
    x, dy = hiparray.zeros((n, c, h, w)), hiparray.zeros((n, k, p, q))
    ops.conv2d_wgrad(x, dy, (k, c // g, r, s), (sh, sw), (ph, pw), (dh, dw), g)
    plan = (ctypes.c_int * 4)()
    _hip.call('tt_conv2d_last_wgrad_launch', plan)
    assert plan[0] == tiles
