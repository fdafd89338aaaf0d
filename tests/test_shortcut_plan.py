"""Where the shortcut of an fp32 down-sampling block is computed behind the tile of its 3x3 convolution and where in workgroups of its own
(nncv_hip_conv_shortcut_plan, host arithmetic only): the line at 200 tiles, and the tiles that come up at all."""
import ctypes

import pytest

from nncv_amd import abi

# filters, pixels and K groups of the tiles that a block of ResNet-18 can get; test_gpu_conv_shortcut.py runs each
TILES = {64: {(16, 16, 4), (32, 16, 8), (32, 32, 4), (32, 32, 8), (64, 32, 4), (64, 64, 1)},
         128: {(16, 16, 16), (32, 16, 8), (64, 32, 4), (64, 64, 1)}, 256: {(16, 16, 16), (32, 16, 8), (64, 32, 4), (64, 64, 1)}}


def plan(N, H, W, C, F):
    p = (ctypes.c_int * 5)()
    return None if abi.lib().nncv_hip_conv_shortcut_plan(N, H, W, C, F, p) else tuple(p)


@pytest.mark.parametrize("C", sorted(TILES))
def test_every_number_of_pixels(C):
    seen, P = set(), 1
    while P < 2_000_000:
        for q in (P, P + 1):
            p = plan(1, 2 * q, 1, C, 2 * C)
            if p is not None:
                rows, cols, kg, tiles, behind = p
                assert tiles == -(-2 * C // rows) * -(-q // cols) and behind == (tiles >= 200), (q, p)
                seen.add((rows, cols, kg))
        P += max(1, P // 200)
    assert seen == TILES[C]


def test_refuses_what_is_no_block():
    for bad in [(0, 8, 8, 64, 128), (1, 0, 8, 64, 128), (1, 8, 8, 0, 128), (1, 8, 8, 64, 0), (1, 8, 8, 40, 80), (1, 8, 8, 64, 72)]:
        assert plan(*bad) is None
    assert abi.lib().nncv_hip_conv_shortcut_plan(1, 8, 8, 64, 128, None) == 1
