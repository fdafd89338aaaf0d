"""Detection heads (detect_head.hip) in runs of tiles with their filters in registers, and of so many channels that a tile's pixels come in parts:
two, three and four tiles a run, a last run and a last tile that are not whole, one slab of channels and two, pieces that do not start on 16 bytes."""
import pytest

import test_gpu_detect_head as heads

pytestmark = pytest.mark.gpu


# channels of each level, anchors, values per box, N, H, W of the first level, merged
@pytest.mark.parametrize("case", [((64,), 3, 85, 8, 79, 81, True), ((128,), 1, 201, 9, 101, 83, True), ((128, 64), 2, 128, 13, 120, 66, True), ((640,), 2, 100, 1, 9, 7, True),
                                  ((64, 1088), 3, 84, 2, 21, 17, True)])
def test_runs(case):
    heads.test_detect_heads(case)
