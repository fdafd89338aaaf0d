"""The squeezed vector from the parts that the depthwise workgroups leave (mobile_block.hip): more parts than one round of
requests takes, one, two and eight threads to an element, channel groups that are not full, as many channels, squeezed elements
and bands as there are room for; against the oracle's evaluator, with the bounds of the block's other tests."""
import pytest

from test_gpu_mobile_block import check_block

pytestmark = pytest.mark.gpu


# cin, exp, cout, K, stride, SQ, N, H, W: bands x groups of channels parts
@pytest.mark.parametrize("case", [
    (8, 264, 16, 3, 1, 256, 1, 41, 9), (8, 264, 16, 3, 1, 8, 1, 43, 9), (16, 768, 24, 3, 1, 192, 1, 37, 7), (40, 240, 40, 5, 1, 64, 1, 47, 33),
    (8, 8, 8, 3, 1, 8, 1, 1, 1), (16, 72, 96, 5, 2, 24, 8, 33, 30), (24, 40, 24, 5, 1, 104, 513, 5, 4), (8, 520, 8, 3, 2, 136, 16, 19, 6)])
def test_many_parts(case):
    tags = check_block(case)
    assert tags.get("se_project") == 1 and sum(v for k, v in tags.items() if k.startswith("dw_block")) == 1, tags
