"""The stream kernel on layers of five to eight channel slabs and on tiles that span several small images, against torch in 64 bits
with every value an fp16 one: an fp16 result is off by its one rounding and the fp32 sums' error."""
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, dev, host, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu

# N, H, W, C, F, tag: two images and more a tile (rows of 3 to 8 pixels), the last tile part empty, filters in 32s, 64s and 128s
CASES = [(41, 7, 7, 512, 512, "1x2x2"), (50, 7, 7, 512, 512, "1x2x2"), (101, 7, 7, 512, 512, "1x4x1"), (41, 8, 8, 384, 512, "1x2x2"), (37, 22, 3, 384, 512, "1x2x2"),
         (111, 3, 8, 192, 192, "1x1x4"), (33, 10, 10, 448, 512, "1x2x2"), (7, 32, 32, 320, 320, "1x2x2"), (19, 9, 11, 256, 256, "1x1x4"),
         # little more than 128 blocks of 32 filters
         (32, 7, 7, 512, 512, "1x1x4"), (18, 5, 31, 448, 160, "1x1x4"), (46, 10, 10, 64, 96, "1x1x4"), (7, 13, 17, 256, 320, "1x1x4")]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
def test_deep_layers_and_tiles_of_several_images(case):
    N, H, W, C, F, form = case
    g = torch.Generator().manual_seed(N + C)
    x, r = torch.randn((N, C, H, W), generator=g).half().float(), torch.randn((N, F, H, W), generator=g).half().float()
    w = (torch.randn((F, C, 3, 3), generator=g) * (2.0 / (9 * C)) ** 0.5).half().float()
    want = torch.relu(torch.nn.functional.conv2d(x.double(), w.double(), padding=1) + r.double()).numpy()
    layer = Conv(abi.F16, w.numpy(), 1, 1, relu=True)
    args, res = (dev(nhwc(x.numpy()), abi.F16), abi.NHWC), dev(nhwc(r.numpy()), abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = nchw(host(layer(*args, residual=res)))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert tags == ["conv3x3_stream<f16,%s>" % form]
    assert rel_l2(got, want) < 4e-4  # half an ulp of eleven bits, 2.8e-4 in the mean over a binade


# with passes in flight the lines are 144 blocks and, from five slabs on, 320: below them the patch kernel
@pytest.mark.parametrize("case", [(5, 28, 28, 128, 128, "conv3x3_patch<f16,1,4>"), (32, 7, 7, 512, 512, "conv3x3_patch<f16,1,4>"),
                                  (6, 28, 28, 128, 128, "conv3x3_stream<f16,1x4x1>"), (41, 7, 7, 512, 512, "conv3x3_stream<f16,1x4x1>")],
                         ids=lambda c: "x".join(map(str, c[:5])))
def test_lines_with_passes_in_flight(case):
    N, H, W, C, F, tag = case
    g = torch.Generator().manual_seed(N)
    x, w = torch.randn((N, C, H, W), generator=g).half().float(), (torch.randn((F, C, 3, 3), generator=g) * (2.0 / (9 * C)) ** 0.5).half().float()
    try:
        abi.check(abi.lib().nncv_hip_set_overlap_hint(4))
        layer, xd = Conv(abi.F16, w.numpy(), 1, 1, relu=True), dev(nhwc(x.numpy()), abi.F16)
        abi.profile_enable(True)
        abi.profile_report()
        got = nchw(host(layer(xd, abi.NHWC)))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
        abi.check(abi.lib().nncv_hip_set_overlap_hint(1))
    assert tags == [tag]
    assert rel_l2(got, torch.relu(torch.nn.functional.conv2d(x.double(), w.double(), padding=1)).numpy()) < 4e-4
