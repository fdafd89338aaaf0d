"""The barrier-free implicit GEMM (conv_direct.hip) where it can go wrong: every form, fewer rounds of K than wave groups, taps
that are not whole rounds, pixel and filter counts that end inside a tile, one and many tiles, windows of every kind,
strides, padding wider than the image; against torch on the CPU."""
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, FP32_MAX_REL, FP16_REL_L2, dev, host, max_rel, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu


def rand(seed, *shape):
    return torch.rand(shape, generator=torch.Generator().manual_seed(seed)).mul_(2).sub_(1)


# N, C, F, H, W, R, stride, pad
BOTH = [(1, 512, 512, 7, 7, 3, 1, 1), (1, 1024, 40, 5, 5, 1, 1, 0), (1, 512, 136, 9, 7, 3, 2, 1), (2, 40, 72, 13, 11, 5, 2, 2), (3, 128, 64, 3, 3, 5, 1, 4)]
F32 = [(1, 4, 8, 1, 1, 1, 1, 0), (1, 32, 40, 5, 7, 3, 1, 1), (2, 20, 36, 9, 9, 3, 1, 1), (6, 64, 96, 29, 39, 3, 2, 1), (3, 512, 1000, 7, 9, 1, 1, 0),
       (3, 256, 256, 15, 20, 3, 1, 1), (1, 12, 20, 40, 33, 7, 2, 3)]


@pytest.mark.parametrize("dt,case", [(d, c) for d in (abi.F32, abi.F16) for c in BOTH] + [(abi.F32, c) for c in F32])
def test_direct_kernel_matches_torch(dt, case):
    tags = check_layer(dt, case)
    assert any("_direct<" in t for t in tags), tags


# every form of the kernel, with taps of whole rounds of K (128 bytes of channels) and without; no pixel or filter count is a
# multiple of the form's tile, and the last round of the others is part empty
FORMS = [
    (abi.F32, 6, 64, 820, 9, 8, 1, 1, 1, "conv1x1_direct<f32,32x32,splitk2>"), (abi.F32, 1, 48, 584, 10, 88, 1, 1, 0, "conv1x1_direct<f32,32x32,splitk2>"),
    (abi.F32, 1, 96, 540, 33, 11, 1, 1, 1, "conv1x1_direct<f32,32x32,splitk4>"), (abi.F32, 15, 8, 84, 10, 24, 3, 1, 0, "conv3x3_direct<f32,32x32,splitk4>"),
    (abi.F32, 1, 192, 1216, 89, 7, 1, 2, 0, "conv1x1_direct<f32,32x32,splitk8>"), (abi.F32, 1, 4, 24, 209, 35, 7, 1, 3, "conv_direct<f32,32x32,splitk8>"),
    (abi.F32, 1, 32, 20, 7, 3, 1, 1, 0, "conv1x1_direct<f32,16x16,splitk4>"), (abi.F32, 1, 4, 28, 4, 9, 1, 1, 0, "conv1x1_direct<f32,16x16,splitk4>"),
    (abi.F32, 1, 32, 20, 11, 4, 5, 1, 2, "conv_direct<f32,16x16,splitk16>"), (abi.F32, 2, 88, 24, 3, 3, 3, 1, 1, "conv3x3_direct<f32,16x16,splitk16>"),
    (abi.F32, 1, 160, 348, 5, 56, 1, 1, 0, "conv1x1_direct<f32,32x16,splitk8>"), (abi.F32, 1, 16, 52, 37, 40, 3, 1, 2, "conv3x3_direct<f32,32x16,splitk8>"),
    (abi.F32, 7, 96, 108, 24, 42, 3, 1, 1, "conv3x3_direct<f32,64x32,splitk4>"), (abi.F32, 12, 88, 108, 35, 17, 3, 1, 1, "conv3x3_direct<f32,64x32,splitk4>"),
    (abi.F32, 9, 32, 424, 62, 31, 3, 1, 3, "conv3x3_direct<f32,64x64>"), (abi.F32, 12, 156, 1188, 53, 13, 1, 1, 0, "conv1x1_direct<f32,64x64>"),
    (abi.F16, 5, 128, 484, 3, 14, 1, 1, 1, "conv1x1_direct<f16,32x32,splitk4>"), (abi.F16, 3, 8, 52, 37, 21, 3, 1, 3, "conv3x3_direct<f16,32x32,splitk4>"),
    (abi.F16, 2, 320, 336, 4, 79, 1, 1, 0, "conv1x1_direct<f16,32x32,splitk8>"), (abi.F16, 2, 8, 36, 31, 60, 7, 1, 3, "conv_direct<f16,32x32,splitk8>"),
    (abi.F16, 11, 128, 100, 11, 6, 1, 1, 1, "conv1x1_direct<f16,16x16,splitk4>"), (abi.F16, 14, 8, 36, 9, 8, 3, 1, 3, "conv3x3_direct<f16,16x16,splitk4>"),
    (abi.F16, 2, 128, 20, 3, 4, 3, 1, 1, "conv3x3_direct<f16,16x16,splitk8>"), (abi.F16, 1, 16, 20, 7, 9, 7, 2, 3, "conv_direct<f16,16x16,splitk8>"),
    (abi.F16, 1, 640, 20, 4, 11, 3, 1, 1, "conv3x3_direct<f16,16x16,splitk16>"), (abi.F16, 1, 232, 20, 6, 17, 5, 2, 2, "conv_direct<f16,16x16,splitk16>"),
    (abi.F16, 1, 320, 164, 79, 3, 1, 1, 1, "conv1x1_direct<f16,32x16,splitk8>"), (abi.F16, 8, 32, 68, 13, 3, 3, 1, 3, "conv3x3_direct<f16,32x16,splitk8>"),
    (abi.F16, 7, 64, 68, 9, 50, 3, 1, 1, "conv3x3_direct<f16,64x32,splitk4>"), (abi.F16, 15, 8, 68, 65, 4, 7, 1, 3, "conv_direct<f16,64x32,splitk4>"),
    (abi.F16, 17, 128, 76, 8, 59, 3, 1, 1, "conv3x3_direct<f16,64x64,splitk4>"), (abi.F16, 9, 24, 76, 15, 60, 7, 1, 3, "conv_direct<f16,64x64,splitk4>"),
    (abi.F16, 19, 128, 68, 60, 65, 3, 1, 1, "conv3x3_direct<f16,64x64>"), (abi.F16, 14, 48, 84, 86, 63, 5, 1, 2, "conv_direct<f16,64x64>"),
]


@pytest.mark.parametrize("case", FORMS, ids=lambda c: "%s-%s" % (c[9], "lines" if c[2] * (2 if c[0] == abi.F16 else 4) % 128 == 0 else "any"))
def test_every_form(case):
    assert check_layer(case[0], case[1:9]) == [case[9]]


def test_fp32_stride_2_layers_come_here():
    """3x3 stride-2 layers that the implicit GEMM's model would take, and does not get."""
    for case in ((3, 64, 640, 56, 80, 3, 2, 1), (17, 64, 608, 2, 183, 3, 2, 1), (1, 64, 44, 93, 75, 3, 2, 1)):
        tags = check_layer(abi.F32, case)
        assert tags[0].startswith("conv3x3_direct<f32"), (case, tags)


def check_layer(dt, case):
    """The layer with a residual and ReLU against torch; the tags of its launches."""
    N, C, F, H, W, R, stride, pad = case
    oh, ow = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - R) // stride + 1
    x, w, r = rand(1, N, C, H, W), rand(2, F, C, R, R) * (2.0 / (R * R * C)) ** 0.5, rand(3, N, F, oh, ow)
    if dt == abi.F16:
        x, w, r = x.half().float(), w.half().float(), r.half().float()
    want = torch.relu(torch.nn.functional.conv2d(x.double(), w.double(), stride=stride, padding=pad) + r.double()).numpy()
    layer = Conv(dt, w.numpy(), stride, pad, relu=True)
    args = dev(nhwc(x.numpy()), dt), abi.NHWC
    res = dev(nhwc(r.numpy()), dt)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = nchw(host(layer(*args, residual=res)))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert max_rel(got, want) < FP32_MAX_REL if dt == abi.F32 else rel_l2(got, want) < FP16_REL_L2
    return tags
