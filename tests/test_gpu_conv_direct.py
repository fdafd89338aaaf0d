"""The barrier-free implicit GEMM (conv_direct.hip) where it can go wrong: fewer rounds of K than wave groups, taps that are
not whole rounds, pixel and filter counts that end inside a tile, one and many tiles, windows of every kind, strides,
padding wider than the image; against torch on the CPU."""
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
       (7, 256, 256, 15, 20, 3, 1, 1), (1, 12, 20, 40, 33, 7, 2, 3)]


@pytest.mark.parametrize("dt,case", [(d, c) for d in (abi.F32, abi.F16) for c in BOTH] + [(abi.F32, c) for c in F32])
def test_direct_kernel_matches_torch(dt, case):
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
    assert any("_direct<" in t for t in tags), tags
    assert max_rel(got, want) < FP32_MAX_REL if dt == abi.F32 else rel_l2(got, want) < FP16_REL_L2
