"""3x3 layers whose filters come as fragments (conv_ring.hip) where they can go wrong: both tile heights, pixels and filters that
end inside a tile, one slab and many, rows shorter than a load's eight pixels, one-row and one-column images, images with odd and
even sizes; against torch on the CPU.  And the shortcut's filters riding on the centre tap, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from nncv_amd import abi, synth
from gpu_util import Conv, FP16_REL_L2, Model, dev, host, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,F,H,W,act,bp", [
    (41, 64, 128, 46, 17, "relu", 64), (61, 64, 120, 21, 38, None, 64), (7, 192, 352, 49, 81, "silu", 64), (37, 128, 264, 31, 29, "relu", 128),
    (1500, 64, 72, 5, 9, "relu", 64), (2500, 64, 96, 1, 8, None, 64), (2000, 128, 72, 9, 1, "relu", 64), (20, 256, 512, 41, 40, "silu", 64),
    (64, 128, 200, 89, 31, "relu", 128), (71, 256, 488, 53, 20, "silu", 128), (20, 512, 232, 45, 90, None, 128)])
def test_matches_torch(N, C, F, H, W, act, bp):
    g = torch.Generator().manual_seed(N * C + F)
    x = torch.rand((N, C, H, W), generator=g).mul_(2).sub_(1).half().float()
    w = (torch.rand((F, C, 3, 3), generator=g).mul_(2).sub_(1) * (2.0 / (9 * C)) ** 0.5).half().float()
    f = {None: lambda v: v, "relu": torch.relu, "silu": torch.nn.functional.silu}[act]
    layer = Conv(abi.F16, w.numpy(), 2, 1, relu={None: abi.ACT_NONE, "relu": abi.ACT_RELU, "silu": abi.ACT_SILU}[act])
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(layer(dev(nhwc(x.numpy()), abi.F16), abi.NHWC))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert tags == ["conv_ring<%dx128,frag>" % bp], tags
    pick = sorted({0, 1, N // 2, N - 2, N - 1})
    want = f(torch.nn.functional.conv2d(x[pick], w, stride=2, padding=1)).numpy()
    assert rel_l2(nchw(got)[pick], want) < 2e-3 < FP16_REL_L2


def test_shortcut_rides_on_the_centre_tap():
    """ResNet-18 with 200 tiles and more in the last stride-2 layer: three images, spread over the batch, against the oracle's."""
    n, pick = 139, [0, 70, 138]
    blob = synth.round_fp16(synth.resnet18_params())
    x = synth.round_fp16(synth.uniform(4011, (n, 3, 219, 227), 0.0, 1.0))
    m = Model(blob, abi.F16, abi.ALGO_IGEMM)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(m(dev(x, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    assert tags.get("conv_ring<128x128,frag>") == 1, tags
    want = oracle.resnet18_forward(np.ascontiguousarray(x[pick]), blob)
    assert rel_l2(got[pick], want) < FP16_REL_L2
    assert (got[pick].argmax(1) == want.argmax(1)).all()
