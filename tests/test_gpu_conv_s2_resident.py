"""fp16 3x3 stride-2 layers of 64 channels with their filters in registers (conv3x3s2_resident.hip): rows and columns that end inside a tile,
rows of one tile and of several, odd and even images, filters that end inside a block of 32 and of 128, one tile a workgroup and many; against
torch.  And the shortcut's filters on the centre tap, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from nncv_amd import abi, synth
from gpu_util import Conv, FP16_REL_L2, Model, dev, host, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,F,H,W,act", [(160, 128, 56, 56, "relu"), (150, 96, 55, 57, None), (150, 128, 63, 58, "silu"), (75, 256, 57, 62, "relu"), (32, 128, 160, 160, "silu"),
                                         (36, 128, 159, 121, None), (170, 72, 57, 61, "relu"), (40, 264, 101, 123, "silu")])
def test_against_torch(N, F, H, W, act):
    g = torch.Generator(device="cuda").manual_seed(H * W)
    x = torch.randn((N, 64, H, W), generator=g, device="cuda").half()
    w = (torch.randn((F, 64, 3, 3), generator=g, device="cuda") * (2.0 / 576) ** 0.5).half()
    scale, shift = torch.rand(F, generator=torch.Generator().manual_seed(1)) + 0.5, torch.randn(F, generator=torch.Generator().manual_seed(2))
    bn = [scale.half().numpy(), shift.half().numpy(), np.zeros(F, np.float16), np.full(F, 1 - 1e-5, np.float16)]
    f = {None: lambda v: v, "relu": torch.relu, "silu": torch.nn.functional.silu}[act]
    layer = Conv(abi.F16, w.float().cpu().numpy(), 2, 1, bn=bn, relu={None: abi.ACT_NONE, "relu": abi.ACT_RELU, "silu": abi.ACT_SILU}[act])
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = torch.from_numpy(np.ascontiguousarray(nchw(host(layer(dev(nhwc(x.float().cpu().numpy()), abi.F16), abi.NHWC))))).double()
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert tags == ["conv_ring<s2,resident>"], tags
    pick = sorted({0, 1, N // 2, N - 2, N - 1})
    xc, wc = x.cpu().double()[pick], w.cpu().double()
    b = [torch.from_numpy(v.astype(np.float64)) for v in bn]
    y = torch.nn.functional.batch_norm(torch.nn.functional.conv2d(xc, wc, stride=2, padding=1), b[2], b[3], b[0], b[1], eps=1e-5)
    exact, size = f(y), torch.nn.functional.conv2d(xc.abs(), wc.abs(), stride=2, padding=1) * b[0].view(1, -1, 1, 1)
    # half an ulp of the result, 576 additions in fp32 and a few of BN and the activation
    room = exact.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24 + 580 * 2.0 ** -24 * (size + 4)
    assert ((got[pick] - exact).abs() <= room).all(), ((got[pick] - exact).abs() / room).max()


def test_shortcut_behind_the_tile():
    n, pick = 143, [0, 70, 142]
    blob = synth.round_fp16(synth.resnet18_params())
    x = synth.round_fp16(synth.uniform(4013, (n, 3, 219, 227), 0.0, 1.0))
    m = Model(blob, abi.F16, abi.ALGO_IGEMM)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(m(dev(x, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    assert tags.get("conv_ring<s2,resident>") == 1, tags
    want = oracle.resnet18_forward(np.ascontiguousarray(x[pick]), blob)
    assert rel_l2(got[pick], want) < FP16_REL_L2
    assert (got[pick].argmax(1) == want.argmax(1)).all()
