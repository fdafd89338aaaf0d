"""fp16 3x3 stride-2 layers of 64 channels with their filters in registers (conv3x3s2_resident.hip): rows and columns that end inside a tile,
rows of one tile and of several, odd and even images, filters that end inside a block of 32 and of 128, one tile a workgroup and many; against
torch.  And the shortcut's filters on the centre tap, against the oracle."""
import math

import numpy as np
import pytest
import torch

import graph_bound
import oracle
from nncv_amd import abi, resnet18_spec, synth
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


@pytest.mark.parametrize("N,H,W", [(143, 219, 227), (150, 223, 203), (40, 404, 492)])
def test_values_of_a_block_with_its_shortcut(N, H, W):
    """layer2's first block, value by value: its second one hands its input on (the scale and shift behind its sum are zero)."""
    blob, t, at = synth.round_fp16(synth.resnet18_params()), {}, 0
    for name, shape in resnet18_spec.tensor_table():
        n = math.prod(shape)
        if name in ("layer2.1.bn2.weight", "layer2.1.bn2.bias"):
            blob[at:at + n] = 0
        t[name] = blob[at:at + n].reshape(shape).astype(np.float64)
        at += n
    m = Model(blob, abi.F16)
    xd = (torch.rand((N, 3, H, W), generator=torch.Generator(device="cuda").manual_seed(N), device="cuda") * 2 - 1).half()
    size = lambda v, k: size((v - 1) // 2 + 1, k - 1) if k else v  # of the map after k halvings
    taps = []
    abi.profile_enable(True)
    try:
        for stage, C in ((1, 64), (2, 128)):
            h, w = size(H, stage + 1), size(W, stage + 1)
            logits, tap = torch.empty((N, 1000), device="cuda"), torch.full((N, h, w, C), float("nan"), dtype=torch.float16, device="cuda")
            abi.profile_report()
            abi.check(abi.lib().nncv_hip_resnet18_forward_tap(m.h, xd.data_ptr(), N, H, W, logits.data_ptr(), stage, tap.data_ptr(), None))
            taps.append(np.ascontiguousarray(nchw(host(tap[torch.tensor(sorted({0, 1, N // 2, N - 1}), device="cuda")]))))
        assert abi.profile_report()["conv_ring<s2,resident>"]["launches"] == 1
    finally:
        abi.profile_enable(False)
    params, ops = [], []  # filters and shifts with BatchNorm folded into them, in 64 bits

    def conv(i, name, bn, stride, act):
        w, (g, b, mean, var) = t["layer2.0.%s.weight" % name], [t["layer2.0.%s.%s" % (bn, v)] for v in ("weight", "bias", "running_mean", "running_var")]
        s, o = g / np.sqrt(var + 1e-5), sum(p.size for p in params)
        params.extend([(w * s.reshape(-1, 1, 1, 1)).ravel(), b - mean * s])
        ops.append(abi.graph_op(abi.OP_CONV, [i], len(ops) + 1, F=128, K=w.shape[2], stride=stride, pad=w.shape[2] // 2, act=act, w=o, bias=o + w.size))
        return len(ops)

    y = conv(conv(0, "conv1", "bn1", 2, abi.ACT_RELU), "conv2", "bn2", 1, abi.ACT_NONE)
    s = conv(0, "downsample.0", "downsample.1", 2, abi.ACT_NONE)
    ops.append(abi.graph_op(abi.OP_ADD, [y, s], len(ops) + 1, act=abi.ACT_RELU))
    assert graph_bound.worst(taps[1], ops, taps[0], np.concatenate(params)) < graph_bound.LIMIT
