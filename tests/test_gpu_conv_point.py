"""fp16 1x1 layers of many channels with their filters as fragments (conv_ring.hip) where that can go wrong: pixels and filters that end inside a
tile, eight slabs and many, the smallest and the largest launch of the rule and those next to it, rows of a wider tensor through two joined
layers; against torch."""
import pytest
import torch

import graph_bound
import oracle
from nncv_amd import abi, synth
from gpu_util import Conv, FP16_REL_L2, Graph, dev, host, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,F,H,W,act,point", [
    (2, 512, 512, 42, 43, "relu", True), (7, 640, 72, 32, 32, None, True), (1, 1088, 264, 59, 61, "silu", True), (25, 512, 1000, 8, 16, "relu", True), (3, 576, 136, 64, 66, None, True),
    (1, 512, 128, 83, 85, "relu", False), (16, 512, 1040, 13, 14, "silu", False), (25, 512, 64, 20, 20, None, False), (16, 520, 512, 20, 20, "relu", False)])
def test_against_torch(N, C, F, H, W, act, point):
    g = torch.Generator().manual_seed(C + F)
    x = torch.rand((N, C, H, W), generator=g).mul_(2).sub_(1).half().float()
    w = (torch.rand((F, C, 1, 1), generator=g).mul_(2).sub_(1) * (2.0 / C) ** 0.5).half().float()
    f = {None: lambda v: v, "relu": torch.relu, "silu": torch.nn.functional.silu}[act]
    layer = Conv(abi.F16, w.numpy(), 1, 0, relu={None: abi.ACT_NONE, "relu": abi.ACT_RELU, "silu": abi.ACT_SILU}[act])
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(layer(dev(nhwc(x.numpy()), abi.F16), abi.NHWC))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert (tags == ["conv_ring<64x128,point>"]) == point, tags
    assert rel_l2(nchw(got), f(torch.nn.functional.conv2d(x, w)).numpy()) < 2e-3 < FP16_REL_L2
    exact, size = f(torch.nn.functional.conv2d(x.double(), w.double())), torch.nn.functional.conv2d(x.double().abs(), w.double().abs())
    # every value: half an ulp of it, C additions in fp32 and a few for the activation
    room = exact.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24 + (C + 4) * 2.0 ** -24 * size
    err = (torch.from_numpy(nchw(got)).double() - exact).abs()
    assert (err <= room).all(), float((err / room).max())


@pytest.mark.parametrize("c_,N,H,W", [(128, 3, 50, 51), (192, 1, 63, 65), (64, 4, 45, 47)])
def test_two_joined_layers(c_, N, H, W):
    """... whose results are slices of one tensor and a tensor of their own; the filters of both are one run of fragments."""
    sizes, ops = [], []

    def conv(i, c, f):
        sizes.append(f * c), sizes.append(f)
        w = sum(sizes[:-2])
        ops.append(abi.graph_op(abi.OP_CONV, [i, -1], len(ops) + 1, F=f, K=1, act=abi.ACT_SILU, w=w, bias=w + f * c))
        return len(ops)

    x = conv(0, 16, 512)
    y, z = conv(x, 512, c_), conv(x, 512, c_)
    t = conv(y, c_, 24)
    ops.append(abi.graph_op(abi.OP_CONCAT, [t, z], len(ops) + 1, stride=0))
    conv(len(ops), 24 + c_, 32)
    blob, inp = synth.round_fp16(synth.normal(8400, (sum(sizes),), std=0.05)), synth.round_fp16(synth.normal(8401, (N, 16, H, W)))
    g = Graph(ops, 16, blob, abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(inp, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    assert tags.get("conv_ring<64x128,point>") == 1, tags
    assert rel_l2(got, oracle.run_graph(ops, inp, blob, 16)) < FP16_REL_L2
    assert graph_bound.worst(got, ops, inp, blob) < graph_bound.LIMIT  # every value
    g.close()
