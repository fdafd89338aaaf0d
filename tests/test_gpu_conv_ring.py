"""The fp16 implicit GEMM through an LDS ring (conv_ring.hip) where it can go wrong: every form, pixel and filter counts that end
inside a tile, K axes that end inside a slab, taps that share a slab, strides and padding, one slab, residual before and
after the activation; against torch on the CPU."""
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, FP16_REL_L2, dev, host, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu

def rand(seed, *shape):
    return torch.rand(shape, generator=torch.Generator().manual_seed(seed)).mul_(2).sub_(1).half().float()


@pytest.mark.parametrize("N,C,F,H,W,R,stride,pad,act", [
    (2, 64, 32, 91, 93, 1, 1, 0, "silu"),     # one slab, pixels end inside a tile
    (3, 96, 136, 37, 41, 1, 1, 0, None),      # the second slab is half full, filters end inside a block
    (20, 256, 120, 40, 40, 1, 2, 0, "relu"),  # strided pixels
    (8, 40, 264, 28, 28, 1, 1, 0, "relu"),    # less than one slab
    (64, 64, 24, 40, 41, 1, 1, 0, "silu"),    # few filters
    (20, 64, 72, 61, 62, 5, 2, 1, "relu"),    # taps of one slab, and halo on every side
    (2, 16, 40, 70, 61, 3, 1, 1, "silu"),     # four taps to a slab
    (9, 24, 72, 61, 62, 3, 2, 1, None),       # taps that straddle slabs
    (8, 40, 72, 64, 64, 5, 1, 4, "relu"),     # padding wider than the centre
    (16, 512, 256, 20, 20, 1, 1, 0, "relu"),  # eight slabs
    (33, 64, 136, 57, 55, 3, 2, 1, None),     # 3x3 stride 2
    (8, 512, 128, 60, 60, 1, 1, 0, "relu"),   # many pixels, eight slabs
])
def test_ring_kernel_matches_torch(N, C, F, H, W, R, stride, pad, act):
    tags = check_layer(N, C, F, H, W, R, stride, pad, act)
    assert all(t.startswith("conv_ring<") for t in tags), tags


# every form of the kernel with every kind of window that comes to it: 1x1 (slabs of 64 channels, the last one part empty), taps of
# whole slabs, and taps that share slabs; no pixel or filter count is a multiple of the form's tile
@pytest.mark.parametrize("N,C,F,H,W,R,stride,pad,form", [
    (1, 8, 8, 6, 6, 1, 2, 0, "64x64"), (12, 64, 72, 64, 17, 3, 1, 2, "64x64"), (10, 16, 40, 12, 28, 3, 1, 2, "64x64"),
    (20, 264, 264, 9, 5, 1, 1, 0, "64x64,2"), (26, 64, 72, 7, 18, 3, 1, 2, "64x64,2"),
    (9, 32, 8, 49, 53, 1, 1, 0, "64x32"), (15, 64, 8, 52, 29, 3, 1, 2, "64x32"), (34, 16, 8, 40, 18, 3, 1, 1, "64x32"),
    (1, 720, 1480, 37, 43, 1, 1, 0, "64x128,2"), (31, 64, 72, 10, 51, 5, 1, 2, "64x128,2"), (6, 16, 72, 33, 102, 5, 1, 2, "64x128,2"),
    (34, 24, 72, 94, 16, 1, 1, 0, "128x128"), (32, 16, 72, 5, 103, 3, 1, 2, "128x128"),
    (6, 200, 848, 85, 7, 1, 1, 0, "128x128,2"), (34, 64, 72, 98, 5, 3, 1, 2, "128x128,2"),
])
def test_every_form(N, C, F, H, W, R, stride, pad, form):
    assert check_layer(N, C, F, H, W, R, stride, pad, "silu") == ["conv_ring<%s>" % form]


def check_layer(N, C, F, H, W, R, stride, pad, act):
    """The layer without and with a residual against torch; the tags of its launches."""
    oh, ow = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - R) // stride + 1
    x, w, r = rand(1, N, C, H, W), (rand(2, F, C, R, R) * (2.0 / (R * R * C)) ** 0.5).half().float(), rand(3, N, F, oh, ow)
    y = torch.nn.functional.conv2d(x, w, stride=stride, padding=pad)
    f = {None: lambda v: v, "relu": torch.relu, "silu": torch.nn.functional.silu}[act]
    code = {None: abi.ACT_NONE, "relu": abi.ACT_RELU, "silu": abi.ACT_SILU}[act]
    layer, xd, rd = Conv(abi.F16, w.numpy(), stride, pad, relu=code), dev(nhwc(x.numpy()), abi.F16), dev(nhwc(r.numpy()), abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        plain, added = host(layer(xd, abi.NHWC)), host(layer(xd, abi.NHWC, residual=rd))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    print(tags, flush=True)
    assert rel_l2(nchw(plain), f(y).numpy()) < 2e-3 < FP16_REL_L2
    assert rel_l2(nchw(added), f(y + r).numpy()) < 2e-3
    return tags


def test_shortcut_filters_ride_along():
    """A ResNet-18 pass whose stride-2 layers are large enough to come here: their 1x1 shortcuts are further tiles of the same
    launch.  Stage outputs of three images, spread over the batch, against the oracle's."""
    import numpy as np
    import oracle
    from nncv_amd import synth
    from gpu_util import Model
    n, pick = 37, [0, 17, 36]
    blob = synth.round_fp16(synth.resnet18_params())
    x = synth.round_fp16(synth.uniform(4005, (n, 3, 219, 227), 0.0, 1.0))
    m = Model(blob, abi.F16, abi.ALGO_IGEMM)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(m(dev(x, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    print(tags, flush=True)
    assert sum(v for k, v in tags.items() if k.startswith("conv_ring<")) >= 1, tags
    want = oracle.resnet18_forward(np.ascontiguousarray(x[pick]), blob)
    assert rel_l2(got[pick], want) < FP16_REL_L2
    assert (got[pick].argmax(1) == want.argmax(1)).all()
