"""The residual blocks of layer1 in one launch each (basic_block.hip) where their strips, rows and slots end, against 64 bits."""
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from nncv_amd import abi, resnet18_spec, synth
from gpu_util import Model

pytestmark = pytest.mark.gpu

TAG = "basic_block<f16,64>"


@pytest.fixture(scope="module")
def net():
    """fp16 ResNet-18 whose second block hands its input on (the scale and shift behind its sum are zero), and the first block's tensors; the network as it
    is, and the second block's."""
    blob, parts, at = synth.round_fp16(synth.resnet18_params()), [], 0
    whole, full = blob.copy(), []
    for k, (_, shape) in enumerate(resnet18_spec.tensor_table()[:25]):
        n = math.prod(shape)
        full.append(torch.from_numpy(whole[at:at + n].reshape(shape).astype(np.float64)))
        if k in (21, 22):
            blob[at:at + n] = 0
        parts.append(torch.from_numpy(blob[at:at + n].reshape(shape).astype(np.float64)))
        at += n
    assert parts[20].shape == (64, 64, 3, 3) and not parts[21].any() and not parts[22].any()
    return Model(blob, abi.F16), parts[5:10], parts[10:15], Model(whole, abi.F16), full[15:20], full[20:25]


def _tap(m, x, stage):
    N, _, H, W = x.shape
    h, w = ((H - 1) // 2) // 2 + 1, ((W - 1) // 2) // 2 + 1
    logits = torch.empty((N, 1000), dtype=torch.float32, device="cuda")
    tap = torch.full((N, h, w, 64), float("nan"), dtype=torch.float16, device="cuda")
    abi.profile_enable(True)
    try:
        abi.profile_report()
        abi.check(abi.lib().nncv_hip_resnet18_forward_tap(m.h, x.data_ptr(), N, H, W, logits.data_ptr(), stage, tap.data_ptr(), None))
        torch.cuda.synchronize()
        rep = abi.profile_report()
    finally:
        abi.profile_enable(False)
    return tap.cpu().double().permute(0, 3, 1, 2), rep


def _layer(x, parts):
    """The convolution under its BatchNorm, and the magnitudes behind each value."""
    w, g, b, mean, var = parts
    s = g / (var + 1e-5).sqrt()
    sh = b - mean * s
    y = F.conv2d(x, w, padding=1) * s.view(1, -1, 1, 1) + sh.view(1, -1, 1, 1)
    return y, lambda e: F.conv2d(e, w.abs(), padding=1) * s.abs().view(1, -1, 1, 1), (b.abs() + mean.abs() * s.abs()).view(1, -1, 1, 1)


def _check(got, x, first, second):
    y, through1, shift1 = _layer(x, first)
    y = torch.relu(y)
    # a sum of 576 products in steps of 16 and its scale, rounded to 24 bits each; what lies between the convolutions is fp16 (11 bits)
    e1 = 40 * 2.0 ** -24 * (through1(x.abs()) + shift1) + 2.0 ** -11 * y
    z, through2, shift2 = _layer(y, second)
    want = torch.relu(z + x)
    bound = through2(e1) + 40 * 2.0 ** -24 * (through2(y) + shift2 + x.abs())
    bound = bound + 2.0 ** -11 * (want + bound) + 2.0 ** -24
    assert torch.isfinite(got).all()
    err = (got - want).abs()
    assert (err <= bound).all(), float((err / bound).max())
    assert float(err.norm() / want.norm()) < 2.0 ** -10  # and two roundings, of 2^-11 at most, on the whole


# two rows a step: rows of 44, 56, 57, 63 and 64 pixels; three: 33, 40 and 42; four: 24, 29 and 32 (all of LDS); rows cut into
# two, three, five and seven columns, the last one shorter: 65, 80, 90, 110, 128 and 256; eight and nine rows, heights that
# are no whole steps, images in one strip and in many, more workgroups than CUs
@pytest.mark.parametrize("shape", [(37, 219, 227), (40, 224, 224), (48, 173, 173), (64, 32, 256), (60, 36, 228), (21, 97, 250), (8, 253, 253), (300, 33, 256),
                                   (12, 180, 240), (60, 130, 129), (37, 219, 160), (70, 91, 168), (103, 77, 96), (300, 35, 115), (65, 125, 128),
                                   (20, 97, 260), (14, 120, 320), (10, 131, 357), (9, 130, 440), (8, 128, 512), (7, 64, 1024)])
def test_block(net, shape):
    m, first, second = net[:3]
    N, H, W = shape
    g = torch.Generator().manual_seed(N * 7919 + H * 131 + W)
    xd = (torch.rand((N, 3, H, W), generator=g) * 2 - 1).half().cuda()
    x, _ = _tap(m, xd, 0)
    got, rep = _tap(m, xd, 1)
    assert rep[TAG]["launches"] == 2
    _check(got, x, first, second)


@pytest.mark.parametrize("shape", [(37, 219, 227), (64, 32, 256), (8, 253, 253), (70, 91, 168), (103, 77, 96), (10, 131, 357), (7, 64, 1024)])
def test_second_block(net, shape):
    """Its input is what the first one leaves: two, three and four rows a step, rows in columns."""
    m, _, _, whole, first, second = net
    N, H, W = shape
    xd = (torch.rand((N, 3, H, W), generator=torch.Generator().manual_seed(N + H + W)) * 2 - 1).half().cuda()
    x, _ = _tap(m, xd, 1)
    got, rep = _tap(whole, xd, 1)
    assert rep[TAG]["launches"] == 2
    _check(got, x, first, second)


@pytest.mark.parametrize("shape", [(20, 99, 256), (70, 99, 160), (90, 99, 128), (20, 99, 310)])
def test_not_finite(net, shape):
    """What is not a number stays where the convolutions carry it: not beyond a strip, a row's end or an image."""
    m = net[0]
    N, H, W = shape
    x = torch.rand((N, 3, H, W), generator=torch.Generator().manual_seed(5)) * 2 - 1
    for n, yy, xx in [(0, 0, 0), (0, H - 1, W - 1), (1, 50, W - 1), (1, 24, 0), (2, 97, 100)]:
        x[n, 1, yy, xx] = float("nan")
    xd = x.half().cuda()
    t, _ = _tap(m, xd, 0)
    got, rep = _tap(m, xd, 1)
    assert rep[TAG]["launches"] == 2 and torch.isnan(t).any()
    nan = torch.isnan(t).any(dim=1, keepdim=True).double()
    for _ in range(4):
        nan = F.max_pool2d(nan, 3, 1, 1)
    keep = (nan == 0).expand_as(got)
    assert torch.isfinite(got[keep]).all() and keep.any()
    clean, _ = _tap(m, torch.nan_to_num(xd), 1)
    assert torch.equal(got[keep], clean[keep])


@pytest.mark.parametrize("shape", [(36, 224, 224), (100, 92, 92), (4, 64, 1028), (31, 160, 160), (7, 256, 256)])
def test_not_taken(net, shape):
    """Too few steps, rows too short and too long: two launches, as before."""
    m = net[0]
    _, rep = _tap(m, torch.rand((shape[0], 3, shape[1], shape[2]), device="cuda").half(), 1)
    assert TAG not in rep
