"""fp32 down-sampling blocks whose 1x1 shortcut runs inside the launch of their 3x3 stride-2 convolution (conv_direct.hip): each tile that comes up, with the
shortcut behind it and in workgroups of its own, the last and the first launch of the line at 200 tiles, pixel counts that end inside a tile; against 64 bits."""
import ctypes
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from nncv_amd import abi, resnet18_spec, synth
from gpu_util import Model

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


@pytest.fixture(scope="module")
def net():
    """fp32 ResNet-18 whose second blocks hand their input on (the scale and shift behind their sums are zero), and its tensors."""
    blob, parts, at = synth.resnet18_params(), {}, 0
    for name, shape in resnet18_spec.tensor_table():
        n = math.prod(shape)
        if name in ["layer%d.1.bn2.%s" % (k, v) for k in (2, 3, 4) for v in ("weight", "bias")]:
            blob[at:at + n] = 0
        parts[name] = torch.from_numpy(blob[at:at + n].reshape(shape).astype(np.float64))
        at += n
    return Model(blob, abi.F32), parts


def _tap(m, x, stage, C, h, w):
    N, _, H, W = x.shape
    logits = torch.empty((N, 1000), dtype=torch.float32, device="cuda")
    tap = torch.full((N, h, w, C), float("nan"), dtype=torch.float32, device="cuda")
    abi.check(abi.lib().nncv_hip_resnet18_forward_tap(m.h, x.data_ptr(), N, H, W, logits.data_ptr(), stage, tap.data_ptr(), None))
    torch.cuda.synchronize()
    return tap


def _conv(x, error, w, bn, stride, pad):
    """The convolution under its BatchNorm, the magnitudes behind each value and a bound on its error where the input's is `error`: every order of
    K rounded additions and products, pieces that a split leaves out and BatchNorm's own roundings among them, is within (K + 16) 2^-24 of the magnitudes."""
    g, b, mean, var = bn
    s = g / (var + 1e-5).sqrt()
    y = F.conv2d(x, w, stride=stride, padding=pad) * s.view(1, -1, 1, 1) + (b - mean * s).view(1, -1, 1, 1)
    through = lambda v: F.conv2d(v, w.abs(), stride=stride, padding=pad) * s.abs().view(1, -1, 1, 1)
    size = through(x.abs()) + (b.abs() + mean.abs() * s.abs()).view(1, -1, 1, 1)
    return y, (w[0].numel() + 16) * U * size + (through(error) if error is not None else 0)


@pytest.mark.parametrize("case", [  # stage, images, rows of pixels, the tile, its number, behind
    (2, 9, 41, 49, (16, 16, 4), 192, 0), (2, 13, 33, 41, (16, 16, 4), 200, 1), (2, 13, 89, 33, (32, 16, 8), 196, 0), (2, 7, 145, 41, (32, 16, 8), 200, 1),
    (2, 20, 323, 33, (32, 32, 4), 516, 1), (2, 20, 65, 82, (32, 32, 8), 248, 1), (2, 37, 129, 33, (64, 32, 4), 198, 0), (2, 13, 41, 321, (64, 32, 4), 200, 1),
    (2, 101, 224, 224, (64, 64, 1), 2476, 1), (3, 20, 35, 33, (16, 16, 16), 192, 0), (3, 13, 65, 33, (16, 16, 16), 208, 1), (3, 9, 33, 209, (32, 16, 8), 192, 0),
    (3, 13, 33, 145, (32, 16, 8), 200, 1), (3, 37, 33, 209, (64, 32, 4), 196, 0), (3, 13, 161, 162, (64, 32, 4), 200, 1), (4, 7, 33, 161, (16, 16, 16), 192, 0),
    (4, 13, 99, 33, (16, 16, 16), 224, 1), (4, 13, 33, 198, (32, 16, 8), 192, 0), (4, 20, 34, 129, (32, 16, 8), 208, 1), (4, 9, 225, 321, (64, 32, 4), 200, 1)],
    ids=lambda c: "layer%d-%dx%dx%d" % c[:4])
def test_block(net, case):
    m, parts = net
    stage, N, H, W, tile, tiles, behind = case
    half = lambda v: (v - 1) // 2 + 1
    h, w = half(half(H)), half(half(W))
    for _ in range(stage - 2):
        h, w = half(h), half(w)
    C = 32 << (stage - 1)
    p = (ctypes.c_int * 5)()
    assert abi.lib().nncv_hip_conv_shortcut_plan(N, h, w, C, 2 * C, p) == 0 and tuple(p) == tile + (tiles, behind), tuple(p)
    print(case, flush=True)
    xd = torch.rand((N, 3, H, W), generator=torch.Generator(device="cuda").manual_seed(stage * 1000 + H), device="cuda") * 2 - 1
    x, got = _tap(m, xd, stage - 1, C, h, w), _tap(m, xd, stage, 2 * C, half(h), half(w))
    pick = torch.tensor(sorted({0, 1, N // 2, N - 2, N - 1}) if N > 20 else range(N), device="cuda")
    x, got = (t[pick].cpu().double().permute(0, 3, 1, 2) for t in (x, got))
    of = lambda name, bn: (parts["layer%d.0.%s.weight" % (stage, name)], [parts["layer%d.0.%s.%s" % (stage, bn, v)] for v in ("weight", "bias", "running_mean", "running_var")])
    y, e = _conv(x, None, *of("conv1", "bn1"), 2, 1)
    y = torch.relu(y)
    z, ez = _conv(y, e, *of("conv2", "bn2"), 1, 1)
    s, es = _conv(x, None, *of("downsample.0", "downsample.1"), 2, 0)
    want = torch.relu(z + s)
    bound = ez + es + U * (z.abs() + s.abs())
    err = (got - want).abs()
    assert torch.isfinite(got).all() and (err <= bound).all(), float((err / bound).max())
    # and without the worst case: roundings of half an ulp of a sum at most, one for each product, as a random walk
    assert float(err.norm() / want.norm()) < (27 * C) ** 0.5 * 2.0 ** -24
