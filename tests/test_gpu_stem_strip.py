"""The fp16 stem kernel (7x7 stride 2 + BN + ReLU + 3x3 stride 2 maximum, stem_pool.hip) where its strips and walks end: the
pooled activation against the same layer in 64 bits."""
import math

import numpy as np
import pytest
import torch

from nncv_amd import abi, resnet18_spec, synth
from gpu_util import Model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    blob = synth.round_fp16(synth.resnet18_params())
    m = Model(blob, abi.F16)
    parts, at = [], 0
    for _, shape in resnet18_spec.tensor_table()[:5]:
        n = math.prod(shape)
        parts.append(torch.from_numpy(blob[at:at + n].reshape(shape).astype(np.float64)))
        at += n
    return m, parts


def _want(x, parts):
    w, g, b, mean, var = parts
    y = torch.nn.functional.conv2d(x.double(), w, stride=2, padding=3)
    y = torch.nn.functional.batch_norm(y, mean, var, g, b, eps=1e-5)
    return torch.nn.functional.max_pool2d(torch.relu(y), 3, 2, 1)


# pooled widths of 15, 16, 30 and 31 (a strip holds 15), of one strip's first column; even and odd convolution heights and widths (the last
# window's row and column then lie outside), odd image widths (pixels through registers), images of which a wave walks
# several (more strips than waves) and parts of one
@pytest.mark.parametrize("shape", [(1, 32, 60), (1, 34, 64), (2, 33, 61), (3, 35, 59), (1, 70, 118), (1, 71, 121), (2, 37, 122), (5, 32, 33),
                                   (1100, 32, 32), (700, 32, 63), (1, 320, 34), (40, 97, 131)])
@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "one_element_off"])
def test_pooled_activation(net, shape, shift):
    m, parts = net
    N, H, W = shape
    g = torch.Generator().manual_seed(N * 7919 + H * 131 + W)
    x = (torch.rand((N, 3, H, W), generator=g) * 2 - 1).half()
    want = _want(x, parts)
    ph, pw = want.shape[2:]
    buf = torch.empty(x.numel() + shift, dtype=torch.float16, device="cuda")
    buf[shift:] = x.reshape(-1).cuda()
    logits = torch.empty((N, 1000), dtype=torch.float32, device="cuda")
    tap = torch.full((N, ph, pw, 64), float("nan"), dtype=torch.float16, device="cuda")
    abi.check(abi.lib().nncv_hip_resnet18_forward_tap(m.h, buf[shift:].data_ptr(), N, H, W, logits.data_ptr(), 0, tap.data_ptr(), None))
    torch.cuda.synchronize()
    got = tap.cpu().double().permute(0, 3, 1, 2)
    # one rounding to 11 bits of the value; before it a sum of 147 products, of values up to some tens, in fp32 (2^-24 each)
    err = (got - want).abs()
    bound = want.abs() * 2.0 ** -11 + 147 * 2.0 ** -24 * 16
    assert torch.isfinite(got).all()
    assert (err <= bound * 1.01).all(), float((err / bound).max())
