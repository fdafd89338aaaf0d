"""fp32 3x3 stride-1 layers through three-way bf16 splits (conv3x3_split.hip): every form at sizes where its tiles, slabs and filter
blocks end raggedly, against torch in 64 bits; infinities, NaN and values that round to infinity in bf16; slices of wider tensors
come with the graph tests."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, dev, host, nchw, nhwc

pytestmark = pytest.mark.gpu

# N, C, F, H, W, form: one slab of 32 channels and several, filters that end inside a block of 64 or 32, images that end inside a
# tile, several images a tile, rows cut into column tiles, fewer pixels than a tile
CASES = [(8, 32, 344, 53, 47, "4,1"), (15, 32, 480, 35, 17, "4,1"), (6, 64, 64, 58, 78, "2,2"), (25, 160, 152, 11, 22, "2,2"), (3, 128, 328, 51, 25, "2,2"),
         (12, 128, 200, 19, 13, "1,4"), (33, 96, 72, 31, 9, "1,4"), (5, 96, 456, 19, 13, "1,4"), (6, 256, 256, 15, 20, "1,4,half"),
         (4, 224, 256, 40, 7, "1,4,half"), (16, 512, 512, 7, 7, "1,4,half"), (5, 128, 128, 25, 17, "1,4,half"),
         # more workgroups on an XCD than it has CUs
         (17, 224, 152, 14, 19, "1,4"), (9, 512, 896, 8, 8, "1,4,half"),
         # whole blocks of filters for little more than half of the CUs
         (7, 256, 256, 15, 20, "1,4"), (5, 192, 440, 9, 25, "1,4")]


def layer_and_reference(case, seed, spoil=None):
    N, C, F, H, W, _ = case
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn((N, C, H, W), generator=g), torch.randn((F, C, 3, 3), generator=g) * (2.0 / (9 * C)) ** 0.5
    r = torch.randn((N, F, H, W), generator=g)
    if spoil:
        spoil(x, w)
    layer = Conv(abi.F32, w.numpy(), 1, 1, relu=False)
    args, res = (dev(nhwc(x.numpy()), abi.F32), abi.NHWC), dev(nhwc(r.numpy()), abi.F32)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = torch.from_numpy(np.ascontiguousarray(nchw(host(layer(*args, residual=res)))))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    return got, torch.nn.functional.conv2d(x.double(), w.double(), padding=1) + r.double(), tags


@pytest.mark.parametrize("case", CASES, ids=lambda c: c[5] + "-" + "x".join(map(str, c[:5])))
def test_every_form(case):
    got, want, tags = layer_and_reference(case, 1)
    assert tags == ["conv3x3_split<f32,%s>" % case[5]]
    err = ((got.double() - want).norm() / want.norm()).item()
    # 9 C / 16 additions of half an ulp at most in a row, as a random walk, and a few ulp at the end
    assert err < 2.0 ** -25 * (9 * case[1] / 48) ** 0.5 + 2.0 ** -24, err


@pytest.mark.parametrize("case", [CASES[2], CASES[8]], ids=lambda c: c[5])
def test_values_that_bf16_does_not_hold(case):
    N, C, F, H, W, _ = case

    def spoil(x, w):
        x[0, 3, 4, 5] = float("inf")
        x[1, 0, 0, 0] = float("nan")
        x[2, C - 1, H - 1, W - 1] = 3.4e38  # rounds to infinity in bf16
        w[5] *= 1e-3

    got, want, _ = layer_and_reference(case, 2, spoil)
    want32 = want.float()
    fin = torch.isfinite(want32)
    assert torch.equal(torch.isnan(got), torch.isnan(want32))
    assert torch.equal(got[torch.isinf(want32)], want32[torch.isinf(want32)])
    large = fin & (want.abs() > 1e6)
    assert large.any() and ((got[large].double() - want[large]).abs() <= 1e-5 * want[large].abs()).all()
    rest = fin & ~large
    assert ((got[rest].double() - want[rest]).norm() / want[rest].norm()).item() < 1e-6
