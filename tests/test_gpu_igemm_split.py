"""fp32 implicit GEMMs on the bf16 matrix pipes (igemm_fast.hip): blocks of 128 x 128 and 256 x 64, one, two and many steps of 16 k,
pixels and filters that end inside a block, windows over the border, residual and activation; against 64 bits, and what infinities,
NaNs and values that bf16 does not hold become, against fp32 on the CPU."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, dev, host, nchw, nhwc, rel_l2

pytestmark = pytest.mark.gpu


def run(x, w, stride, pad, relu=False, res=None):
    layer = Conv(abi.F32, w.numpy(), stride, pad, relu=abi.ACT_RELU if relu else abi.ACT_NONE)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        y = nchw(host(layer(dev(nhwc(x.numpy()), abi.F32), abi.NHWC, residual=None if res is None else dev(nhwc(res.numpy()), abi.F32))))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    return y, tags


# the rounding of fp32 sums of K products is at most K / 2 of 2^-24 a term, sqrt(K) of it in L2; three pieces drop products below 2^-24
@pytest.mark.parametrize("N,C,F,H,W,R,stride,pad,tag", [
    (23, 128, 128, 88, 24, 1, 1, 0, "2,2,1,1"), (13, 16, 128, 95, 29, 5, 1, 2, "2,2,1,1"), (19, 16, 128, 111, 21, 3, 1, 1, "2,2,1,1"),
    (43, 16, 60, 22, 89, 5, 1, 2, "4,1,1,1"), (9, 32, 64, 85, 87, 1, 1, 0, "4,1,1,1"), (6, 48, 64, 107, 109, 1, 1, 0, "4,1,1,1")])
def test_matches_double(N, C, F, H, W, R, stride, pad, tag):
    g = torch.Generator().manual_seed(C * F + R)
    x, w = torch.randn((N, C, H, W), generator=g), torch.randn((F, C, R, R), generator=g) * (2.0 / (R * R * C)) ** 0.5
    pick = [0, N // 2, N - 1]
    want = torch.nn.functional.conv2d(x[pick].double(), w.double(), stride=stride, padding=pad)
    res = torch.randn((N, F) + tuple(want.shape[2:]), generator=g)
    got, tags = run(x, w, stride, pad)
    assert tags == ["igemm_fast<f32,f32,%s,split>" % tag], tags
    assert rel_l2(got[pick], want.numpy()) < 2.0 ** -24 * (R * R * C) ** 0.5
    got, _ = run(x, w, stride, pad, True, res)
    assert rel_l2(got[pick], torch.relu(want + res[pick].double()).numpy()) < 2.0 ** -24 * (R * R * C) ** 0.5


def test_not_finite():
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn((23, 64, 88, 24), generator=g), torch.randn((128, 64, 1, 1), generator=g)
    for i, v in enumerate([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38]):
        x[i, 3 * i, 5 + i, 7] = float(v)
    x[7, :, 9, 9] = 0.0
    w[5, 1], w[77, 63] = 3.4e38, float("inf")
    got, tags = run(x, w, 1, 0)
    assert tags == ["igemm_fast<f32,f32,2,2,1,1,split>"], tags
    want = torch.nn.functional.conv2d(x, w).numpy()
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    assert rel_l2(got[fin] / 1e30, want[fin] / 1e30) < 1e-5
