"""fp16 3x3 layers of 32 channels with their filters in registers (conv3x3_narrow.hip) against torch: images that end inside a tile,
filters that end inside a block of 32, tiles of one trip and of several, residuals before and after nothing else, NaN and infinities."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, dev, host, nchw, nhwc

pytestmark = pytest.mark.gpu

# N, F, H, W, stride, form
CASES = [(3, 8, 126, 181, 1, "s1,32"), (13, 24, 114, 31, 1, "s1,32"), (16, 32, 161, 160, 1, "s1,32"), (8, 64, 65, 162, 1, "s1,64"),
         (9, 40, 151, 149, 1, "s1,64"), (6, 64, 318, 310, 2, "s2,64"), (16, 56, 206, 254, 2, "s2,64")]


@pytest.mark.parametrize("act", [abi.ACT_NONE, abi.ACT_RELU, abi.ACT_SILU])
@pytest.mark.parametrize("case", CASES, ids=lambda c: c[5] + "-" + "x".join(map(str, c[:5])))
def test_against_torch(case, act):
    N, F, H, W, st, form = case
    g = torch.Generator(device="cuda").manual_seed(H)
    x = torch.randn((N, 32, H, W), generator=g, device="cuda").half()
    w = (torch.randn((F, 32, 3, 3), generator=g, device="cuda") * (2.0 / 288) ** 0.5).half()
    x[0, 3, 0, 0], x[N - 1, 31, H - 1, W - 1], x[N - 1, 0, H // 2, W // 2] = float("inf"), float("nan"), float("-inf")
    xc, wc = x.cpu().double(), w.cpu().double()
    want = torch.nn.functional.conv2d(xc, wc, stride=st, padding=1)
    weight = torch.nn.functional.conv2d(xc.abs().nan_to_num(0, 0, 0), wc.abs(), stride=st, padding=1)
    r = torch.randn(want.shape, generator=torch.Generator().manual_seed(1)).half()
    f = {abi.ACT_NONE: lambda v: v, abi.ACT_RELU: torch.relu, abi.ACT_SILU: torch.nn.functional.silu}[act]
    layer, xd, rd = Conv(abi.F16, w.float().cpu().numpy(), st, 1, relu=act), dev(nhwc(x.float().cpu().numpy()), abi.F16), dev(nhwc(r.float().numpy()), abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        plain, added = host(layer(xd, abi.NHWC)), host(layer(xd, abi.NHWC, residual=rd))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert tags == ["conv3x3_narrow<%s>" % form]
    for got, exact in ((plain, f(want)), (added, f(want + r.double()))):
        got = torch.from_numpy(np.ascontiguousarray(nchw(got))).double()
        fin = torch.isfinite(exact)
        # half an ulp of the result, 289 additions in fp32, an ulp or two of the sigmoid
        room = exact.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24 + 289 * 2.0 ** -24 * (weight + 4)
        assert bool(((got - exact).abs() <= room)[fin].all()), ((got - exact).abs() / room)[fin].max()
        if act != abi.ACT_SILU:  # (silu(-inf) is -inf * 0 here and in the other kernels)
            assert torch.equal(torch.isnan(got), torch.isnan(exact)) and torch.equal(got[torch.isinf(exact)], exact[torch.isinf(exact)])
