"""fp32 kernels on the bf16 matrix pipes (split.hpp) over the whole range of fp32: operands down to the subnormal numbers and up to
where sums are large, values of very different size in one sum, sums that one product is all of; each kernel, against 64 bits, with the error of ordinary operands as the bar."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, dev, host, nchw, nhwc
from test_gpu_gemm_split import operands, product
from test_gpu_split_again import relative

pytestmark = pytest.mark.gpu

# powers of two on the one operand and the other: small ones and subnormal ones with products near 1 and at 2^-40, both small; large
# operands, and sums that the scaled products do not hold (those are taken again with the fp32 instructions)
SCALES = [(-100, 100), (-112, 95), (-118, 95), (-126, 90), (-135, 95), (95, -112), (95, -118), (90, -126), (95, -135), (-60, -60), (60, 10),
          (-118, 110), (-126, 120), (-135, 120), (110, -118), (120, -126), (120, -135), (60, 30), (45, 60)]


def taken_again(sa, sb):
    return sa + sb > 72 or max(sa, sb) > 100


def bar(K):  # fp32 instructions: half an ulp for every k, as a random walk, twice that allowed
    return 2.0 ** -24 * (K / 3) ** 0.5 + 2.0 ** -24


def split_bar(K):  # as in the kernels' own tests: half an ulp for every 16 k
    return 2.0 ** -25 * (K / 48) ** 0.5 + 2.0 ** -24


@pytest.mark.parametrize("sa,sb", SCALES)
@pytest.mark.parametrize("M,N,K", [(1023, 1023, 1001), (1499, 1002, 778)])
def test_product(M, N, K, sa, sb):
    a, b, _ = operands(M, N, K)
    a, b = torch.ldexp(a, torch.tensor(sa)), torch.ldexp(b, torch.tensor(sb))
    got, tags = product(a, b, torch.zeros(M, N))
    assert tags[0].startswith("gemm_split")
    scale = 2.0 ** -(sa + sb)
    assert relative(got.double() * scale, (a.double() @ b.double()) * scale) < (bar(K) if taken_again(sa, sb) else split_bar(K))


LAYERS = [(6, 64, 64, 29, 39, 3, 1, 1, "conv3x3_split<f32"), (6, 256, 256, 15, 20, 3, 1, 1, "conv3x3_split<f32"), (6, 64, 128, 58, 78, 3, 2, 1, "conv3x3_direct<f32,64x32"),
          (23, 128, 128, 88, 24, 1, 1, 0, "igemm_fast<f32,f32,2,2"), (43, 16, 60, 22, 89, 5, 1, 2, "igemm_fast<f32,f32,4,1")]


def layer(case, x, w):
    N, C, F, H, W, R, stride, pad, tag = case
    conv = Conv(abi.F32, w.numpy(), stride, pad)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = torch.from_numpy(np.ascontiguousarray(nchw(host(conv(dev(nhwc(x.numpy()), abi.F32), abi.NHWC)))))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert len(tags) == 1 and tags[0].startswith(tag), tags
    return got


def values(case, seed):
    N, C, F, H, W, R, stride, pad, _ = case
    g = torch.Generator().manual_seed(seed)
    return torch.randn((N, C, H, W), generator=g), torch.randn((F, C, R, R), generator=g) * (2.0 / (R * R * C)) ** 0.5


@pytest.mark.parametrize("sx,sw", SCALES)
@pytest.mark.parametrize("case", LAYERS, ids=lambda c: c[8])
def test_layer(case, sx, sw):
    N, C, F, H, W, R, stride, pad, _ = case
    x, w = values(case, 6)
    x, w = torch.ldexp(x, torch.tensor(sx)), torch.ldexp(w, torch.tensor(sw))
    got = layer(case, x, w)
    scale, pick = 2.0 ** -(sx + sw), [0, N - 1]
    want = torch.nn.functional.conv2d(x[pick].double(), w.double(), stride=stride, padding=pad) * scale
    assert relative(got[pick].double() * scale, want) < (bar(R * R * C) if taken_again(sx, sw) else split_bar(R * R * C))


# A sum that is one product: two dropped products of 2^-8 x 2^-17 at most, and a rounding of 2^-24
LONE = 2.0 ** -23 * 1.01


def test_a_product_that_is_a_sum_of_its_own():
    M, N, K = 1499, 1002, 778
    g = torch.Generator().manual_seed(8)
    a, b = torch.zeros(M, K), torch.rand((K, N), generator=g) + 1
    col = torch.arange(M) % K
    a[torch.arange(M), col] = torch.rand(M, generator=g) + 1
    got, tags = product(a, b, torch.zeros(M, N))
    assert tags[0].startswith("gemm_split")
    want = a[torch.arange(M), col].double().view(M, 1) * b[col].double()
    assert ((got.double() - want).abs() / want).max().item() < LONE


@pytest.mark.parametrize("case", LAYERS, ids=lambda c: c[8])
def test_a_filter_of_one_weight(case):
    N, C, F, H, W, R, stride, pad, _ = case
    g = torch.Generator().manual_seed(9)
    x, w = torch.rand((N, C, H, W), generator=g) + 1, torch.zeros(F, C, R, R)
    f = torch.arange(F)
    w[f, f % C, R // 2, R // 2] = torch.rand(F, generator=g) + 1
    want = x[:, f % C, ::stride, ::stride].double() * w[f, f % C, R // 2, R // 2].double().view(1, F, 1, 1)
    assert ((layer(case, x, w).double() - want).abs() / want).max().item() < LONE


@pytest.mark.parametrize("case", LAYERS, ids=lambda c: c[8])
def test_sizes_that_meet_in_one_sum(case):
    """A pixel whose large channels meet small filters and whose small channels meet large ones: every product counts."""
    N, C, F, H, W, R, stride, pad, _ = case
    x, w = values(case, 7)
    s = torch.where(torch.arange(C) % 2 == 0, -120, 0)
    x, w = torch.ldexp(x, s.view(1, C, 1, 1)), torch.ldexp(w, -120 - s.view(1, C, 1, 1))
    got, pick = layer(case, x, w), [0, N - 1]
    want = torch.nn.functional.conv2d(x[pick].double(), w.double(), stride=stride, padding=pad)
    # (results near 2^-120: an ulp of theirs ends at 2^-149)
    assert relative(got[pick], want) < split_bar(R * R * C)
