"""fp32 products through three-way bf16 splits (gemm_split.hip): every form at sizes one off its tiles and rounds, against
64 bits, with the error of the fp32 instructions as the bar; infinities, NaN and values that round to infinity in bf16."""
import pytest
import torch

from nncv_amd import abi

pytestmark = pytest.mark.gpu


def product(a, b, c):
    (M, K), N = a.shape, b.shape[1]
    ad, bd, d = a.cuda(), b.cuda(), c.cuda()
    abi.profile_enable(True)
    try:
        abi.profile_report()
        abi.check(abi.lib().nncv_hip_matmul_f32(ad.data_ptr(), bd.data_ptr(), d.data_ptr(), M, N, K, None))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    return d.cpu(), tags


def operands(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    return tuple(torch.randn(s, generator=g) for s in ((M, K), (K, N), (M, N)))


SHAPES = [(1023, 1023, 1001, "64x64,splitk8"), (673, 1377, 833, "64x64,splitk8"), (2207, 2747, 3233, "64x64,splitk4"),
          (3260, 2201, 383, "64x64"), (3999, 4001, 385, "64x64"), (179, 2227, 1735, "32x64,splitk8"), (2390, 190, 1057, "32x64,splitk8"),
          (1499, 1002, 778, "32x64,splitk4"), (193, 3199, 353, "32x64,splitk4")]


@pytest.mark.parametrize("M,N,K,form", SHAPES)
def test_every_form(M, N, K, form):
    a, b, c = operands(M, N, K)
    got, tags = product(a, b, c)
    assert tags == ["gemm_split<%s>" % form]
    want = c.double() + a.double() @ b.double()
    err = ((got.double() - want).norm() / want.norm()).item()
    # K / 16 additions of half an ulp at most in a row, each wave's part of them, and a few ulp at the end: as a random walk
    # 2^-25 sqrt(K / 16 / 3), plus 2^-24
    assert err < 2.0 ** -25 * (K / 48) ** 0.5 + 2.0 ** -24, err


@pytest.mark.parametrize("M,N,K", [(1023, 1025, 1001), (179, 2227, 1735), (1023, 1023, 1001)])
def test_values_that_bf16_does_not_hold(M, N, K):
    a, b, c = operands(M, N, K)
    a[3, 5] = float("inf")
    a[M - 1, K - 1] = float("nan")
    b[7, N - 1] = -float("inf")
    a[40, 1] = 3.4e38  # rounds to infinity in bf16
    b[1, :] *= 1e-3
    got, tags = product(a, b, c)
    assert tags[0].startswith("gemm_split")
    want = c.double() + a.double() @ b.double()
    fin = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)].float())
    rows = torch.ones(M, dtype=torch.bool)
    rows[40] = False  # (its own scale)
    for r in (rows, ~rows):
        g, w = got[r][fin[r]].double(), want[r][fin[r]]
        assert ((g - w).norm() / w.norm()).item() < 2e-6 * (K / 4096) ** 0.5 + 2.0 ** -24
