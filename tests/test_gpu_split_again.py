"""fp32 kernels on the bf16 matrix pipes (split.hpp) where a wave's sums are not finite and it takes them again with the fp32 instructions:
every form with every wave doing so, at sizes that end inside tiles, and what such a call takes."""
import numpy as np
import pytest
import torch

import oracle
from nncv_amd import abi, synth
from gpu_util import Conv, Model, dev, host, max_rel, nchw, nhwc
from test_gpu_conv3x3_split import CASES
from test_gpu_gemm_split import SHAPES, operands, product

pytestmark = pytest.mark.gpu

HUGE = 3.4e38  # infinity in bf16: a sum with it in is a NaN there, whatever it is multiplied by

# N, C, F, H, W, R, stride, pad, tag.  Taps of whole rounds and others, blocks of 128 x 128 and 256 x 64, windows over the border
LAYERS = [(N, C, F, H, W, 3, 1, 1, "conv3x3_split<f32,%s>" % form) for N, C, F, H, W, form in CASES] + [
    (7, 96, 108, 24, 42, 3, 1, 1, "conv3x3_direct<f32,64x32,splitk4>"), (12, 88, 108, 35, 17, 3, 1, 1, "conv3x3_direct<f32,64x32,splitk4>"),
    (6, 64, 128, 58, 78, 3, 2, 1, "conv3x3_direct<f32,64x32,splitk4>"),
    (23, 128, 128, 88, 24, 1, 1, 0, "igemm_fast<f32,f32,2,2,1,1,split>"), (13, 16, 128, 95, 29, 5, 1, 2, "igemm_fast<f32,f32,2,2,1,1,split>"),
    (43, 16, 60, 22, 89, 5, 1, 2, "igemm_fast<f32,f32,4,1,1,1,split>")]


def relative(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("M,N,K,form", SHAPES)
def test_every_product(M, N, K, form):
    a, b, c = operands(M, N, K)
    a[:, 5], b[5] = HUGE, 0.0
    got, tags = product(a, b, c)
    assert tags == ["gemm_split<%s>" % form]
    # K roundings of half an ulp in a row, as a random walk: 2^-25 sqrt(K / 3) with products of both signs, twice that allowed
    assert relative(got, c.double() + a.double() @ b.double()) < 2.0 ** -24 * (K / 3) ** 0.5


def layer_of(case, seed):
    N, C, F, H, W, R, stride, pad, _ = case
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn((N, C, H, W), generator=g), torch.randn((F, C, R, R), generator=g) * (2.0 / (R * R * C)) ** 0.5
    return x, w


@pytest.mark.parametrize("case", LAYERS, ids=lambda c: c[8] + "-" + "x".join(map(str, c[:5])))
def test_every_layer(case):
    N, C, F, H, W, R, stride, pad, tag = case
    x, w = layer_of(case, 3)
    x[:, C // 2], w[:, C // 2] = HUGE, 0.0
    pick = sorted({0, N // 2, N - 1})
    want = torch.nn.functional.conv2d(x[pick].double(), w.double(), stride=stride, padding=pad)
    r = torch.randn((N,) + tuple(want.shape[1:]), generator=torch.Generator().manual_seed(4))
    layer = Conv(abi.F32, w.numpy(), stride, pad)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = nchw(host(layer(dev(nhwc(x.numpy()), abi.F32), abi.NHWC, residual=dev(nhwc(r.numpy()), abi.F32))))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
    assert tags == [tag]
    assert relative(torch.from_numpy(np.ascontiguousarray(got))[pick], want + r[pick].double()) < 2.0 ** -24 * (R * R * C / 3) ** 0.5


def microseconds(call, n=10):
    call()
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    e[0].record()
    for _ in range(n):
        call()
    e[1].record()
    torch.cuda.synchronize()
    return e[0].elapsed_time(e[1]) * 1e3 / n


# Every wave walks twice, the second time at a third of the rate and with its operands one step of eight k ahead: 2 to 4 times the usual.  (One
# lane a sum, one k after the other, took 10 to 90 times.)
SLOWEST = 8


@pytest.mark.parametrize("M,N,K", [(1023, 1023, 1001), (2207, 2747, 3233), (1499, 1002, 778)])
def test_a_product_of_nan_is_not_much_slower(M, N, K):
    a, b, c = (t.cuda() for t in operands(M, N, K))
    s = torch.cuda.current_stream().cuda_stream
    call = lambda m: abi.check(abi.lib().nncv_hip_matmul_f32(m.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, s))
    usual = microseconds(lambda: call(a))
    nan = torch.full_like(a, float("nan"))
    assert microseconds(lambda: call(nan)) < SLOWEST * usual
    assert torch.isnan(c).all()


@pytest.mark.parametrize("case", [LAYERS[2], LAYERS[8], LAYERS[10], LAYERS[-5], LAYERS[-3], LAYERS[-1]], ids=lambda c: c[8])
def test_a_layer_of_nan_is_not_much_slower(case):
    N, C, F, H, W, R, stride, pad, _ = case
    x, w = layer_of(case, 5)
    layer, xd = Conv(abi.F32, w.numpy(), stride, pad), dev(nhwc(x.numpy()), abi.F32)
    out = torch.empty((N, (H + 2 * pad - R) // stride + 1, (W + 2 * pad - R) // stride + 1, F), device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    call = lambda: abi.check(abi.lib().nncv_hip_conv_forward(layer.h, xd.data_ptr(), N, H, W, abi.NHWC, None, out.data_ptr(), s))
    usual = microseconds(call)
    xd.fill_(float("nan"))
    assert microseconds(call) < SLOWEST * usual
    assert torch.isnan(out).all()


def test_a_network_whose_sums_are_large():
    """An fp32 ResNet-18 with one pixel of 3e31: the sums around it are above 2^80 from the first layer on, so every kernel on the bf16 pipes, the
    shortcuts inside the stride-2 layers among them, takes them again; against the oracle, image by image."""
    blob = synth.resnet18_params()
    x = synth.uniform(77, (6, 3, 231, 309), 0.0, 1.0)
    x[2, 1, 100, 140] = 3e31
    m = Model(blob, abi.F32)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(m(dev(x, abi.F32)))
        tags = abi.profile_report()
    finally:
        abi.profile_enable(False)
    assert tags["conv3x3_direct<f32,64x32,splitk4>"]["launches"] == 2 and any(t.startswith("conv3x3_split<") for t in tags), list(tags)
    want = oracle.hwp_resnet18_forward(x, blob)
    assert np.isfinite(want).all() and np.abs(want[2]).max() > 2.0 ** 100
    for i in range(6):
        assert max_rel(got[i], want[i]) < 1e-5  # 20 layers of fp32 sums, each off by 1e-6 of its largest at most; 3e-7 where none is taken again
