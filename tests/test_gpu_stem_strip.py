"""The stem kernels (7x7 stride 2 + BN + ReLU + 3x3 stride 2 maximum, stem_pool.hip and stem_pool_split.hip) where their strips and walks
end: the pooled activation against the same layer in 64 bits."""
import math
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from nncv_amd import abi, resnet18_spec, synth
from gpu_util import Model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[abi.F16, abi.F32], ids=["f16", "f32"])
def net(request):
    blob = synth.resnet18_params()
    if request.param == abi.F16:
        blob = synth.round_fp16(blob)
    m = Model(blob, request.param)
    parts, at = [], 0
    for _, shape in resnet18_spec.tensor_table()[:5]:
        n = math.prod(shape)
        parts.append(torch.from_numpy(blob[at:at + n].reshape(shape).astype(np.float64)))
        at += n
    return m, parts, torch.float16 if request.param == abi.F16 else torch.float32


def _pooled(m, x, shift=0):
    N, _, H, W = x.shape
    ph, pw = ((H - 1) // 2) // 2 + 1, ((W - 1) // 2) // 2 + 1
    buf = torch.empty(x.numel() + shift, dtype=x.dtype, device="cuda")
    buf[shift:] = x.reshape(-1).cuda()
    logits = torch.empty((N, 1000), dtype=torch.float32, device="cuda")
    tap = torch.full((N, ph, pw, 64), float("nan"), dtype=x.dtype, device="cuda")
    abi.profile_enable(True)
    try:
        abi.profile_report()
        abi.check(abi.lib().nncv_hip_resnet18_forward_tap(m.h, buf[shift:].data_ptr(), N, H, W, logits.data_ptr(), 0, tap.data_ptr(), None))
        torch.cuda.synchronize()
        assert any(t.startswith("stem_conv7x7_bn_relu_maxpool<") for t in abi.profile_report())
    finally:
        abi.profile_enable(False)
    return tap.cpu().permute(0, 3, 1, 2)


def _want(x, parts):
    w, g, b, mean, var = parts
    y = torch.nn.functional.conv2d(x.double(), w, stride=2, padding=3)
    y = torch.nn.functional.batch_norm(y, mean, var, g, b, eps=1e-5)
    return torch.nn.functional.max_pool2d(torch.relu(y), 3, 2, 1)


def _terms(x, parts):
    """The largest sum of magnitudes behind a pooled value."""
    w, g, b, mean, var = parts
    s = g.abs() / (var + 1e-5).sqrt()
    y = torch.nn.functional.conv2d(x.double().abs(), w.abs(), stride=2, padding=3) * s.view(1, -1, 1, 1) + (b.abs() + mean.abs() * s).view(1, -1, 1, 1)
    return torch.nn.functional.max_pool2d(y, 3, 2, 1)


# pooled widths of 15, 16, 30 and 31 (a strip holds 15), of one strip's first column; even and odd convolution heights and widths (the last
# window's row and column then lie outside), odd image widths (fp16: pixels through registers), images of which a wave walks
# several (more strips than waves) and parts of one
@pytest.mark.parametrize("shape", [(1, 32, 60), (1, 34, 64), (2, 33, 61), (3, 35, 59), (1, 70, 118), (1, 71, 121), (2, 37, 122), (5, 32, 33),
                                   (1100, 32, 32), (700, 32, 63), (1, 320, 34), (40, 97, 131)])
@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "one_element_off"])
def test_pooled_activation(net, shape, shift):
    m, parts, dtype = net
    N, H, W = shape
    g = torch.Generator().manual_seed(N * 7919 + H * 131 + W)
    x = (torch.rand((N, 3, H, W), generator=g) * 2 - 1).to(dtype)
    want = _want(x, parts)
    got = _pooled(m, x, shift).double()
    # fp16: one rounding to 11 bits; before it, and for fp32, a sum of 147 products in steps of 16, each rounded to 24 bits, the products that the
    # three pieces leave out (2^-24) and the two roundings of BN
    err = (got - want).abs()
    bound = 16 * 2.0 ** -24 * _terms(x, parts) + (want.abs() * 2.0 ** -11 if dtype == torch.float16 else 0)
    assert torch.isfinite(got).all()
    assert (err <= bound).all(), float((err / bound).max())


def test_fp32_sums_taken_again(net):
    """Pixels whose products bf16 pieces do not hold: NaN, infinities (in even columns too: the padding's zero weight is not multiplied then) and
    values whose sums leave the range of the split ones."""
    m, parts, dtype = net
    if dtype != torch.float32:
        pytest.skip("fp16 sums are not split")
    x = torch.rand((2, 3, 101, 133), generator=torch.Generator().manual_seed(3)) * 2 - 1
    for n, c, y, xx, v in [(0, 0, 0, 0, np.nan), (0, 1, 50, 62, np.nan), (0, 2, 100, 132, np.nan), (1, 0, 10, 20, np.inf), (1, 1, 61, 65, -np.inf),
                           (1, 2, 90, 100, 3.4e38), (0, 0, 30, 120, 2e31)]:
        x[n, c, y, xx] = float(v)
    want, got = _want(x, parts).float(), _pooled(m, x)
    assert torch.isnan(want).any() and torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    fin = torch.isfinite(want)
    t = _terms(x, parts)
    assert ((got.double() - want.double()).abs()[fin] <= 147 * 2.0 ** -24 * t[fin]).all()


SEPARATE = """
import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, FP32_MAX_REL, Model, dev, host, max_rel, rel_l2
for dt in (abi.F32, abi.F16):
    half = synth.round_fp16 if dt == abi.F16 else (lambda v: v)
    blob = half(synth.resnet18_params())
    m = Model(blob, dt)
    for shape in [(2, 3, 66, 64), (3, 3, 33, 47)]:
        x = half(synth.uniform(91, shape, 0.0, 1.0))
        abi.profile_enable(True)
        abi.profile_report()
        got = host(m(dev(x, dt)))
        tags = list(abi.profile_report())
        abi.profile_enable(False)
        assert any(t.startswith("maxpool") for t in tags) and not any(t.startswith("stem_conv7x7_bn_relu_maxpool") for t in tags), tags
        want = oracle.resnet18_forward(x, blob)
        err = max_rel(got, want) if dt == abi.F32 else rel_l2(got, want)
        assert err < (FP32_MAX_REL if dt == abi.F32 else FP16_REL_L2), (dt, shape, err)
        print(dt, shape, err, flush=True)
"""


def test_the_stem_as_separate_launches():
    """Packing, implicit GEMM and pool: what images of 2 GB in all and more, beyond the fused kernels' range, still take; here by its switch, which a process
    reads once."""
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, NNCV_HIP_NO_STEM_FUSION="1", PYTHONPATH=os.pathsep.join([here, os.path.dirname(here)]))
    r = subprocess.run([sys.executable, "-c", SEPARATE], env=env, capture_output=True, text=True, timeout=100)
    print(r.stdout, flush=True)
    assert r.returncode == 0, r.stderr[-2000:]
