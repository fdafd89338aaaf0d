"""The image layer (image_pairs_kernel) where a workgroup walks several tiles: more tiles than workgroups, the last ones cut by the image."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Graph, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,F,C,N,H,W", [(6, 32, 3, 7, 390, 404), (6, 40, 1, 8, 388, 390), (3, 16, 3, 9, 386, 402), (3, 64, 4, 7, 400, 398)])
def test_runs_of_tiles(k, F, C, N, H, W):
    g = torch.Generator().manual_seed(k * F)
    w, b = (torch.randn((F, C, k, k), generator=g) * (2.0 / (C * k * k)) ** 0.5).half().float(), torch.randn(F, generator=g).half().float()  # (an fp16 graph holds its parameters in fp16)
    x = torch.randn((N, C, H, W), generator=g).half().float()
    pad = 2 if k == 6 else 1
    op = abi.graph_op(abi.OP_CONV, [0, -1], 1, F=F, K=k, stride=2, pad=pad, act=abi.ACT_NONE, w=0, bias=w.numel())
    net = Graph([op], C, np.concatenate([w.numpy().ravel(), b.numpy()]), abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = torch.from_numpy(np.ascontiguousarray(host(net(dev(x.numpy(), abi.F16)))).astype(np.float64))
        tags = list(abi.profile_report())
    finally:
        abi.profile_enable(False)
        net.close()
    assert any(t.startswith("conv_pairs<f16,%s" % ("6x3" if k == 6 else "3x2")) for t in tags), tags
    want = torch.nn.functional.conv2d(x.double(), w.double(), b.double(), stride=2, padding=pad)
    weight = torch.nn.functional.conv2d(x.double().abs(), w.double().abs(), stride=2, padding=pad)
    # half an ulp of the result, C k k + 1 additions in fp32
    room = want.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24 + (C * k * k + 1) * 2.0 ** -24 * (weight + 4)
    assert got.shape == want.shape and bool(((got - want).abs() <= room).all()), ((got - want).abs() / room).max()
