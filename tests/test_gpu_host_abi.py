"""The host-buffer entry points of the reference's ABI at the sizes where their staging changes form: one or several
bands of rows, pieces and ranges of images, operands above the staging limit, strided views, filter windows that do not
fit LDS; and the NCHW <-> NHWC re-laying kernel at the edges of its 64 x 64 tiles."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv, FP32_MAX_REL, FP16_REL_L2, dev, host, max_rel, rel_l2

pytestmark = pytest.mark.gpu


def rand(seed, *shape):
    return torch.rand(shape, generator=torch.Generator().manual_seed(seed)).mul_(2).sub_(1)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 5, 2), (130, 70, 900), (700, 600, 601), (1025, 1023, 513), (5, 2000, 2000), (3000, 17, 100),
                                   (3001, 3000, 1500)])
def test_matmul_on_host_memory(M, N, K):
    a, b, c = rand(1, M, K), rand(2, K, N), rand(3, M, N)
    want = c.double() + a.double() @ b.double()
    an, bn, cn = a.numpy(), np.asfortranarray(b.numpy()) if M == 130 else b.numpy(), c.numpy().copy()
    wide = np.zeros((M, N + 3), np.float32)  # a view with another row pitch
    wide[:, :N] = cn
    for got in (cn, wide[:, :N]):
        abi.matmul(an, bn, got)
        assert max_rel(got, want.numpy()) < FP32_MAX_REL
    assert (wide[:, N:] == 0).all()


@pytest.mark.parametrize("N,C,F,H,W,R,stride", [(1, 1, 1, 1, 1, 1, 1), (1, 64, 64, 58, 58, 3, 1), (5, 3, 7, 131, 67, 7, 2), (6, 33, 65, 66, 68, 3, 1),
                                                (2, 2, 3, 100, 99, 96, 1), (9, 40, 20, 203, 251, 3, 2)])
def test_convolution_on_host_memory(N, C, F, H, W, R, stride):
    x, w = rand(4, N, C, H, W), rand(5, F, C, R, R)
    oh, ow = (H - R) // stride + 1, (W - R) // stride + 1
    out = rand(6, N, F, oh, ow)
    want = out + torch.nn.functional.conv2d(x, w, stride=stride)
    got = out.numpy().copy()
    big = np.zeros((N, C, H + 1, W + 2), np.float32)
    big[:, :, 1:, 2:] = x.numpy()
    abi.batch_nchw_conv(big[:, :, 1:, 2:] if C == 33 else x.numpy(), w.numpy(), got)
    assert max_rel(got, want.numpy()) < FP32_MAX_REL


@pytest.mark.parametrize("dt", [abi.F32, abi.F16])
@pytest.mark.parametrize("N,C,F,H,W,res", [(2, 3, 5, 7, 9, False), (1, 64, 64, 8, 8, True), (3, 65, 63, 5, 13, True), (2, 128, 128, 21, 3, True), (4, 8, 16, 1, 1, False)])
def test_nchw_layer_at_the_edges_of_the_relayout_tiles(dt, N, C, F, H, W, res):
    x, w, r = rand(7, N, C, H, W), rand(8, F, C, 3, 3) * (2.0 / (9 * C)) ** 0.5, rand(9, N, F, H, W)
    if dt == abi.F16:
        x, w, r = x.half().float(), w.half().float(), r.half().float()
    want = torch.nn.functional.conv2d(x, w, padding=1) + (r if res else 0)
    got = host(Conv(dt, w.numpy(), 1, 1)(dev(x.numpy(), dt), abi.NCHW, residual=dev(r.numpy(), dt) if res else None))
    assert max_rel(got, want.numpy()) < FP32_MAX_REL if dt == abi.F32 else rel_l2(got, want.numpy()) < FP16_REL_L2
