"""Three chained 5x5 max-pools in one launch (maxpool5_chain3): NaN and infinities pass as through torch's pooling, at maps around the
block sizes and numbers of channel vectors that are no multiple of eight."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Graph, dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [abi.F32, abi.F16])
@pytest.mark.parametrize("N,C,H,W", [(1, 8, 1, 3), (3, 24, 16, 16), (5, 8, 17, 16), (2, 40, 32, 17), (1, 16, 40, 40)])
def test_special_values_pass_through_the_chain(dt, N, C, H, W):
    rng = np.random.default_rng(H * W)
    w = rng.standard_normal((C, 3)).astype(np.float16).astype(np.float32)
    x = rng.standard_normal((N, 3, H, W)).astype(np.float16).astype(np.float32)
    x[0, 1, 0, 0] = np.inf
    if H > 10:
        x[0, 0, H // 2, W // 3], x[N - 1, 2, H - 1, W - 1], x[0, :, 6, 6] = np.nan, -np.inf, -np.inf
    ops = [abi.graph_op(abi.OP_CONV, [0, -1], 1, F=C, K=1, stride=1, pad=0, act=abi.ACT_NONE, w=0, bias=3 * C)]
    ops += [abi.graph_op(abi.OP_MAXPOOL, [i], i + 1, K=5, stride=1, pad=2) for i in (1, 2, 3)]
    ops.append(abi.graph_op(abi.OP_CONCAT, [1, 2, 3, 4], 5))
    g = Graph(ops, 3, np.concatenate([w.ravel(), np.zeros(C, np.float32)]), dt)
    try:
        got = torch.from_numpy(np.ascontiguousarray(host(g(dev(x, dt)))).astype(np.float32))
    finally:
        g.close()
    y = got[:, :C]
    for i in (1, 2, 3):
        y = torch.nn.functional.max_pool2d(y, 5, 1, 2)
        assert torch.equal(torch.isnan(got[:, i * C:(i + 1) * C]), torch.isnan(y))
        assert torch.equal(torch.nan_to_num(got[:, i * C:(i + 1) * C], nan=1.0), torch.nan_to_num(y, nan=1.0))
