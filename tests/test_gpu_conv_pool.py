"""The end of MobileNetV3 in fewer launches: a pointwise convolution that leaves only its means (conv_pool.hip), and a last layer that
writes the caller's fp32 tensor itself.  Tiles of 32 pixels and blocks of 32 filters with remainders, channel counts around a trip of 96,
the largest map and the first one beyond it, filter counts that are whole vectors of four, of eight, and neither."""
import pytest
import torch

import graph_bound
import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, Graph, dev, host, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [abi.F16, abi.F32])
@pytest.mark.parametrize("case", [  # N, H, W, channels, filters, outputs
    (1, 1, 1, 8, 8, 8), (2, 5, 13, 24, 40, 12), (3, 8, 8, 96, 576, 1000), (2, 4, 8, 104, 72, 6), (1, 16, 32, 128, 33 * 8, 20), (32, 7, 7, 96, 576, 1000),
    (2, 19, 27, 16, 64, 44), (2, 7, 7, 136, 64, 40), (33, 16, 32, 16, 32, 16)])
def test_means_and_last_layer(case, dt):
    N, H, W, C, F, O = case
    pool = dt == abi.F16 and H * W <= 512 and C <= 128 and N * H * W <= 16384
    w1, w2, w3 = C * 8, F * C, O * F
    at = [0, w1, w1 + w2, w1 + w2 + F, w1 + w2 + F + w3]
    ops = [abi.graph_op(abi.OP_CONV, [0, -1], 1, F=C, K=1, act=abi.ACT_NONE, w=at[0]),
           abi.graph_op(abi.OP_CONV, [1, -1], 2, F=F, K=1, act=abi.ACT_HARDSWISH, w=at[1], bias=at[2]),
           abi.graph_op(abi.OP_GAVGPOOL, [2], 3, stride=0),
           abi.graph_op(abi.OP_CONV, [3, -1], 4, F=O, K=1, act=abi.ACT_NONE, w=at[3], bias=at[4])]
    blob = synth.normal(8200, (at[4] + O,), std=0.3)
    x = synth.normal(8201, (N, 8, H, W))
    if dt == abi.F16:
        blob, x = synth.round_fp16(blob), synth.round_fp16(x)
    launches = abi.graph_plan(ops, 8, dt, N, H, W)[2]
    g = Graph(ops, 8, blob, dt)
    out = torch.empty(N * O + 1, dtype=torch.float32, device="cuda")  # the caller's tensor at 16 bytes and one float further on
    xd = dev(x, dt)
    torch.cuda.synchronize()
    want = oracle.run_graph(ops, x, blob, 8)
    abi.profile_enable(True)
    try:
        for shift in (0, 1):
            abi.profile_report()
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            abi.check(abi.lib().nncv_hip_graph_forward(g.h, xd.data_ptr(), N, H, W, out.data_ptr() + 4 * shift, N * O, None))
            tags = {k: v["launches"] for k, v in abi.profile_report().items()}
            print(case, dt, tags, flush=True)
            got = host(out)[shift:shift + N * O].reshape(want.shape)
            # fp16: three layers of rounded results, as in the other tests of merged layers; fp32: sums of up to 576 terms
            assert rel_l2(got, want) < (3e-3 if dt == abi.F16 else 1e-5) < FP16_REL_L2
            assert dt == abi.F32 or graph_bound.worst(got.reshape(N, O, 1, 1), ops, x, blob) < graph_bound.LIMIT  # every value
            assert tags.get("conv_pool", 0) == int(pool) and tags.get("global_avgpool", 0) == int(not pool), tags
            ends = tags.get("relayout", 0) - int("image_to_nhwc" not in tags)  # (one of them may lay the input out)
            assert (O % 4 == 0 or ends == 1) and (O != 1000 or ends == 0), tags
            assert (launches[3] == -1) == (ends == 0) and (launches[1] == 3) == (launches[2] == -1) == pool, launches  # the plan is of these launches
    finally:
        abi.profile_enable(False)
        g.close()
