"""The image layer straight from the NCHW image (conv_pairs.hip): launches that take the eight-row tiles, rows and columns that
do not fill them, both windows, one and two blocks of filters, one to four channels; against the oracle's evaluator."""
import numpy as np
import pytest

import oracle
from nncv_amd import abi, synth
from gpu_util import Graph, dev, host, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,pad,F,act,shape", [
    (6, 2, 32, abi.ACT_SILU, (8, 3, 130, 518)), (6, 2, 40, abi.ACT_RELU, (5, 4, 258, 450)), (3, 1, 16, abi.ACT_HARDSWISH, (9, 3, 131, 322)),
    (3, 1, 64, abi.ACT_NONE, (13, 1, 115, 258)), (6, 2, 8, abi.ACT_SILU, (1, 2, 4, 2)), (3, 1, 24, abi.ACT_SILU, (2, 3, 1, 2))])
def test_image_layer(k, pad, F, act, shape):
    N, C, H, W = shape
    w = synth.normal(8400 + k, (F, C, k, k), std=float(np.sqrt(2.0 / (C * k * k))))
    blob = synth.round_fp16(np.concatenate([w.ravel(), synth.normal(8401, (F,), std=0.1)]))
    ops = [abi.graph_op(abi.OP_CONV, [0, -1], 1, F=F, K=k, stride=2, pad=pad, act=act, w=0, bias=F * C * k * k)]
    x = synth.round_fp16(synth.uniform(8402, shape, -1.0, 1.0))
    g = Graph(ops, C, blob, abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(x, abi.F16)))
        tags = sorted(abi.profile_report())
    finally:
        abi.profile_enable(False)
    print(k, pad, F, shape, tags, flush=True)
    assert any(t.startswith("conv_pairs<f16,") for t in tags) and "image_to_nhwc" not in tags, tags
    assert rel_l2(got, oracle.run_graph(ops, x, blob, C)) < 2e-3
    g.close()
