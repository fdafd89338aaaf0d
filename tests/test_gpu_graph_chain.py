"""C3 blocks whose first bottleneck layer is computed by the launch of the two pointwise layers in front of it (conv_ring.hip) where that can
go wrong: one slab of channels and several, a slab that is not full, pixels that end inside a tile, a first result that others read too and one that
nothing else reads, chains of bottlenecks, rows of a wider tensor, and the first size below the line; against the oracle's evaluator."""
import pytest

import graph_bound
import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, Graph, dev, host, rel_l2

pytestmark = pytest.mark.gpu


# c1, c_, bottlenecks, shortcut, N, H, W, activation of the chained layer, whether it is
@pytest.mark.parametrize("case", [(64, 32, 1, True, 2, 131, 129, abi.ACT_SILU, True), (40, 32, 2, True, 1, 190, 181, abi.ACT_RELU, True), (96, 32, 1, False, 3, 111, 105, abi.ACT_NONE, True),
                                  (128, 64, 2, True, 1, 129, 131, abi.ACT_SILU, True), (192, 64, 1, False, 2, 97, 89, abi.ACT_SILU, True), (72, 64, 1, True, 1, 128, 128, abi.ACT_HARDSWISH, True),
                                  (64, 32, 1, True, 1, 181, 181, abi.ACT_SILU, False), (64, 48, 1, True, 2, 131, 129, abi.ACT_SILU, False)])
def test_chained_layer(case):
    c1, c_, n, shortcut, N, H, W, act, chained = case
    sizes, ops = [], []

    def take(k):
        sizes.append(k)
        return sum(sizes[:-1])

    def op(kind, ins, **kw):
        ops.append(abi.graph_op(kind, ins, len(ops) + 1, **kw))
        return len(ops)

    def conv(i, c, f, k=1, act=abi.ACT_SILU):
        return op(abi.OP_CONV, [i, -1], F=f, K=k, stride=1, pad=k // 2, act=act, w=take(f * c * k * k), bias=take(f))

    x = conv(0, 8, c1)
    y = conv(x, c1, c_)
    for _ in range(n):
        t = conv(conv(y, c_, c_, act=act), c_, c_, 3)
        y = op(abi.OP_ADD, [y, t], stride=0) if shortcut else t
    z = conv(x, c1, c_)
    conv(op(abi.OP_CONCAT, [y, z], stride=0), 2 * c_, c1)
    blob = synth.round_fp16(synth.normal(8300, (sum(sizes),), std=(2.0 / c1) ** 0.5 / 2))
    inp = synth.round_fp16(synth.normal(8301, (N, 8, H, W)))
    launches = abi.graph_plan(ops, 8, abi.F16, N, H, W)[2]
    g = Graph(ops, 8, blob, abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(inp, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    print(case, tags, flush=True)
    assert tags.get("conv_ring<chain>", 0) == int(chained) and (launches[2] == -1) == chained, tags
    assert rel_l2(got, oracle.run_graph(ops, inp, blob, 8)) < FP16_REL_L2
    assert graph_bound.worst(got, ops, inp, blob) < graph_bound.LIMIT  # every value
    g.close()
