"""A C3 block behind [up-sampled, skip] whose launch reads the tensor of half the size itself (conv_ring.hip) where that can go wrong: with and without the
chained layer, pixels that end inside a tile, a last slab that is not full, several images, a source that is a slice of a wider tensor; and what must keep
the copy: another reader, the second place in the concatenation, part of a slab, launches of other tiles.  Against the oracle's evaluator."""
import pytest

import graph_bound
import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, Graph, dev, host, rel_l2

pytestmark = pytest.mark.gpu


# channels up-sampled, of the skip, c_, N, H, W of the small tensor, what else, whether the copy is saved
@pytest.mark.parametrize("case", [(128, 128, 64, 3, 41, 37, "", True), (64, 104, 64, 1, 75, 67, "", True), (256, 256, 128, 5, 33, 35, "", True), (64, 200, 128, 3, 59, 45, "", True),
                                  (128, 128, 64, 3, 41, 37, "sliced", True), (128, 128, 64, 3, 41, 37, "reader", False), (128, 128, 64, 3, 41, 37, "second", False),
                                  (72, 128, 64, 3, 41, 37, "", False), (128, 128, 64, 1, 9, 11, "", False), (256, 256, 128, 7, 20, 20, "", False)])
def test_block_behind_upsampling(case):
    cu, cs, c_, N, H, W, other, saved = case
    sizes, ops = [], []

    def take(k):
        sizes.append(k)
        return sum(sizes[:-1])

    def op(kind, ins, **kw):
        ops.append(abi.graph_op(kind, ins, len(ops) + 1, **kw))
        return len(ops)

    def conv(i, c, f, k=1, s=1):
        return op(abi.OP_CONV, [i, -1], F=f, K=k, stride=s, pad=k // 2, act=abi.ACT_SILU, w=take(f * c * k * k), bias=take(f))

    skip = conv(0, 8, cs)
    small = conv(skip, cs, cu, 3, 2)
    if other == "sliced":  # the source of the up-sampling lies in a tensor of twice the channels, which another layer reads
        wide = op(abi.OP_CONCAT, [conv(small, cu, cu), small], stride=0)
    up = op(abi.OP_UPSAMPLE2X, [small], stride=0)
    cat = op(abi.OP_CONCAT, [skip, up] if other == "second" else [up, skip], stride=0)
    y = conv(cat, cu + cs, c_)
    t = conv(conv(y, c_, c_), c_, c_, 3)
    z = conv(cat, cu + cs, c_)
    ends = [t, z]
    if other == "reader":
        ends.append(conv(cat, cu + cs, 16))
    if other == "sliced":
        ends.append(op(abi.OP_UPSAMPLE2X, [conv(wide, 2 * cu, 16)], stride=0))
    conv(op(abi.OP_CONCAT, ends, stride=0), 2 * c_ + 16 * (len(ends) - 2), 32)
    blob = synth.round_fp16(synth.normal(8500, (sum(sizes),), std=0.05))
    inp = synth.round_fp16(synth.normal(8501, (N, 8, 2 * H, 2 * W)))
    launches = abi.graph_plan(ops, 8, abi.F16, N, 2 * H, 2 * W)[2]
    g = Graph(ops, 8, blob, abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(inp, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    print(case, tags, flush=True)
    assert tags.get("upsample2x", 0) == int(not saved) + int(other == "sliced"), tags
    assert (launches[up - 1] == -1) == saved
    assert rel_l2(got, oracle.run_graph(ops, inp, blob, 8)) < FP16_REL_L2
    assert graph_bound.worst(got, ops, inp, blob) < graph_bound.LIMIT  # every value
    g.close()
