"""C3 blocks (two 1x1 convolutions of one tensor, n bottlenecks behind the first, concatenation, 1x1) where their merged form
can go wrong: channel halves that end inside a filter tile, pixel counts that are no multiple of a tile, chains of residuals
whose rows are widened, no residual at all, maps so small that the two convolutions stay apart; against the oracle's evaluator."""
import pytest

import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, FP32_MAX_REL, Graph, dev, host, max_rel, rel_l2

pytestmark = pytest.mark.gpu


# c1, c_, n, shortcut, N, H, W, whether fp16 joins the two convolutions
@pytest.mark.parametrize("dt", [abi.F16, abi.F32])
@pytest.mark.parametrize("case", [(64, 32, 1, True, 2, 93, 101, True), (48, 40, 3, True, 3, 61, 57, True), (128, 72, 2, False, 1, 121, 99, True),
                                  (256, 128, 1, True, 8, 40, 40, True), (32, 8, 2, True, 1, 200, 90, True), (512, 256, 1, True, 1, 3, 5, False)])
def test_c3_block(case, dt):
    c1, c_, n, shortcut, N, H, W, joins = case
    sizes, ops = [], []

    def take(k):
        sizes.append(k)
        return sum(sizes[:-1])

    def op(kind, ins, **kw):
        ops.append(abi.graph_op(kind, ins, len(ops) + 1, **kw))
        return len(ops)

    def conv(i, c, f, k=1):
        return op(abi.OP_CONV, [i, -1], F=f, K=k, stride=1, pad=k // 2, act=abi.ACT_SILU, w=take(f * c * k * k), bias=take(f))

    x = conv(0, c1, c1)
    y = conv(x, c1, c_)
    for _ in range(n):
        t = conv(conv(y, c_, c_), c_, c_, 3)
        y = op(abi.OP_ADD, [y, t], stride=0) if shortcut else t
    z = conv(x, c1, c_)
    conv(op(abi.OP_CONCAT, [y, z], stride=0), 2 * c_, c1)
    blob = synth.normal(8200, (sum(sizes),), std=(2.0 / c1) ** 0.5 / 2)
    inp = synth.normal(8201, (N, c1, H, W))
    if dt == abi.F16:
        blob, inp = synth.round_fp16(blob), synth.round_fp16(inp)
    launches = abi.graph_plan(ops, c1, dt, N, H, W)[2]
    g = Graph(ops, c1, blob, dt)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(inp, dt)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    print(case, tags, flush=True)
    assert "concat_slice" not in " ".join(tags), tags  # both inputs of the concatenation are written in place
    convs = sum(o.kind == abi.OP_CONV for o in ops)
    if dt == abi.F16 and joins:
        assert launches[z - 1] == -1
    assert sum(v for k, v in tags.items() if "conv" in k or "igemm" in k) == convs - int(dt == abi.F16 and joins), tags
    want = oracle.run_graph(ops, inp, blob, c1)
    assert (rel_l2(got, want) < FP16_REL_L2) if dt == abi.F16 else (max_rel(got, want) < FP32_MAX_REL)
    g.close()
