"""The merged detection heads (detect_head.hip) where they can go wrong: pixels that do not fill a tile, pieces of the output
that start off 16 bytes, anchors that end inside a wave's filters, the fewest and the most values a box, one to three levels,
heads that stay operators of their own (too many filters, channels that are no whole slabs); against the oracle's evaluator."""
import pytest

import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, Graph, dev, host, rel_l2

pytestmark = pytest.mark.gpu


# channels of each level, anchors, values per box, N, H, W of the first level, merged
@pytest.mark.parametrize("case", [((64,), 3, 85, 2, 9, 7, True), ((64, 128), 3, 85, 3, 16, 12, True), ((64, 128, 192), 4, 64, 1, 23, 29, True),
                                  ((64, 64), 2, 128, 5, 13, 40, True), ((128,), 1, 201, 1, 64, 64, True), ((64, 128), 3, 86, 1, 8, 8, False),
                                  ((72,), 3, 85, 2, 9, 7, False), ((64,), 3, 20, 2, 9, 7, False)])
def test_detect_heads(case):
    channels, A, F, N, H, W, merged = case
    sizes, ops = [], []

    def take(k):
        sizes.append(k)
        return sum(sizes[:-1])

    def conv(i, c, f, k, s, act):
        ops.append(abi.graph_op(abi.OP_CONV, [i, -1], len(ops) + 1, F=f, K=k, stride=s, pad=k // 2, act=act, w=take(f * c * k * k), bias=take(f)))
        return len(ops)

    levels, prev, c = [], 0, 8
    for i, f in enumerate(channels):
        prev = conv(prev, c, f, 3, 2 if i else 1, abi.ACT_SILU)
        levels.append(prev)
        c = f
    heads = [conv(t, f, A * F, 1, 1, abi.ACT_NONE) for t, f in zip(levels, channels)]
    at_anchors, at_strides = take(len(channels) * A * 2), take(len(channels))
    ops.append(abi.graph_op(abi.OP_YOLO_DETECT, heads, len(ops) + 1, F=F, K=A, stride=0, w=at_anchors, bias=at_strides))
    blob = synth.normal(8300, (sum(sizes),), std=0.05)
    blob[at_anchors:at_strides] = synth.uniform(8301, (at_strides - at_anchors,), 1.0, 8.0)
    blob[at_strides:] = [8.0 * 2 ** i for i in range(len(channels))]
    blob, x = synth.round_fp16(blob), synth.round_fp16(synth.normal(8302, (N, 8, H, W)))
    g = Graph(ops, 8, blob, abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(x, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    print(case, tags, flush=True)
    assert tags.get("detect_head", 0) == int(merged) and ("yolo_detect" in tags) != merged, tags
    want = oracle.run_graph(ops, x, blob, 8)
    assert rel_l2(got.reshape(want.shape), want) < 3e-3 < FP16_REL_L2
    # classes and objectness apart from the much larger coordinates
    boxes = want.reshape(N, -1, F)
    assert rel_l2(got.reshape(boxes.shape)[:, :, 4:], boxes[:, :, 4:]) < 3e-3
    g.close()
