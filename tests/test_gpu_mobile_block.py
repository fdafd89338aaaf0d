"""Inverted-residual blocks as two launches (mobile_block.hip) where they can go wrong: channel groups that are not full,
bands of an image, strips that overrun a row, one and many K steps, no expansion, no gate, maps smaller than the window's
padding, images too wide for the LDS image (the block's operators then run one by one); against the oracle's evaluator."""
import pytest

import oracle
from nncv_amd import abi, synth
from gpu_util import FP16_REL_L2, Graph, dev, host, rel_l2

pytestmark = pytest.mark.gpu


# cin, exp (= cin: no expansion), cout, K, stride, SQ (0: no gate), N, H, W
@pytest.mark.parametrize("case", [
    (16, 16, 16, 3, 2, 8, 2, 57, 33), (16, 72, 24, 3, 2, 0, 3, 31, 29), (24, 88, 24, 3, 1, 0, 1, 28, 28), (24, 96, 40, 5, 2, 24, 2, 27, 25),
    (40, 240, 40, 5, 1, 64, 3, 14, 13), (96, 576, 96, 5, 1, 144, 2, 7, 7), (48, 288, 96, 5, 2, 72, 5, 3, 2), (8, 40, 8, 5, 1, 8, 40, 19, 6),
    (32, 104, 56, 3, 1, 16, 130, 9, 9), (16, 64, 16, 5, 1, 16, 1, 6, 700)])
def test_inverted_residual_block(case):
    cin, exp, cout, K, stride, sq, N, H, W = case
    tags = check_block(case)
    merged = exp != cin or sq > 0
    assert sum(v for k, v in tags.items() if k.startswith("dw_block")) == int(merged and W < 700), tags
    assert tags.get("se_project", 0) == int(sq > 0 and W < 700), tags


# every instance of the depthwise kernel (window, stride, outputs a thread takes at a time, 16-channel steps of the expansion), and
# between them every instance of the projection: one, two or three slices of 256 channels, 16, 48 or 96 filters, 16 or
# 32 pixels a tile, and expanded tensors of up to 32 channels
EVERY = [
    (24, 24, 8, 3, 1, 200, 2, 6, 7, "3,1,1,0"), (8, 40, 56, 3, 1, 40, 70, 15, 15, "3,1,1,1"), (8, 40, 24, 3, 1, 136, 70, 19, 12, "3,1,1,1"),
    (8, 40, 24, 3, 1, 136, 2, 7, 6, "3,1,1,1"), (32, 24, 8, 3, 1, 8, 3, 7, 6, "3,1,1,3"), (72, 24, 8, 3, 1, 40, 2, 6, 9, "3,1,1,6"),
    (24, 24, 8, 3, 1, 40, 2, 6, 27, "3,1,2,0"), (8, 520, 8, 3, 1, 40, 70, 13, 18, "3,1,2,1"), (8, 264, 8, 3, 1, 24, 70, 11, 21, "3,1,2,1"),
    (8, 40, 8, 3, 1, 8, 40, 15, 27, "3,1,2,1"), (32, 24, 8, 3, 1, 136, 2, 6, 25, "3,1,2,3"), (72, 24, 16, 3, 1, 72, 2, 6, 22, "3,1,2,6"),
    (24, 24, 8, 3, 1, 40, 2, 7, 37, "3,1,4,0"), (8, 520, 56, 3, 1, 256, 70, 6, 39, "3,1,4,1"), (8, 520, 24, 3, 1, 256, 40, 14, 30, "3,1,4,1"),
    (8, 264, 56, 3, 1, 8, 40, 16, 26, "3,1,4,1"), (8, 264, 24, 3, 1, 24, 40, 31, 13, "3,1,4,1"), (32, 24, 16, 3, 1, 200, 2, 8, 35, "3,1,4,3"),
    (72, 24, 24, 3, 1, 8, 2, 7, 34, "3,1,4,6"), (24, 24, 24, 3, 2, 40, 2, 6, 6, "3,2,1,0"), (8, 520, 56, 3, 2, 24, 2, 7, 7, "3,2,1,1"),
    (8, 520, 24, 3, 2, 200, 2, 6, 7, "3,2,1,1"), (8, 264, 56, 3, 2, 40, 2, 6, 7, "3,2,1,1"), (16, 584, 8, 3, 2, 40, 2, 6, 6, "3,2,1,1"),
    (8, 264, 24, 3, 2, 200, 2, 6, 7, "3,2,1,1"), (8, 264, 8, 3, 2, 40, 3, 6, 7, "3,2,1,1"), (16, 40, 56, 3, 2, 256, 2, 6, 6, "3,2,1,1"),
    (8, 24, 56, 3, 2, 8, 2, 6, 7, "3,2,1,1"), (8, 40, 16, 3, 2, 24, 2, 6, 7, "3,2,1,1"), (32, 24, 16, 3, 2, 136, 2, 6, 7, "3,2,1,3"),
    (56, 24, 16, 3, 2, 136, 2, 7, 7, "3,2,1,6"), (24, 24, 8, 3, 2, 24, 2, 7, 37, "3,2,2,0"), (16, 24, 16, 3, 2, 8, 2, 7, 33, "3,2,2,1"),
    (32, 24, 8, 3, 2, 40, 2, 7, 34, "3,2,2,3"), (56, 24, 8, 3, 2, 256, 2, 8, 33, "3,2,2,6"), (24, 24, 8, 3, 2, 24, 1, 3, 260, "3,2,4,0"),
    (8, 24, 8, 3, 2, 40, 1, 3, 259, "3,2,4,1"), (32, 24, 8, 3, 2, 200, 1, 3, 284, "3,2,4,3"), (56, 24, 8, 3, 2, 24, 1, 3, 272, "3,2,4,6"),
    (24, 24, 16, 5, 1, 24, 2, 7, 6, "5,1,1,0"), (8, 24, 8, 5, 1, 8, 2, 6, 7, "5,1,1,1"), (32, 24, 16, 5, 1, 256, 2, 6, 6, "5,1,1,3"),
    (72, 24, 8, 5, 1, 200, 2, 6, 6, "5,1,1,6"), (24, 24, 24, 5, 1, 24, 2, 8, 18, "5,1,2,0"), (8, 24, 8, 5, 1, 136, 2, 7, 18, "5,1,2,1"),
    (32, 24, 8, 5, 1, 40, 2, 7, 17, "5,1,2,3"), (72, 24, 8, 5, 1, 256, 2, 7, 17, "5,1,2,6"), (24, 24, 16, 5, 1, 8, 2, 7, 34, "5,1,4,0"),
    (8, 24, 8, 5, 1, 136, 2, 7, 40, "5,1,4,1"), (40, 24, 16, 5, 1, 200, 2, 7, 34, "5,1,4,3"), (88, 24, 16, 5, 1, 72, 2, 7, 34, "5,1,4,6"),
    (24, 24, 8, 5, 2, 136, 2, 6, 6, "5,2,1,0"), (8, 24, 8, 5, 2, 8, 2, 6, 8, "5,2,1,1"), (32, 24, 48, 5, 2, 72, 2, 6, 6, "5,2,1,3"),
    (56, 24, 24, 5, 2, 40, 2, 8, 8, "5,2,1,6"), (24, 24, 16, 5, 2, 24, 2, 7, 33, "5,2,2,0"), (8, 24, 16, 5, 2, 24, 2, 7, 39, "5,2,2,1"),
    (32, 24, 8, 5, 2, 136, 2, 7, 39, "5,2,2,3"), (56, 24, 16, 5, 2, 200, 2, 8, 33, "5,2,2,6"), (24, 24, 8, 5, 2, 40, 1, 3, 267, "5,2,4,0"),
    (8, 24, 8, 5, 2, 200, 1, 3, 267, "5,2,4,1"), (32, 24, 8, 5, 2, 72, 1, 3, 270, "5,2,4,3"), (56, 24, 16, 5, 2, 72, 1, 3, 263, "5,2,4,6"),
]


@pytest.mark.parametrize("case", EVERY, ids=lambda c: "-".join(map(str, c)))
def test_every_instance(case):
    tags = check_block(case[:9])
    assert tags.get("dw_block<%s>" % case[9]) == 1 and tags.get("se_project") == 1, tags


def check_block(case):
    """The block against the oracle's evaluator; launches by tag."""
    cin, exp, cout, K, stride, sq, N, H, W = case
    sizes, ops = [], []

    def take(n):
        sizes.append(n)
        return sum(sizes[:-1])

    def conv(i, o, c, f, k, s, act, kind=abi.OP_CONV, res=-1):
        w = take(f * (1 if kind == abi.OP_DWCONV else c) * k * k)
        bn = (take(f), take(f), take(f), take(f))
        ops.append(abi.graph_op(kind, [i, res] if kind == abi.OP_CONV else [i], o, F=f, K=k, stride=s, pad=k // 2, act=act, w=w, eps=1e-3, bn=bn))
        return o

    t = conv(0, 1, cin, cin, 1, 1, abi.ACT_NONE)
    x0 = t
    if exp != cin:
        t = conv(t, 2, cin, exp, 1, 1, abi.ACT_HARDSWISH)
    t = conv(t, 3, exp, exp, K, stride, abi.ACT_RELU if K == 3 else abi.ACT_HARDSWISH, kind=abi.OP_DWCONV)
    if sq:
        ops.append(abi.graph_op(abi.OP_GAVGPOOL, [t], 4, stride=0))
        ops.append(abi.graph_op(abi.OP_CONV, [4], 5, F=sq, K=1, act=abi.ACT_RELU, w=take(sq * exp), bias=take(sq)))
        ops.append(abi.graph_op(abi.OP_CONV, [5], 6, F=exp, K=1, act=abi.ACT_HARDSIGMOID, w=take(exp * sq), bias=take(exp)))
        ops.append(abi.graph_op(abi.OP_SCALE, [t, 6], 7, stride=0))
        t = 7
    conv(t, 8, exp, cout, 1, 1, abi.ACT_NONE, res=x0 if stride == 1 and cin == cout else -1)
    ids = {0: 0}  # tensor ids without gaps
    for i, o in enumerate(ops):
        ids[o.out] = i + 1
    for o in ops:
        o.out = ids[o.out]
        for k in range(4):
            if o.inputs[k] >= 0:
                o.inputs[k] = ids[o.inputs[k]]
    blob = synth.normal(8100, (sum(sizes),), std=0.3)
    for o in ops:  # variances are positive
        if o.gamma >= 0:
            f = o.F if o.kind == abi.OP_CONV else exp
            blob[o.var:o.var + f] = synth.uniform(8103 + o.out, (f,), 0.5, 1.5)
    blob, x = synth.round_fp16(blob), synth.round_fp16(synth.normal(8102, (N, cin, H, W)))
    g = Graph(ops, cin, blob, abi.F16)
    abi.profile_enable(True)
    try:
        abi.profile_report()
        got = host(g(dev(x, abi.F16)))
        tags = {k: v["launches"] for k, v in abi.profile_report().items()}
    finally:
        abi.profile_enable(False)
    print(case, tags, flush=True)
    want = oracle.run_graph(ops, x, blob, cin)
    assert rel_l2(got, want) < 3e-3 < FP16_REL_L2
    g.close()
    return tags
