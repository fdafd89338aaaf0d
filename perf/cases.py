"""What programs built on this framework have it do, as cases that can be timed.

A case names one kind of call and its sizes.  `prepare` makes what such a program holds before the call (inputs, weights,
handles, output buffers), `run` makes the call once through the C ABI (include/nncv_hip.h, bound by nncv_amd/abi.py).
Device calls are enqueued on one stream of the program's own, as a serving loop does; host calls (the `_mlir_ciface_*`
functions) take and return host memory and are synchronous by their nature.

Kinds:
  resnet18     nncv_hip_resnet18_forward: the network on a batch that lies in device memory
  serve        the same with several passes in flight, each on a handle and stream of its own
  classify     nncv_hip_resnet18_classify_u8: 8-bit image -> preprocessing, network, top-1
  forward_abi  _mlir_ciface_forward / _f16: the reference's own call, host input, host parameter blob
  matmul       nncv_hip_matmul_f32, C += A.B in device memory
  matmul_abi   _mlir_ciface_matmul on host arrays
  conv         nncv_hip_conv_forward: one fused convolution layer in device memory
  conv_abi     _mlir_ciface_batch_nchw_conv on host arrays (the filter is an argument of the call)
  graph        nncv_hip_graph_forward: MobileNetV3-small and YOLOv5s as operator lists
"""
import ctypes
import math

import numpy as np
import torch

from nncv_amd import abi, mobilenetv3_spec, resnet18_spec, yolov5s_spec


def listed():
    return [
        # one image, half precision: the smallest network call; launches and their gaps are what it costs
        {"name": "resnet18_f16_b1", "kind": "resnet18", "dtype": "f16", "N": 1, "H": 224, "W": 224},
        # the benchmark's batch, one pass after the other on one stream
        {"name": "resnet18_f16_b32", "kind": "resnet18", "dtype": "f16", "N": 32, "H": 224, "W": 224},
        # offline scoring of a large batch
        {"name": "resnet18_f16_b256", "kind": "resnet18", "dtype": "f16", "N": 256, "H": 224, "W": 224},
        # the benchmark's serving loop: four requests of 32 images in flight on four streams
        {"name": "serve_f16_b32_x4", "kind": "serve", "dtype": "f16", "N": 32, "H": 224, "W": 224, "in_flight": 4},
        # photographs of no special size, full precision, from bytes to labels
        {"name": "classify_f32_b6_odd", "kind": "classify", "dtype": "f32", "N": 6, "H": 231, "W": 309, "channels": 3},
        # the reference driver's call: one 256x256 picture on the host, full precision
        {"name": "forward_abi_f32_b1", "kind": "forward_abi", "net": "resnet18", "dtype": "f32", "N": 1, "H": 256, "W": 256},
        # a ragged product in device memory (no dimension a multiple of a tile, rows not 16-byte aligned)
        {"name": "matmul_f32_ragged", "kind": "matmul", "M": 1500, "N": 1001, "K": 777},
        # the reference's matmul program: 1024 cubed on host arrays
        {"name": "matmul_abi_1024", "kind": "matmul_abi", "M": 1024, "N": 1024, "K": 1024},
        # the reference's convolution program: one 3x3 layer on host arrays, the input padded by the caller
        {"name": "conv_abi_3x3", "kind": "conv_abi", "N": 1, "C": 64, "F": 64, "H": 58, "W": 58, "R": 3, "stride": 1},
        # one down-sampling layer of the network alone, half precision, at the layer sweep's batch
        {"name": "conv_f16_3x3_s2", "kind": "conv", "dtype": "f16", "N": 64, "C": 64, "F": 128, "H": 56, "W": 56, "R": 3, "stride": 2,
         "pad": 1, "nchw": False, "residual": False},
        # the small-network graph at a serving batch
        {"name": "mobilenetv3_f16_b32", "kind": "graph", "net": "mobilenetv3", "dtype": "f16", "N": 32, "H": 224, "W": 224},
        # object detection at its native size
        {"name": "yolov5s_f16_b16", "kind": "graph", "net": "yolov5s", "dtype": "f16", "N": 16, "H": 640, "W": 640},
    ]


def _log(rng, lo, hi):
    """An integer of lo..hi, spread evenly over its logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(["resnet18", "resnet18", "serve", "classify", "forward_abi", "matmul", "matmul_abi", "conv", "conv", "conv_abi",
                       "graph", "graph"])
    if kind in ("resnet18", "serve", "classify", "forward_abi"):
        c = {"kind": kind, "dtype": rng.choice(["f16", "f16", "f32"]), "N": 1, "H": rng.randint(96, 320), "W": rng.randint(96, 320)}
        if kind == "resnet18":
            c["N"] = _log(rng, 1, 256 if c["dtype"] == "f16" else 32)
        elif kind == "serve":
            c.update(dtype="f16", N=_log(rng, 1, 32), in_flight=rng.randint(2, 4))
        elif kind == "classify":
            c.update(N=_log(rng, 1, 16), channels=rng.choice([3, 4]))
        else:
            c.update(N=_log(rng, 1, 32), net=rng.choice(["resnet18", "resnet18", "mobilenetv3"]))
        budget = 256 * 224 * 224 if c["dtype"] == "f16" else 32 * 224 * 224  # pixels of the largest call
        c["N"] = max(1, min(c["N"], budget // (c["H"] * c["W"] * c.get("in_flight", 1))))
        return c
    if kind in ("matmul", "matmul_abi"):
        top = 4096 if kind == "matmul" else 2048
        size = [_log(rng, 16, top) for _ in range(3)]
        if rng.random() < 0.4:  # whole rows of 16 bytes
            size = [(v + 3) // 4 * 4 for v in size]
        return {"kind": kind, "M": size[0], "N": size[1], "K": size[2]}
    if kind == "conv":
        R, stride = rng.choice([(1, 1), (1, 2), (3, 1), (3, 1), (3, 2), (5, 1), (7, 2)])
        C, F = _log(rng, 3, 512), _log(rng, 16, 512)
        if rng.random() < 0.7:  # the channel counts of ordinary networks
            C, F = 1 << max(4, round(math.log2(C))), 1 << max(4, round(math.log2(F)))
        c = {"kind": kind, "dtype": rng.choice(["f16", "f16", "f32"]), "N": _log(rng, 1, 64), "C": C, "F": F, "H": _log(rng, 7, 112),
             "W": _log(rng, 7, 112), "R": R, "stride": stride, "pad": R // 2, "nchw": rng.random() < 0.2, "residual": rng.random() < 0.3}
        while work(c)["flops"] > (1e11 if c["dtype"] == "f16" else 2e10) and c["N"] > 1:
            c["N"] //= 2
        return c
    if kind == "conv_abi":
        R, stride = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2), (5, 1), (7, 2)])
        c = {"kind": kind, "N": _log(rng, 1, 16), "C": _log(rng, 3, 256), "F": _log(rng, 8, 256), "H": 0, "W": 0, "R": R, "stride": stride}
        c["H"], c["W"] = (stride * _log(rng, 6, 64) + R for _ in range(2))
        while work(c)["flops"] > 1e10 and c["N"] > 1:
            c["N"] //= 2
        return c
    c = {"kind": "graph", "net": rng.choice(["mobilenetv3", "yolov5s"]), "dtype": rng.choice(["f16", "f16", "f32"]), "N": 1}
    if c["net"] == "mobilenetv3":
        c.update(N=_log(rng, 1, 64), H=rng.randint(96, 288), W=rng.randint(96, 288))
    else:
        c.update(N=_log(rng, 1, 16 if c["dtype"] == "f16" else 4), H=32 * rng.randint(6, 20), W=32 * rng.randint(6, 20))
    return c


# ---- inputs --------------------------------------------------------------------------------------

class _Random:
    """Seeded inputs, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def uniform(self, shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def blob(self, table):
        """A flat fp32 parameter array with the distributions of nncv_amd/synth.py: Kaiming-normal filters, BatchNorm
        statistics around (1, 0, 0, 1), small biases."""
        parts = []
        for name, shape in table:
            if name == "fc.weight":
                a = self.normal(shape, 0.01)
            elif name == "model.24.anchors":
                a = torch.tensor([[v / yolov5s_spec.STRIDES[l] for v in yolov5s_spec.ANCHORS_PX[l]] for l in range(3)], device="cuda")
            elif name == "model.24.stride":
                a = torch.tensor(yolov5s_spec.STRIDES, device="cuda")
            elif len(shape) >= 2:
                a = self.normal(shape, math.sqrt(2.0 / math.prod(shape[1:])))
            elif name.endswith("running_var") or (name.endswith(".weight") and len(shape) == 1):
                a = self.uniform(shape, 0.5, 1.5)
            else:
                a = self.normal(shape, 1.0 if name.startswith("model.24.") else 0.1)
            parts.append(a.reshape(-1).float())
        return torch.cat(parts)


def _torch_dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.float32


def _code(case):
    return abi.F16 if case["dtype"] == "f16" else abi.F32


def _stream():
    """The program's stream for device work."""
    if not hasattr(_stream, "s"):
        _stream.s = torch.cuda.Stream()
    return _stream.s.cuda_stream


class _Handle:
    """A library handle, given back with the state that holds it."""

    def __init__(self, h, destroy):
        if not h:
            raise abi.NncvHipError(abi.lib().nncv_hip_last_error().decode())
        self.h, self._destroy = h, destroy

    def __del__(self):
        if self.h:
            self._destroy(self.h)
            self.h = None


def _resnet18(blob, case, passes):
    L = abi.lib()
    return _Handle(L.nncv_hip_resnet18_create_ex(blob.ctypes.data, blob.size, _code(case), abi.ALGO_AUTO, passes), L.nncv_hip_resnet18_destroy)


_TABLES = {"resnet18": resnet18_spec.tensor_table, "mobilenetv3": mobilenetv3_spec.tensor_table, "yolov5s": yolov5s_spec.tensor_table}


def _empty(shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


# ---- the calls -----------------------------------------------------------------------------------

def prepare(case, seed):
    rnd, L, kind = _Random(seed), abi.lib(), case["kind"]
    s = {"kind": kind, "case": case, "lib": L, "stream": _stream()}
    N = case.get("N")
    if kind in ("resnet18", "serve", "classify", "forward_abi"):
        H, W = case["H"], case["W"]
        blob = rnd.blob(_TABLES[case.get("net", "resnet18")]()).to(_torch_dtype(case)).cpu().numpy()
        if kind == "classify":
            x = [torch.randint(0, 256, (N, H, W, case["channels"]), generator=rnd.g, device="cuda", dtype=torch.uint8)]
        else:
            x = [rnd.uniform((N, 3, H, W)).to(_torch_dtype(case)) for _ in range(case.get("in_flight", 1))]
        if kind == "forward_abi":
            s.update(x=x[0].cpu().numpy(), blob=blob)
            return s
        first = _resnet18(blob, case, case.get("in_flight", 0))
        s.update(x=x, handles=[first], logits=[_empty((N, 1000)) for _ in x], streams=[s["stream"]])
        if kind == "serve":
            st, found = (ctypes.c_void_p * len(x))(), ctypes.c_int(0)
            abi.check(L.nncv_hip_pick_streams(len(x), st, ctypes.byref(found)))
            s["streams"] = list(st)
            s["handles"] += [_Handle(L.nncv_hip_resnet18_clone(first.h), L.nncv_hip_resnet18_destroy) for _ in x[1:]]
        if kind == "classify":
            s["top1"] = _empty((N,), torch.int32)
    elif kind in ("matmul", "matmul_abi"):
        M, K = case["M"], case["K"]
        a, b, c = rnd.uniform((M, K), -1, 1), rnd.uniform((K, N), -1, 1), rnd.uniform((M, N), -1, 1)
        if kind == "matmul_abi":
            a, b, c = a.cpu().numpy(), b.cpu().numpy(), c.cpu().numpy()
        s.update(a=a, b=b, c=c)
    elif kind == "conv":
        C, F, H, W, R = (case[k] for k in "CFHWR")
        dt, (oh, ow) = _torch_dtype(case), _out_hw(case)
        w = rnd.normal((F, C, R, R), math.sqrt(2.0 / (C * R * R))).to(dt).cpu().numpy()
        bn = [v.to(dt).cpu().numpy() for v in (rnd.uniform((F,), 0.5, 1.5), rnd.normal((F,), 0.1), rnd.normal((F,), 0.1), rnd.uniform((F,), 0.5, 1.5))]
        order = (lambda n, c, h, w: (n, c, h, w)) if case["nchw"] else (lambda n, c, h, w: (n, h, w, c))
        s.update(handle=_Handle(L.nncv_hip_conv_create(_code(case), w.ctypes.data, F, C, R, R, case["stride"], case["pad"],
                                                       *[v.ctypes.data for v in bn], 1, abi.ALGO_AUTO), L.nncv_hip_conv_destroy),
                 x=rnd.normal(order(N, C, H, W)).to(dt), out=_empty(order(N, F, oh, ow), dt),
                 residual=rnd.normal(order(N, F, oh, ow)).to(dt) if case["residual"] else None)
    elif kind == "conv_abi":
        C, F, H, W, R = (case[k] for k in "CFHWR")
        oh, ow = _out_hw(case)
        s.update(x=rnd.normal((N, C, H, W)).cpu().numpy(), w=rnd.normal((F, C, R, R), math.sqrt(2.0 / (C * R * R))).cpu().numpy(),
                 out=rnd.normal((N, F, oh, ow)).cpu().numpy())
    elif kind == "graph":
        H, W = case["H"], case["W"]
        ops = (mobilenetv3_spec if case["net"] == "mobilenetv3" else yolov5s_spec).graph_ops()
        blob = rnd.blob(_TABLES[case["net"]]()).to(_torch_dtype(case)).cpu().numpy()
        s["handle"] = _Handle(abi.graph_create(ops, 3, blob), L.nncv_hip_graph_destroy)
        s.update(x=rnd.uniform((N, 3, H, W)).to(_torch_dtype(case)), out=_empty((N,) + abi.graph_output_shape(s["handle"].h, H, W)))
    return s


def run(s):
    L, case, kind = s["lib"], s["case"], s["kind"]
    if kind in ("resnet18", "serve"):
        for h, x, y, st in zip(s["handles"], s["x"], s["logits"], s["streams"]):
            abi.check(L.nncv_hip_resnet18_forward(h.h, x.data_ptr(), case["N"], case["H"], case["W"], y.data_ptr(), st))
        return s["logits"]
    if kind == "classify":
        abi.check(L.nncv_hip_resnet18_classify_u8(s["handles"][0].h, s["x"][0].data_ptr(), case["N"], case["H"], case["W"], case["channels"],
                                                  s["logits"][0].data_ptr(), s["top1"].data_ptr(), s["stream"]))
        return {"logits": s["logits"][0], "top1": s["top1"]}
    if kind == "forward_abi":
        return abi.forward(s["x"], s["blob"])
    if kind == "matmul":
        abi.check(L.nncv_hip_matmul_f32(s["a"].data_ptr(), s["b"].data_ptr(), s["c"].data_ptr(), case["M"], case["N"], case["K"], s["stream"]))
        return s["c"]
    if kind == "matmul_abi":
        return abi.matmul(s["a"], s["b"], s["c"])
    if kind == "conv":
        abi.check(L.nncv_hip_conv_forward(s["handle"].h, s["x"].data_ptr(), case["N"], case["H"], case["W"], abi.NCHW if case["nchw"] else abi.NHWC,
                                          s["residual"].data_ptr() if case["residual"] else None, s["out"].data_ptr(), s["stream"]))
        return s["out"]
    if kind == "conv_abi":
        return abi.batch_nchw_conv(s["x"], s["w"], s["out"])
    abi.check(L.nncv_hip_graph_forward(s["handle"].h, s["x"].data_ptr(), case["N"], case["H"], case["W"], s["out"].data_ptr(), s["out"].numel(),
                                       s["stream"]))
    return s["out"]


# ---- what a call cannot do without ---------------------------------------------------------------

def _out_hw(case):
    R, st, pad = case["R"], case["stride"], case.get("pad", 0)
    return (case["H"] + 2 * pad - R) // st + 1, (case["W"] + 2 * pad - R) // st + 1


def _conv_flops(N, C, F, R, h, w, st, pad):
    oh, ow = (h + 2 * pad - R) // st + 1, (w + 2 * pad - R) // st + 1
    return 2 * N * oh * ow * F * C * R * R, oh, ow


def _resnet18_flops(N, H, W):
    total, h, w = _conv_flops(N, 3, 64, 7, H, W, 2, 3)
    h, w, cin = (h - 1) // 2 + 1, (w - 1) // 2 + 1, 64
    for k, f in enumerate(resnet18_spec.WIDTHS):
        st = 2 if k else 1
        a, oh, ow = _conv_flops(N, cin, f, 3, h, w, st, 1)
        total += a + 3 * _conv_flops(N, f, f, 3, oh, ow, 1, 1)[0] + (_conv_flops(N, cin, f, 1, h, w, st, 0)[0] if k else 0)
        h, w, cin = oh, ow, f
    return total + 2 * N * 512 * 1000


def _mobilenetv3_flops(N, H, W):
    side = math.sqrt(H * W)  # the convolutions scale with the area; the table is for square images
    return N * mobilenetv3_spec.flops_per_image(int(round(side)))


def work(case):
    """Inputs and parameters read once, outputs written once; twice the multiplications of the direct algorithm."""
    kind = case["kind"]
    if kind in ("matmul", "matmul_abi"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * (M * K + K * N + 2 * M * N), "flops": 2 * M * N * K}
    if kind in ("conv", "conv_abi"):
        e = 2 if case.get("dtype") == "f16" else 4
        flops, oh, ow = _conv_flops(case["N"], case["C"], case["F"], case["R"], case["H"], case["W"], case["stride"], case.get("pad", 0))
        outs = 2 if kind == "conv_abi" or case["residual"] else 1  # conv_abi accumulates into its output
        return {"bytes": e * (case["N"] * case["C"] * case["H"] * case["W"] + case["F"] * case["C"] * case["R"] ** 2 + outs * case["N"] * case["F"] * oh * ow),
                "flops": flops}
    N, H, W = case["N"] * case.get("in_flight", 1), case["H"], case["W"]
    net, e = case.get("net", "resnet18"), 2 if case["dtype"] == "f16" else 4
    pixels = N * H * W * (case["channels"] if kind == "classify" else 3 * e)
    if net == "yolov5s":
        outputs = 4 * N * 85 * 3 * sum((H // s) * (W // s) for s in (8, 16, 32))
        return {"bytes": pixels + e * yolov5s_spec.NUM_ELEMENTS + outputs, "flops": N * yolov5s_spec.flops_per_image(H, W)}
    spec = resnet18_spec if net == "resnet18" else mobilenetv3_spec
    return {"bytes": pixels + e * spec.NUM_ELEMENTS + (e if kind == "forward_abi" else 4) * N * 1000,
            "flops": (_resnet18_flops if net == "resnet18" else _mobilenetv3_flops)(N, H, W)}


def tolerance(case):
    """fp32: sums of a few thousand terms in another order.  fp16: a single layer rounds its result once; a network rounds
    every activation.  Top-1 labels are the same but for ties."""
    if case.get("dtype", "f32") == "f32":
        return {"rel": 1e-5, "differ": 0.01}
    return {"rel": 1e-3 if case["kind"] == "conv" else 5e-3, "differ": 0.01}
