"""A list of graph operators in 64 bits, with a bound for each value of what a pass in fp16 (fp32 sums) makes of it.

A stored value is rounded once, by at most 2^-11 of itself, an error spread evenly: a standard deviation of 2^-11 / sqrt(3) of it at most.  Roundings of
different values are independent, so variances are what convolutions with squared filters, means and sums of them make; an activation multiplies an error
by its steepest slope.  Sums of K products in fp32 add K roundings of 2^-24 of them.  LIMIT standard deviations are allowed for every value: one in 10^15 of a
normal distribution lies beyond eight.  The value of another pixel or channel is hundreds of them off (a block of 64 to 192 channels)."""
import math

import numpy as np
import torch
import torch.nn.functional as F

from nncv_amd import abi

LIMIT = 8
_ACT = {abi.ACT_NONE: (lambda v: v, 1.0), abi.ACT_RELU: (torch.relu, 1.0), abi.ACT_HARDSWISH: (F.hardswish, 1.5), abi.ACT_SILU: (F.silu, 1.1)}


def _stored(v, var):
    return v, var + (v * 2.0 ** -11) ** 2 / 3 + 2.0 ** -50


def evaluate(ops, x, blob):
    """-> (values, standard deviations) of the last operator's result, NCHW, 64 bits."""
    blob, x = torch.from_numpy(np.asarray(blob, np.float64)), torch.from_numpy(np.asarray(x, np.float64))
    vals = {0: (x, torch.zeros_like(x))}
    for o in ops:
        ins = [vals[t] for t in o.inputs if t >= 0]
        a, va = ins[0]
        if o.kind == abi.OP_CONV:
            assert len(ins) == 1 and o.gamma < 0
            w = blob[o.w:o.w + o.F * a.shape[1] * o.K * o.K].reshape(o.F, a.shape[1], o.K, o.K)
            y = F.conv2d(a, w, blob[o.bias:o.bias + o.F] if o.bias >= 0 else None, o.stride, o.pad)
            act, slope = _ACT[o.act]
            var = F.conv2d(va, w ** 2, None, o.stride, o.pad) + w[0].numel() * 2.0 ** -48 * F.conv2d(a ** 2, w ** 2, None, o.stride, o.pad)
            vals[o.out] = _stored(act(y), var * slope ** 2 + y ** 2 * 2.0 ** -40)  # (fast exponentials and reciprocals: 2^-20)
        elif o.kind == abi.OP_GAVGPOOL:
            vals[o.out] = _stored(a.mean((2, 3), keepdim=True), va.mean((2, 3), keepdim=True) / (a.shape[2] * a.shape[3]))
        elif o.kind == abi.OP_ADD:
            vals[o.out] = _stored(_ACT[o.act][0](a + ins[1][0]), va + ins[1][1])
        elif o.kind == abi.OP_CONCAT:
            vals[o.out] = tuple(torch.cat([i[k] for i in ins], 1) for k in (0, 1))
        elif o.kind == abi.OP_UPSAMPLE2X:
            vals[o.out] = tuple(i.repeat_interleave(2, 2).repeat_interleave(2, 3) for i in (a, va))
        else:
            raise ValueError("operator kind %d" % o.kind)
    v, var = vals[ops[-1].out]
    return v, var.sqrt()


def worst(got, ops, x, blob):
    """The largest error of a value, in standard deviations; infinite if one is not a number."""
    want, sd = evaluate(ops, x, blob)
    r = (torch.from_numpy(np.asarray(got, np.float64)) - want).abs() / sd
    return math.inf if torch.isnan(r).any() else float(r.max())
