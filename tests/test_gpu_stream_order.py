"""How calls on different streams are ordered (StreamOrder, runtime.hpp): a call waits for the previous call's work and for
nothing else.  Other streams of the program keep running, a capture that is open elsewhere stays open, an earlier stream may be
gone, and the results are those of calls made one after the other."""
import ctypes
import time

import numpy as np
import pytest
import torch

from nncv_amd import abi, synth
from gpu_util import Conv, Model, dev

pytestmark = pytest.mark.gpu

N, H, W = 2, 64, 64


@pytest.fixture(scope="module")
def half_blob():
    return synth.round_fp16(synth.resnet18_params())


def half_a_second():
    """Cycles for torch.cuda._sleep that take about half a second (it ends by itself)."""
    torch.cuda._sleep(1000)
    torch.cuda.synchronize()
    t = time.perf_counter()
    torch.cuda._sleep(2_000_000)
    torch.cuda.synchronize()
    return int(2_000_000 * 0.5 / (time.perf_counter() - t))


def asleep(stream, cycles):
    """An event behind half a second of work on `stream`."""
    e = torch.cuda.Event()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(cycles)
        e.record()
    return e


def forward(m, x, out, stream):
    return abi.lib().nncv_hip_resnet18_forward(m.h, x.data_ptr(), N, H, W, out.data_ptr(), stream)


def image(seed):
    return dev(synth.round_fp16(synth.uniform(seed, (N, 3, H, W), 0.0, 1.0)), abi.F16)


def test_a_second_stream_waits_for_the_first_one_only(half_blob):
    m, xa, xb = Model(half_blob, abi.F16, abi.ALGO_IGEMM), image(81), image(82)
    want_a, want_b = m(xa).clone(), m(xb).clone()
    oa, ob = torch.empty_like(want_a), torch.empty_like(want_b)
    s1, s2, other = (torch.cuda.Stream() for _ in range(3))
    m2 = Model(half_blob, abi.F16, abi.ALGO_IGEMM)  # a handle that has seen one stream only
    abi.check(forward(m2, xa, oa, s1.cuda_stream))
    torch.cuda.synchronize()
    oa.zero_()
    cycles = half_a_second()
    torch.cuda.synchronize()
    busy = asleep(other, cycles)
    abi.check(forward(m2, xa, oa, s1.cuda_stream))
    abi.check(forward(m2, xb, ob, s2.cuda_stream))
    assert not busy.query(), "the calls returned only when an unrelated stream had finished"
    torch.cuda.synchronize()
    assert torch.equal(oa, want_a) and torch.equal(ob, want_b)


def test_a_host_call_does_not_wait_for_unrelated_streams():
    """_mlir_ciface_matmul behind a device call that left work pending, again and again."""
    a, b = synth.uniform(83, (64, 48), -1, 1), synth.uniform(84, (48, 80), -1, 1)
    c = np.zeros((64, 80), np.float32)
    abi.matmul(a, b, c)
    ad, bd, cd = dev(a), dev(b), torch.zeros((64, 80), device="cuda")
    cycles = half_a_second()
    torch.cuda.synchronize()
    # a stream whose work the library's own stream does not queue behind (streams share a few hardware queues)
    for other in [torch.cuda.Stream() for _ in range(8)]:
        busy = asleep(other, cycles)
        abi.matmul(a, b, np.zeros((64, 80), np.float32))
        free = not busy.query()
        torch.cuda.synchronize()
        if free:
            break
    else:
        pytest.skip("every stream shares a hardware queue with the library's")
    s1 = next(s for s in (torch.cuda.Stream() for _ in range(8)) if s.cuda_stream != other.cuda_stream)
    for _ in range(3):
        abi.check(abi.lib().nncv_hip_matmul_f32(ad.data_ptr(), bd.data_ptr(), cd.data_ptr(), 64, 80, 48, s1.cuda_stream))
        torch.cuda.synchronize()  # the device call has ended; the library has not been told
        busy = asleep(other, cycles)
        got = np.zeros((64, 80), np.float32)
        abi.matmul(a, b, got)
        assert not busy.query()
        assert np.array_equal(got, c)
        torch.cuda.synchronize()


def test_calls_on_two_streams_while_a_capture_is_open(half_blob):
    m, xa, xb = Model(half_blob, abi.F16, abi.ALGO_IGEMM), image(85), image(86)
    want_a, want_b = m(xa).clone(), m(xb).clone()
    oa, ob = torch.empty_like(want_a), torch.empty_like(want_b)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    fresh = Model(half_blob, abi.F16, abi.ALGO_IGEMM)
    abi.check(forward(fresh, xa, oa, s1.cuda_stream))  # (the workspace is there from now on)
    torch.cuda.synchronize()
    v = torch.zeros(64, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):  # global mode: what is unsafe under a capture fails for every thread
        v.add_(1.0)
        ra = forward(fresh, xa, oa, s1.cuda_stream)
        rb = forward(fresh, xb, ob, s2.cuda_stream)
        message = abi.lib().nncv_hip_last_error().decode()
    assert ra == 0 and rb == 0, message
    torch.cuda.synchronize()
    assert torch.equal(oa, want_a) and torch.equal(ob, want_b)
    for k in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert float(v[0]) == k + 1


def test_an_earlier_stream_may_be_gone(half_blob):
    L = abi.lib()
    m, xa, xb = Model(half_blob, abi.F16, abi.ALGO_IGEMM), image(87), image(88)
    want_a, want_b = m(xa).clone(), m(xb).clone()
    s2 = torch.cuda.Stream()
    for rounds in (1, 7):  # a pass run directly, and replayed
        fresh, oa, ob = Model(half_blob, abi.F16, abi.ALGO_IGEMM), torch.empty_like(want_a), torch.empty_like(want_b)
        s1 = ctypes.c_void_p()
        assert L.hipStreamCreate(ctypes.byref(s1)) == 0
        for _ in range(rounds):
            abi.check(forward(fresh, xa, oa, s1))
        assert L.hipStreamDestroy(s1) == 0
        abi.check(forward(fresh, xb, ob, s2.cuda_stream))
        torch.cuda.synchronize()
        assert torch.equal(oa, want_a) and torch.equal(ob, want_b)


def test_a_pass_recorded_into_the_callers_graph(half_blob):
    """The recorded launches neither wait for an event nor complete one; eager passes in between stay ordered as before."""
    m, xa, xb = Model(half_blob, abi.F16, abi.ALGO_IGEMM), image(89), image(90)
    want_a, want_b = m(xa).clone(), m(xb).clone()
    oa, ob = torch.empty_like(want_a), torch.empty_like(want_b)
    torch.cuda.synchronize()
    g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(g, stream=side):
        abi.check(forward(m, xa, oa, torch.cuda.current_stream().cuda_stream))
    for k in range(3):
        oa.fill_(float(k))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(oa, want_a), k
        abi.check(forward(m, xb, ob, side.cuda_stream))
        torch.cuda.synchronize()
        assert torch.equal(ob, want_b), k


@pytest.mark.parametrize("layout", [abi.NHWC, abi.NCHW])
def test_a_chain_of_layers_over_streams_without_waits(layout):
    """Each call reads what the one before wrote, on another stream: one launch a call (NHWC), and several (NCHW)."""
    c, n = 64, 4
    w = (synth.normal(91, (c, c, 3, 3)) * 0.05).astype(np.float32)
    conv = Conv(abi.F32, w, 1, 1)
    x = dev(synth.normal(92, (n, 28, 28, c) if layout == abi.NHWC else (n, c, 28, 28)))
    bufs = [torch.empty_like(x) for _ in range(9)]

    def chain(streams):
        src = x
        for k, b in enumerate(bufs):
            abi.check(abi.lib().nncv_hip_conv_forward(conv.h, src.data_ptr(), n, 28, 28, layout, None, b.data_ptr(), streams[k % len(streams)]))
            src = b
        torch.cuda.synchronize()
        return bufs[-1].clone()

    want = chain([torch.cuda.Stream().cuda_stream])
    for b in bufs:
        b.zero_()
    torch.cuda.synchronize()
    assert torch.equal(chain([torch.cuda.Stream().cuda_stream for _ in range(4)]), want)


@pytest.mark.parametrize("M,N,K", [(20, 30, 40), (700, 500, 64)])
def test_products_accumulate_over_streams(M, N, K):
    """C += A.B over and over, each call on another stream than the one before: every call reads what the previous one wrote, from
    other compute units and caches than those that wrote it.  Whole numbers, so the sum is exact."""
    g = torch.Generator().manual_seed(7)
    a, b = (torch.randint(-3, 4, s, generator=g).float().cuda() for s in ((M, K), (K, N)))
    c = torch.zeros((M, N), device="cuda")
    streams = [torch.cuda.Stream().cuda_stream for _ in range(3)]
    torch.cuda.synchronize()
    for k in range(600):
        abi.check(abi.lib().nncv_hip_matmul_f32(a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, streams[k % 3]))
    torch.cuda.synchronize()
    assert torch.equal(c.cpu(), 600 * (a.cpu() @ b.cpu()))
