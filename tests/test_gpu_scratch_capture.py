"""Split f32 products and f32 decode beside graphs: eager calls that need a buffer while another
stream is recorded, and the same calls recorded themselves (then unsplit, without a buffer)."""
from ctypes import byref, c_size_t, c_void_p

import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
D = th.TileDtype
GLOBAL, THREAD_LOCAL = 0, 1   # hipStreamCaptureMode


def put(dev, stream, x):
    b = dev.alloc(x.size, D.F32)
    b.copy_from_host(np.ascontiguousarray(x, np.float32).reshape(-1), stream)
    return b


class Product:
    """64 x 4096 x 96, split over K when eager; exact in whole numbers."""
    m, k, n = 64, 4096, 96

    def __init__(self, dev, stream, rng):
        a, b = rng.integers(-3, 4, (self.m, self.k)), rng.integers(-3, 4, (self.k, self.n))
        self.a, self.b = put(dev, stream, a), put(dev, stream, b)
        self.ref = (a @ b).astype(np.float32).reshape(-1)
        self.out = dev.alloc(self.ref.size, D.F32)

    def call(self, stream):
        th.matmul(self.a, self.b, self.out, self.m, self.k, self.n, D.F32, D.F32, stream=stream)

    def check(self, stream):
        assert np.array_equal(self.out.copy_to_host(stream), self.ref)


class Decode:
    """2 sequences of 3000 positions, split over the positions when eager."""
    B, L, NH, NKV, Dh = 2, 3000, 8, 2, 128

    def __init__(self, dev, stream, rng):
        q = rng.standard_normal((self.B, self.NH, self.Dh)).astype(np.float32)
        k, v = (rng.standard_normal((self.B, self.NKV, self.L, self.Dh)).astype(np.float32)
                for _ in range(2))
        self.q, self.k, self.v = (put(dev, stream, x) for x in (q, k, v))
        self.ref = orc.attention_decode(q, k, v, orc.F32, self.B, self.L, self.L, self.Dh, self.NH,
                                        self.NKV).reshape(-1)
        self.out = dev.alloc(self.ref.size, D.F32)

    def call(self, stream):
        th.attention_decode(self.q, self.k, self.v, self.out, self.B, self.L, self.L, self.Dh,
                            self.NH, self.NKV, D.F32, None, 0, stream)

    def check(self, stream):
        # weighted means of V ~ N(0, 1): the bound of tests/test_gpu_f32_attention.py
        assert np.abs(self.out.copy_to_host(stream) - self.ref).max() < 1e-5


def record(stream, mode, body):
    hip, graph, run = th.lib(), c_void_p(), c_void_p()
    stream.synchronize()
    assert hip.hipStreamBeginCapture(c_void_p(stream.handle), mode) == 0
    body()
    assert hip.hipStreamEndCapture(c_void_p(stream.handle), byref(graph)) == 0
    assert hip.hipGraphInstantiate(byref(run), graph, None, None, c_size_t(0)) == 0
    return graph, run


def drop(graph, run):
    assert th.lib().hipGraphExecDestroy(run) == 0 and th.lib().hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("op", [Product, Decode])
def test_buffer_while_another_stream_is_recorded(dev, op):
    rng = np.random.default_rng(8)
    recorded, eager = dev.create_stream(), dev.create_stream()   # no buffer yet
    x = rng.standard_normal((4, 256)).astype(np.float32)
    xb, yb = put(dev, recorded, x), put(dev, recorded, np.zeros_like(x))
    work = op(dev, eager, rng)
    eager.synchronize()

    def body():
        th.softmax(xb, yb, 4, 256, D.F32, recorded)
        work.call(eager)

    graph, run = record(recorded, GLOBAL, body)
    work.check(eager)
    assert th.lib().hipGraphLaunch(run, c_void_p(recorded.handle)) == 0
    got = yb.copy_to_host(recorded).reshape(x.shape)
    assert np.abs(got - orc.softmax(x, 4, 256).reshape(x.shape)).max() < 1e-6
    drop(graph, run)


@pytest.mark.parametrize("op", [Product, Decode])
def test_recorded_unsplit(dev, op):
    rng = np.random.default_rng(9)
    s = dev.create_stream()
    work, other = op(dev, s, rng), op(dev, s, rng)
    graph, run = record(s, THREAD_LOCAL, lambda: work.call(s))
    for _ in range(3):
        work.out.copy_from_host(np.zeros_like(work.ref), s)
        other.call(s)   # eager work between the replays, split on the stream's buffer
        assert th.lib().hipGraphLaunch(run, c_void_p(s.handle)) == 0
        other.call(s)
        work.check(s)
        other.check(s)
    s.synchronize()
    drop(graph, run)
