"""Two threads queue split products on one stream: each call's partials and merge go in one
piece, also while the stream's scratch grows."""
import threading

import numpy as np
import pytest

import tilers_hip as th

pytestmark = pytest.mark.gpu
D = th.TileDtype


def test_two_threads_one_stream(dev):
    stream = dev.create_stream()
    rng = np.random.default_rng(3)
    shapes = [(64, 2048, 64 + 64 * i) for i in range(12)]   # (m, k, n): growing partials

    def upload(x):
        b = dev.alloc(x.size, D.F32)
        b.copy_from_host(x.reshape(-1), stream)
        return b

    work = []
    for t in range(2):
        for m, k, n in shapes:
            # whole numbers up to 3: every order of the sums gives the same f32
            a = rng.integers(-3, 4, (m, k)).astype(np.float32)
            b = rng.integers(-3, 4, (k, n)).astype(np.float32)
            work.append((t, upload(a), upload(b), dev.alloc(m * n, D.F32), (m, k, n),
                         (a.astype(np.float64) @ b).reshape(-1)))
    stream.synchronize()
    start, errors = threading.Barrier(2), []

    def run(t):
        try:
            start.wait(timeout=30)
            for _ in range(5):
                for own, a, b, c, (m, k, n), _ in work:
                    if own == t:
                        th.matmul(a, b, c, m, k, n, D.F32, D.F32, False, stream=stream)
        except Exception as e:   # shown by the test's thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for _, _, _, c, shape, ref in work:
        assert np.array_equal(c.copy_to_host(stream), ref.astype(np.float32)), shape
    stream.close()


def test_two_threads_per_thread_stream(dev, stream):
    """hipStreamPerThread is one handle for a stream of its own in each thread: split products
    and a split decode without a workspace, repeated by two threads on it at the same time,
    give what one thread gives on an ordinary stream."""
    from types import SimpleNamespace
    mine = SimpleNamespace(handle=2)   # hipStreamPerThread
    rng = np.random.default_rng(4)
    m, k, n, rounds = 64, 4096, 96, 40
    B, L, NH, NKV, Dh = 1, 6000, 8, 2, 128

    def upload(x):
        b = dev.alloc(x.size, D.F32)
        b.copy_from_host(x.reshape(-1).astype(np.float32), stream)
        return b

    def product(w, c, s):
        th.matmul(w.a, w.b, c, m, k, n, D.F32, D.F32, False, stream=s)

    def decode(w, o, s):
        th.attention_decode(w.q, w.k, w.v, o, B, L, L, Dh, NH, NKV, D.F32, None, 0, s)

    work = []
    for _ in range(2):
        a, b = rng.integers(-3, 4, (m, k)), rng.integers(-3, 4, (k, n))
        w = SimpleNamespace(a=upload(a), b=upload(b), ref=(a @ b).reshape(-1).astype(np.float32),
                            q=upload(rng.standard_normal(NH * Dh)),
                            k=upload(rng.standard_normal(NKV * L * Dh)),
                            v=upload(rng.standard_normal(NKV * L * Dh)),
                            c=[dev.alloc(m * n, D.F32) for _ in range(rounds)],
                            o=[dev.alloc(NH * Dh, D.F32) for _ in range(rounds + 1)])
        decode(w, w.o[rounds], stream)
        work.append(w)
    stream.synchronize()
    start, errors = threading.Barrier(2), []

    def run(w):
        try:
            start.wait(timeout=30)
            for i in range(rounds):
                product(w, w.c[i], mine)
                decode(w, w.o[i], mine)
            th._lib.check(th.lib().th_stream_sync(mine.handle))
        except Exception as e:   # shown by the test's thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(w,)) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for w in work:
        once = w.o[rounds].copy_to_host(stream)
        for i in range(rounds):
            assert np.array_equal(w.c[i].copy_to_host(stream), w.ref), i
            assert np.array_equal(w.o[i].copy_to_host(stream), once), i
