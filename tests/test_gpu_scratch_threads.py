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
