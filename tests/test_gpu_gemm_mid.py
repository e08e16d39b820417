"""16-bit products on 128 x 64 and 64 x 64 tiles, with and without a split of K: bit-exact on
integer-valued inputs (every f32 partial sum is a whole number, in any order)."""
import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc
from tests.tolerances import assert_gemm_close

pytestmark = pytest.mark.gpu
D = th.TileDtype
ORC = {D.F32: orc.F32, D.F16: orc.F16, D.BF16: orc.BF16}


def put(dev, stream, x, dtype, offset=0):
    b = dev.alloc(x.size + offset, dtype)
    b.copy_from_host(np.concatenate([np.zeros(offset, x.dtype), x.reshape(-1)]), stream)
    return b


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m,k,n,bsz", [
    (65, 8, 8, 1),         # K less than a stage, one chunk of it
    (64, 64, 64, 1),       # one stage, one tile
    (127, 72, 72, 2),      # tail of one chunk, ragged tiles, a batch
    (129, 320, 136, 1),    # as many stages as the ring and one more
    (300, 1096, 200, 1),   # tail, K split with a short last slice
    (200, 4096, 1024, 1),  # K split
    (1000, 504, 1000, 1),  # 64 x 64, about one per CU, K % 32 != 0
    (2000, 264, 2056, 1),  # 128 x 64, several per CU
    (70, 128, 264, 9),     # a batch of ragged tiles
])
def test_mid_tiles_exact(dev, stream, trans, m, k, n, bsz):
    rng = np.random.default_rng(m + 7 * k + 13 * n)
    a = rng.integers(-4, 5, (bsz, m, k)).astype(np.float32)
    b = rng.integers(-4, 5, (bsz, k, n)).astype(np.float32)
    ref = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32).ravel()
    bs = np.ascontiguousarray(b.transpose(0, 2, 1)) if trans else b
    for dt, out, off in ((D.BF16, D.F32, 0), (D.F16, D.F16, 0), (D.BF16, D.BF16, 1)):
        ab, bb = (put(dev, stream, orc.narrow(x.ravel(), ORC[dt]), dt) for x in (a, bs))
        guard = np.full(ref.size + 256, 9, out.host_dtype)
        cb = put(dev, stream, guard, out, off)   # off: C not on 16 bytes, scalar stores
        th.matmul(ab, bb, cb.as_raw_ptr() + off * out.itemsize, m, k, n, dt, out, trans, batch=bsz,
                  stream=stream)
        got = cb.copy_to_host(stream)[off:]
        want = ref if out == D.F32 else orc.narrow(ref, ORC[out])
        assert np.array_equal(got[:ref.size], want)
        assert np.array_equal(got[ref.size:], guard[ref.size:])   # nothing past C


@pytest.mark.parametrize("dt,out", [(D.BF16, D.BF16), (D.F16, D.F32), (D.BF16, D.F16)])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m,k,n", [(130, 4096, 136), (500, 200, 1000), (90, 96, 44)])
def test_mid_tiles_silu_mul(dev, stream, dt, out, trans, m, k, n):
    """In place (UP and C one buffer): every element is read and written by one lane."""
    if not trans and n % 8:
        n = 48
    rng = np.random.default_rng(m + n)
    a = orc.narrow(rng.standard_normal(m * k).astype(np.float32), ORC[dt])
    b = orc.narrow((rng.standard_normal(n * k) * 0.05).astype(np.float32), ORC[dt])
    up = rng.standard_normal(m * n).astype(np.float32)
    up = up if out == D.F32 else orc.narrow(up, ORC[out])
    cb = put(dev, stream, up, out)
    th.matmul_silu_mul(put(dev, stream, a, dt), put(dev, stream, b, dt), cb, cb, m, k, n, dt, out,
                       trans, stream=stream)
    got = cb.copy_to_host(stream)
    bw = orc.widen(b, ORC[dt]).astype(np.float64)
    x = (orc.widen(a, ORC[dt]).reshape(m, k).astype(np.float64)
         @ (bw.reshape(n, k).T if trans else bw.reshape(k, n)))
    upw = up if out == D.F32 else orc.widen(up, ORC[out])
    ref = (x / (1 + np.exp(-x)) * upw.reshape(m, n)).astype(np.float32).reshape(-1)
    if out == D.F32:
        assert_gemm_close(got, ref, "silu_mul")
    else:
        assert_gemm_close(orc.widen(got, ORC[out]), ref, "silu_mul", u16_dtype=ORC[out])


@pytest.mark.parametrize("warm", [True, False])
def test_mid_tiles_recorded(dev, warm):
    """A split product recorded into a graph: split if the stream's scratch is there already,
    unsplit if not (recording never allocates), the same bits on every replay."""
    from ctypes import byref, c_size_t, c_void_p

    hip, s = th.lib(), dev.create_stream()
    m, k, n = 8, 4096, 1024
    rng = np.random.default_rng(5)
    a = rng.integers(-4, 5, (m, k)).astype(np.float32)
    b = rng.integers(-4, 5, (k, n)).astype(np.float32)
    ab, bb = (put(dev, s, orc.narrow(x.ravel(), orc.BF16), D.BF16) for x in (a, b))
    zero = np.zeros(m * n, np.float32)
    cb, other = put(dev, s, zero, D.F32), put(dev, s, zero, D.F32)

    def call(c):
        th.matmul(ab, bb, c, m, k, n, D.BF16, D.F32, stream=s)

    if warm:
        call(other)
    s.synchronize()
    graph, run = c_void_p(), c_void_p()
    assert hip.hipStreamBeginCapture(c_void_p(s.handle), 1) == 0
    call(cb)
    assert hip.hipStreamEndCapture(c_void_p(s.handle), byref(graph)) == 0
    assert hip.hipGraphInstantiate(byref(run), graph, None, None, c_size_t(0)) == 0
    ref = (a.astype(np.float64) @ b).astype(np.float32).ravel()
    for _ in range(4):
        cb.copy_from_host(zero, s)
        call(other)   # eager work through the same scratch
        assert hip.hipGraphLaunch(run, c_void_p(s.handle)) == 0
        call(other)
        assert np.array_equal(cb.copy_to_host(s), ref)
        assert np.array_equal(other.copy_to_host(s), ref)
    s.synchronize()
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
