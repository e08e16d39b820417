"""16-bit products with few rows of A and B stored N x K: bit-exact on integer-valued inputs
(every f32 partial sum is a whole number, whatever the split of K over waves)."""
import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc
from tests.tolerances import assert_gemm_close

pytestmark = pytest.mark.gpu
D = th.TileDtype
ORC = {D.F32: orc.F32, D.F16: orc.F16, D.BF16: orc.BF16}


def put(dev, stream, x, dtype):
    b = dev.alloc(x.size, dtype)
    b.copy_from_host(x.reshape(-1), stream)
    return b


@pytest.mark.parametrize("dt", [D.BF16, D.F16])
@pytest.mark.parametrize("m,k,n,bsz", [
    (1, 8, 1, 1),          # no whole stage: the tail of K alone
    (8, 64, 16, 1),        # one stage, one wave of four
    (9, 56, 17, 2),        # sixteen-row variant, a column past the block, a batch
    (8, 200, 300, 1),      # three stages (a wave without any), then a tail
    (16, 1096, 33, 3),     # more stages than the ring, tail of one 8-value chunk
    (17, 320, 40, 1),      # 32-row variant
    (33, 576, 31, 1),      # 64-row variant, a wave of three stages
    (64, 4096, 64, 1),     # largest M
    (5, 136, 6563, 1),     # two column blocks per workgroup, ragged
    (12, 72, 13000, 1),    # four column blocks, ragged
    (64, 264, 12999, 1),   # four column blocks, largest M
    (3, 64, 900, 16),      # four column blocks by the batch
])
def test_few_rows_exact(dev, stream, dt, m, k, n, bsz):
    rng = np.random.default_rng(m + 7 * k + 13 * n)
    a = rng.integers(-4, 5, (bsz, m, k)).astype(np.float32)
    b = rng.integers(-4, 5, (bsz, n, k)).astype(np.float32)
    ref = (a.astype(np.float64) @ b.transpose(0, 2, 1).astype(np.float64)).astype(np.float32)
    ab, bb = (put(dev, stream, orc.narrow(x.ravel(), ORC[dt]), dt) for x in (a, b))
    for out in (D.F32, dt):
        guard = np.full(bsz * m * n + 256, 9, out.host_dtype)
        cb = put(dev, stream, guard, out)
        th.matmul(ab, bb, cb, m, k, n, dt, out, True, batch=bsz, stream=stream)
        got = cb.copy_to_host(stream)
        want = ref.ravel() if out == D.F32 else orc.narrow(ref.ravel(), ORC[out])
        assert np.array_equal(got[:ref.size], want)
        assert np.array_equal(got[ref.size:], guard[ref.size:])   # nothing past C


@pytest.mark.parametrize("dt,out", [(D.BF16, D.BF16), (D.F16, D.F32), (D.BF16, D.F16)])
@pytest.mark.parametrize("m,k,n", [(8, 4096, 100), (20, 1000, 7000), (64, 512, 50)])
def test_few_rows_silu_mul(dev, stream, dt, out, m, k, n):
    rng = np.random.default_rng(m + n)
    a = orc.narrow(rng.standard_normal(m * k).astype(np.float32), ORC[dt])
    b = orc.narrow((rng.standard_normal(n * k) * 0.05).astype(np.float32), ORC[dt])
    up = rng.standard_normal(m * n).astype(np.float32)
    up = up if out == D.F32 else orc.narrow(up, ORC[out])
    ub, cb = put(dev, stream, up, out), dev.alloc(m * n, out)
    th.matmul_silu_mul(put(dev, stream, a, dt), put(dev, stream, b, dt), ub, cb, m, k, n, dt, out,
                       True, stream=stream)
    got = cb.copy_to_host(stream)
    x = (orc.widen(a, ORC[dt]).reshape(m, k).astype(np.float64)
         @ orc.widen(b, ORC[dt]).reshape(n, k).T.astype(np.float64))
    upw = up if out == D.F32 else orc.widen(up, ORC[out])
    ref = (x / (1 + np.exp(-x)) * upw.reshape(m, n)).astype(np.float32).reshape(-1)
    if out == D.F32:
        assert_gemm_close(got, ref, "silu_mul")
    else:
        assert_gemm_close(orc.widen(got, ORC[out]), ref, "silu_mul", u16_dtype=ORC[out])
