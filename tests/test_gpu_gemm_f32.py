"""f32 products on 64 x 64 tiles, with and without a split of K: bit-exact on integer-valued
inputs (every partial sum is a whole number below 2^24, whatever the order)."""
import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc

from tests.tolerances import assert_gemm_close

pytestmark = pytest.mark.gpu
D = th.TileDtype


def put(dev, stream, x):
    b = dev.alloc(x.size, D.F32)
    b.copy_from_host(x.reshape(-1), stream)
    return b


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m,k,n,bsz", [
    (1, 1, 1, 1),          # fewer than four values in every row
    (5, 3, 2, 2),
    (63, 64, 65, 1),       # tile edges; K one whole stage
    (64, 65, 64, 1),       # K one past it; unaligned rows
    (65, 67, 61, 3),       # ragged in every dimension, a batch
    (128, 128, 132, 1),    # aligned rows, a column group past the tile edge
    (33, 1027, 70, 1),     # split K, last slice short, unaligned rows
    (64, 4096, 64, 1),     # one tile, the largest number of slices
    (200, 2000, 300, 1),   # split K, aligned rows
    (999, 256, 1000, 1),   # one round of workgroups: no split
])
def test_matmul_f32_small_tiles_exact(dev, stream, trans, m, k, n, bsz):
    rng = np.random.default_rng(m + 7 * k + 13 * n)
    a = rng.integers(-8, 9, (bsz, m, k)).astype(np.float32)
    b = rng.integers(-8, 9, (bsz, k, n)).astype(np.float32)
    ref = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    cb = put(dev, stream, np.full(bsz * m * n + 64, 9.5, np.float32))
    th.matmul(put(dev, stream, a), put(dev, stream, b.transpose(0, 2, 1).copy() if trans else b),
              cb, m, k, n, D.F32, D.F32, trans, batch=bsz, stream=stream)
    got = cb.copy_to_host(stream)
    assert np.array_equal(got[:ref.size].reshape(ref.shape), ref)
    assert (got[ref.size:] == 9.5).all()   # nothing written past C


@pytest.mark.parametrize("out_dt", [D.F32, D.F16, D.BF16])
@pytest.mark.parametrize("m,k,n", [(70, 90, 130), (40, 3000, 50)])   # plain and split K
def test_matmul_f32_small_tiles_silu_mul(dev, stream, out_dt, m, k, n):
    rng = np.random.default_rng(m)
    o = {D.F32: orc.F32, D.F16: orc.F16, D.BF16: orc.BF16}[out_dt]
    a = rng.standard_normal(m * k).astype(np.float32)
    b = (rng.standard_normal(k * n) * 0.05).astype(np.float32)
    up32 = rng.standard_normal(m * n).astype(np.float32)
    up = up32 if out_dt == D.F32 else orc.narrow(up32, o)
    ub, cb = dev.alloc(m * n, out_dt), dev.alloc(m * n, out_dt)
    ub.copy_from_host(up, stream)
    th.matmul_silu_mul(put(dev, stream, a), put(dev, stream, b), ub, cb, m, k, n, D.F32, out_dt,
                       stream=stream)
    raw = cb.copy_to_host(stream)
    x = a.reshape(m, k).astype(np.float64) @ b.reshape(k, n).astype(np.float64)
    upw = up if out_dt == D.F32 else orc.widen(up, o)
    ref = (x / (1 + np.exp(-x)) * upw.reshape(m, n)).astype(np.float32).reshape(-1)
    if out_dt == D.F32:
        assert_gemm_close(raw, ref, "silu_mul f32")
    else:
        assert_gemm_close(orc.widen(raw, o), ref, "silu_mul", u16_dtype=o)
