"""Ragged M and N on the whole-tile assembly GEMM (the last tile row and column overlap the
ones before them): the same bits as the LDS-DMA kernel's edge tiles on random operands."""
import os

import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc
from tests.tolerances import assert_gemm_close

pytestmark = pytest.mark.gpu
D = th.TileDtype
ORC = {D.F32: orc.F32, D.F16: orc.F16, D.BF16: orc.BF16}


def fill(dev, stream, n, dtype, std, seed):
    b = dev.alloc(n, dtype)
    th.fill_random(b, n, dtype, "normal", 0.0, std, seed, stream)
    return b


def both(call, c, stream):
    out = []
    old = os.environ.get("TILERS_HIP_GEMM_ASM")
    try:
        for asm in ("1", "0"):
            os.environ["TILERS_HIP_GEMM_ASM"] = asm
            c.copy_from_host(np.full(len(c), 3, c.dtype.host_dtype), stream)
            call()
            out.append(c.copy_to_host(stream))
    finally:
        if old is None:
            os.environ.pop("TILERS_HIP_GEMM_ASM", None)
        else:
            os.environ["TILERS_HIP_GEMM_ASM"] = old
    return out


# enough 256 x 256 tiles, and little enough K, that smaller tiles or a split of K are estimated
# longer (for all but the 1281-row product by half as much again)
@pytest.mark.parametrize("m,k,n,ind,outd,bt,bsz", [
    (3841, 256, 4096, D.BF16, D.F32, False, 1),   # one row over: 255 rows recomputed
    (4095, 384, 3848, D.F16, D.F16, False, 1),    # one short of whole; eight columns over
    (2048, 256, 4088, D.BF16, D.BF16, False, 2),  # ragged N only, a batch
    (3900, 256, 3900, D.F16, D.F32, True, 1),     # B stored N x K: N not a multiple of 8
    (1281, 384, 3999, D.BF16, D.F16, True, 3),    # odd N: rows of C on odd 2-byte offsets
    (1501, 384, 2497, D.BF16, D.F16, True, 4),    # odd N: rows of C on odd 2-byte offsets
])
def test_ragged_matmul_same_bits_as_dma_kernel(dev, stream, m, k, n, ind, outd, bt, bsz):
    a = fill(dev, stream, bsz * m * k, ind, 1.0, 0x51)
    b = fill(dev, stream, bsz * k * n, ind, 0.05, 0x52)
    c = dev.alloc(bsz * m * n + 512, outd)
    got, ref = both(lambda: th.matmul(a, b, c, m, k, n, ind, outd, bt, batch=bsz, stream=stream),
                    c, stream)
    assert np.array_equal(got, ref)   # the guard after C among it


@pytest.mark.parametrize("ind", [D.BF16, D.F16])
@pytest.mark.parametrize("outd", [D.BF16, D.F16])
@pytest.mark.parametrize("bt", [False, True])
def test_ragged_silu_mul_close_to_dma_kernel(dev, stream, ind, outd, bt):
    """Every variant of the fused program, whole and overlapping tiles, against the LDS-DMA
    kernel's expf and division: the GEMM tolerance."""
    m, k, n = 4000, 256, 3848
    a = fill(dev, stream, m * k, ind, 1.0, 0x71)
    b = fill(dev, stream, k * n, ind, 0.2, 0x72)
    up = fill(dev, stream, m * n, outd, 1.0, 0x73)
    c = dev.alloc(m * n, outd)
    got, ref = both(lambda: th.matmul_silu_mul(a, b, up, c, m, k, n, ind, outd, bt, stream=stream),
                    c, stream)
    assert_gemm_close(orc.widen(got, ORC[outd]), orc.widen(ref, ORC[outd]), "silu_mul",
                      u16_dtype=ORC[outd])


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("m,k,n,dt,bt", [(3900, 256, 3848, D.F16, False),
                                         (4000, 256, 3848, D.BF16, True)])
def test_ragged_silu_mul(dev, stream, in_place, m, k, n, dt, bt):
    """Tiles that overlap must not read what another wrote where UP and C are one buffer."""
    a = fill(dev, stream, m * k, dt, 1.0, 0x61)
    b = fill(dev, stream, k * n, dt, 0.05, 0x62)
    up = fill(dev, stream, m * n, dt, 1.0, 0x63)
    up_host = up.copy_to_host(stream)
    c = up if in_place else dev.alloc(m * n, dt)
    th.matmul_silu_mul(a, b, up, c, m, k, n, dt, dt, bt, stream=stream)
    got = orc.widen(c.copy_to_host(stream), ORC[dt]).reshape(m, n)[-300:]
    ref = orc.matmul_silu_mul(a.copy_to_host(stream), b.copy_to_host(stream), up_host, m, k, n,
                              ORC[dt], ORC[dt], b_trans=bt, row0=m - 300, nrows=300)
    assert_gemm_close(got, orc.widen(ref.reshape(-1), ORC[dt]).reshape(300, n),
                      f"silu_mul in_place={in_place}", u16_dtype=ORC[dt])
