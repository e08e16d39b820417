"""Softmax and RMSNorm with a workgroup per row (rows that the aligned register kernels do not
take): column counts around each size of the kernel, pointers off 16 bytes, in place, masks."""
import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc
from tests.tolerances import assert_softmax_close, assert_within_ulp16

pytestmark = pytest.mark.gpu
D = th.TileDtype
ORC = {D.F32: orc.F32, D.F16: orc.F16, D.BF16: orc.BF16}


def rows_op(dev, stream, op, x, rows, cols, dtype, x_off=0, in_place=False):
    """op on rows placed x_off elements into a buffer, guard values around the output."""
    pad = np.full(x_off + 32, 3, x.dtype)
    xb = dev.alloc(x.size + x_off + 32, dtype)
    xb.copy_from_host(np.concatenate([pad[:x_off], x.ravel(), pad[:32]]), stream)
    yb = xb
    if not in_place:
        yb = dev.alloc(x.size + x_off + 32, dtype)
        yb.copy_from_host(np.full(x.size + x_off + 32, 3, x.dtype), stream)
    off = x_off * dtype.itemsize
    if op == "softmax":
        th.softmax(xb.as_raw_ptr() + off, yb.as_raw_ptr() + off, rows, cols, dtype, stream)
    else:
        th.rms_norm(xb.as_raw_ptr() + off, yb.as_raw_ptr() + off, rows, cols, 1e-6, dtype, stream)
    got = yb.copy_to_host(stream)
    assert (got[:x_off] == pad[:x_off]).all() and (got[x_off + x.size:] == pad[:32]).all()
    return got[x_off:x_off + x.size]


def check(op, got, xw, rows, cols, dtype):
    xw = xw.reshape(rows, cols).astype(np.float32)
    if op == "softmax":
        ref = orc.softmax(xw, rows, cols)
        if dtype == D.F32:
            assert_softmax_close(got.reshape(rows, cols), ref)
        else:
            assert_within_ulp16(orc.widen(got, ORC[dtype]).reshape(rows, cols), ref, ORC[dtype])
        return
    x64 = xw.astype(np.float64)
    ref = x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-6)
    if dtype == D.F32:
        # one rounding each of the sum's terms, the root, the reciprocal and the product
        assert (np.abs(got.reshape(rows, cols) - ref) <= 1e-5 * np.abs(ref) + 1e-30).all()
    else:
        assert_within_ulp16(orc.widen(got, ORC[dtype]).reshape(rows, cols),
                            ref.astype(np.float32), ORC[dtype])


# vectors per row around 64 x 4, 256 x 4, 1024 x {2, 4, 8, 13, 16}; rows enough for the rule
SIZES = [(3, 1), (5, 2), (70, 255), (9, 257), (40, 1025), (40, 2047), (40, 2049), (60, 4097),
         (130, 8193), (130, 13313), (130, 16384)]


@pytest.mark.parametrize("op", ["softmax", "rms_norm"])
@pytest.mark.parametrize("dtype", [D.F32, D.BF16, D.F16])
@pytest.mark.parametrize("rows,vecs", SIZES)
def test_rows_wide_sizes(dev, stream, op, dtype, rows, vecs):
    e = 16 // dtype.itemsize
    cols = vecs * e - (1 if vecs < 16384 else 0)   # one short of whole vectors: ragged rows
    rng = np.random.default_rng(rows + cols)
    x = (rng.standard_normal(rows * cols) * 2).astype(np.float32)
    x = x if dtype == D.F32 else orc.narrow(x, ORC[dtype])
    got = rows_op(dev, stream, op, x, rows, cols, dtype)
    check(op, got, x if dtype == D.F32 else orc.widen(x, ORC[dtype]), rows, cols, dtype)


@pytest.mark.parametrize("op", ["softmax", "rms_norm"])
@pytest.mark.parametrize("dtype", [D.F32, D.BF16])
@pytest.mark.parametrize("x_off", [1, 3])
@pytest.mark.parametrize("in_place", [False, True])
def test_rows_wide_offset_and_in_place(dev, stream, op, dtype, x_off, in_place):
    rows, cols = 37, 5003
    rng = np.random.default_rng(x_off)
    x = (rng.standard_normal(rows * cols) * 2).astype(np.float32)
    x = x if dtype == D.F32 else orc.narrow(x, ORC[dtype])
    got = rows_op(dev, stream, op, x, rows, cols, dtype, x_off, in_place)
    check(op, got, x if dtype == D.F32 else orc.widen(x, ORC[dtype]), rows, cols, dtype)


@pytest.mark.parametrize("dtype", [D.F32, D.F16])
def test_softmax_rows_wide_masks(dev, stream, dtype):
    """Rows of -inf next to finite ones: threads, waves and whole rows without a finite value;
    a row of -inf gives NaN, an infinite or NaN score a row of NaN where the sum is NaN; the
    type's lowest value masks as any other finite score does."""
    cols = 9001
    rng = np.random.default_rng(4)
    x = rng.standard_normal((6, cols)).astype(np.float32)
    x[0, :8000] = -np.inf
    x[1, 5:] = -np.inf
    x[2] = -np.inf
    x[3, 17] = np.inf
    x[4, 8999] = np.nan
    x[5, ::2] = np.finfo(np.float32 if dtype == D.F32 else np.float16).min
    xd = x if dtype == D.F32 else orc.narrow(x.ravel(), ORC[dtype])
    got = rows_op(dev, stream, "softmax", xd, 6, cols, dtype)
    got = (got if dtype == D.F32 else orc.widen(got, ORC[dtype])).reshape(6, cols)
    ok = [0, 1, 5]
    xw = x if dtype == D.F32 else orc.widen(xd, ORC[dtype]).reshape(6, cols)
    ref = orc.softmax(np.ascontiguousarray(xw[ok]), 3, cols)
    if dtype == D.F32:
        assert_softmax_close(got[ok], ref)
    else:
        assert_within_ulp16(got[ok], ref, ORC[dtype])
    assert np.isnan(got[2]).all() and np.isnan(got[4]).all() and np.isnan(got[3, 17])
