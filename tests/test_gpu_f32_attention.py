"""f32 causal GQA prefill and GQA decode on the fp32 matrix cores, against the oracle's sequential f32 loops.

The sums run in another order than the oracle's and the exponentials in base 2; outputs are
weighted means of V ~ N(0, 1), so the bound is 1e-5 absolute, that of the single-head f32
kernel (tests/test_gpu_ops.py, test_attention_f32_shapes)."""
import numpy as np
import pytest

import tilers_hip as th
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
D = th.TileDtype


def put(dev, stream, x, offset=0):
    b = dev.alloc(x.size + offset, D.F32)
    b.copy_from_host(np.concatenate([np.zeros(offset, np.float32), x.reshape(-1)]), stream)
    return b


def prefill(dev, stream, q, k, v, B, S, start, max_seq, Dh, NH, NKV, offset=0):
    bufs = [put(dev, stream, x, offset) for x in (q, k, v)]
    ob = put(dev, stream, np.full(q.size, 7.0, np.float32), offset)
    th.attention_prefill(*(b.as_raw_ptr() + 4 * offset for b in bufs + [ob]), B, S, start, max_seq,
                         Dh, NH, NKV, D.F32, stream)
    return ob.copy_to_host(stream)[offset:].reshape(q.shape)


def inputs(rng, B, S, max_seq, Dh, NH, NKV):
    return (rng.standard_normal((B, S, NH, Dh)).astype(np.float32),
            rng.standard_normal((B, NKV, max_seq, Dh)).astype(np.float32),
            rng.standard_normal((B, NKV, max_seq, Dh)).astype(np.float32))


@pytest.mark.parametrize("Dh", [64, 128])
@pytest.mark.parametrize("B,S,start,extra,NH,NKV", [
    (1, 1, 0, 0, 2, 2),        # one query, one position
    (3, 1, 5, 2, 4, 4),        # one query after a few cached positions
    (1, 31, 0, 0, 4, 2),       # less than one 32-query group
    (1, 33, 31, 1, 4, 1),      # a second group of one query; diagonal off the block edges
    (2, 64, 0, 0, 8, 2),       # one whole query block and stage
    (1, 65, 64, 0, 4, 4),      # one query over, start on a stage edge
    (2, 300, 37, 3, 8, 8),     # 16 (batch, kv head) units on 8 XCDs: grouped work order
    (1, 257, 1000, 60, 4, 1),  # a chunk after cached positions, rows past it not read
    (1, 601, 0, 0, 29, 29),    # 290 items: a short second round, not a multiple of 8
    (4, 130, 0, 0, 56, 14),    # 672 items: a third round
])
def test_prefill_f32_shapes(dev, stream, Dh, B, S, start, extra, NH, NKV):
    rng = np.random.default_rng(S * 7 + start + Dh)
    max_seq = start + S + extra
    q, k, v = inputs(rng, B, S, max_seq, Dh, NH, NKV)
    if extra:
        k[:, :, start + S:] = v[:, :, start + S:] = np.nan   # never written by a program
    got = prefill(dev, stream, q, k, v, B, S, start, max_seq, Dh, NH, NKV)
    ref = orc.attention_prefill(q, k, v, orc.F32, B, S, start, max_seq, Dh, NH, NKV)
    err = np.abs(got - ref.reshape(q.shape)).max()
    assert err < 1e-5, f"max err {err:.3e}"


def test_prefill_f32_unaligned_views(dev, stream):
    """Views 4 bytes off 16-byte alignment stay on the general kernel."""
    rng = np.random.default_rng(11)
    q, k, v = inputs(rng, 1, 70, 90, 64, 4, 2)
    got = prefill(dev, stream, q, k, v, 1, 70, 20, 90, 64, 4, 2, offset=1)
    ref = orc.attention_prefill(q, k, v, orc.F32, 1, 70, 20, 90, 64, 4, 2)
    assert np.abs(got - ref.reshape(q.shape)).max() < 1e-5


@pytest.mark.parametrize("Dh", [64, 128])
@pytest.mark.parametrize("pos", [0, 40, 69, 99])
def test_prefill_f32_later_positions_do_not_reach_a_query(dev, stream, Dh, pos):
    """NaN and infinities at position `pos` of K and V: queries before it are those of the
    finite inputs bit for bit, whatever stage and block `pos` shares with them; a query that
    sees an infinite V value has it in that column."""
    rng = np.random.default_rng(pos + Dh)
    q, k, v = inputs(rng, 1, 100, 100, Dh, 2, 1)
    clean = prefill(dev, stream, q, k, v, 1, 100, 0, 100, Dh, 2, 1)
    for kind in ("k nan", "v nan", "v inf"):
        kb, vb = k.copy(), v.copy()
        if kind == "k nan":
            kb[:, :, pos, 3] = np.nan
        else:
            vb[:, :, pos, 5] = np.nan if kind == "v nan" else np.inf
        got = prefill(dev, stream, q, kb, vb, 1, 100, 0, 100, Dh, 2, 1)
        assert np.array_equal(got[:, :pos], clean[:, :pos]), kind
        if kind != "k nan":
            seen = got[:, pos:, :, 5]
            assert (np.isnan(seen) if kind == "v nan" else seen == np.inf).all(), kind
            rest = np.delete(got[:, pos:], 5, axis=3)
            assert np.array_equal(rest, np.delete(clean[:, pos:], 5, axis=3)), kind


@pytest.mark.parametrize("B,L,extra,NH,NKV,Dh,ws", [
    (1, 1, 0, 4, 4, 128, "none"),       # one position
    (3, 513, 7, 16, 1, 128, "full"),    # G = 16, chunk boundary + 1, rows past L not read
    (2, 1024, 0, 8, 8, 128, "none"),    # G = 1, whole chunks
    (1, 9000, 40, 8, 1, 64, "full"),    # G = 8, head_dim 64, 18 splits
    (2, 4500, 0, 4, 2, 128, "part"),    # a workspace that holds fewer records than the plan
    (2, 4500, 0, 4, 2, 128, "tiny"),    # one too small for any split
    (64, 700, 0, 32, 8, 64, "none"),    # 512 items: unsplit
    (1, 200, 0, 6, 2, 128, "none"),     # G = 3: the general kernel
])
def test_decode_f32_shapes(dev, stream, B, L, extra, NH, NKV, Dh, ws):
    rng = np.random.default_rng(L * 3 + NH)
    max_seq = L + extra
    q = rng.standard_normal((B, NH, Dh)).astype(np.float32)
    k, v = (rng.standard_normal((B, NKV, max_seq, Dh)).astype(np.float32) for _ in range(2))
    k[:, :, L:] = v[:, :, L:] = np.nan
    bufs = [put(dev, stream, x) for x in (q, k, v)]
    ob = put(dev, stream, np.full(q.size, 7.0, np.float32))
    rec = B * NH * (Dh + 2) * 4
    size = {"none": 0, "full": th.attention_decode_workspace_size(B, L, Dh, NH, NKV),
            "part": 5 * rec, "tiny": rec + 8}[ws]
    # a guard after the workspace shows a write past it
    wb = put(dev, stream, np.full(size // 4 + 1024, 3.0, np.float32)) if size else None
    th.attention_decode(*bufs, ob, B, L, max_seq, Dh, NH, NKV, D.F32, wb, size, stream)
    got = ob.copy_to_host(stream).reshape(q.shape)
    ref = orc.attention_decode(q, k, v, orc.F32, B, L, max_seq, Dh, NH, NKV)
    err = np.abs(got - ref.reshape(q.shape)).max()
    assert err < 1e-5, f"max err {err:.3e}"
    if wb is not None:
        assert (wb.copy_to_host(stream)[size // 4:] == 3.0).all()


@pytest.mark.parametrize("B,L,NH,NKV,Dh", [(1, 3000, 8, 2, 128), (2, 700, 4, 4, 64)])
def test_decode_static_f32(dev, stream, B, L, NH, NKV, Dh):
    """f32 without allocation: the general kernel, close to the split kernel's result."""
    rng = np.random.default_rng(L)
    q = rng.standard_normal((B, NH, Dh)).astype(np.float32)
    k, v = (rng.standard_normal((B, NKV, L, Dh)).astype(np.float32) for _ in range(2))
    bufs = [put(dev, stream, x) for x in (q, k, v)]
    out = [put(dev, stream, np.full(q.size, 7.0, np.float32)) for _ in range(2)]
    th.attention_decode(*bufs, out[0], B, L, L, Dh, NH, NKV, D.F32, None, 0, stream)
    th._lib.check(th.lib().th_attention_decode_static(
        *(b.as_raw_ptr() for b in bufs), out[1].as_raw_ptr(), B, L, L, Dh, NH, NKV, int(D.F32),
        stream.handle))
    got, static = (o.copy_to_host(stream).reshape(q.shape) for o in out)
    ref = orc.attention_decode(q, k, v, orc.F32, B, L, L, Dh, NH, NKV).reshape(q.shape)
    assert np.abs(got - ref).max() < 1e-5 and np.abs(static - ref).max() < 1e-5
