"""The calls that this library's speed is judged by: its tile ops (rows, matrix products,
attention) through the public Python entry points, on tensors that already lie in GPU memory.

A case is a dict of plain values.  `op` names the entry point, the other entries are its
sizes, types and options:

  softmax, rms_norm   rows, cols, dtype
  matmul, swiglu      m, k, n, dtype (A, B), out (C, UP), trans (B stored N x K)
  prefill, decode     batch, seq (queries, or cached positions), start (prefill: cached
                      positions before the queries), heads, kv_heads, head_dim, dtype
"""
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tile-rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tilers_hip as th  # noqa: E402

DTYPES = {"f32": (torch.float32, th.TileDtype.F32), "f16": (torch.float16, th.TileDtype.F16),
          "bf16": (torch.bfloat16, th.TileDtype.BF16)}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
EPS = 1e-6


def listed():
    return [
        # the norm of a decode step's few tokens in a wide model: the smallest call
        dict(name="rms_norm step", op="rms_norm", rows=8, cols=16384, dtype="bf16"),
        # probabilities over a vocabulary whose rows are not 16-byte aligned
        dict(name="softmax vocabulary", op="softmax", rows=256, cols=50257, dtype="f32"),
        # the square product of the benchmark
        dict(name="matmul square", op="matmul", m=4096, k=4096, n=4096, dtype="bf16", out="f32",
             trans=False),
        # the MLP's down projection in a decode step of eight sequences
        dict(name="matmul step", op="matmul", m=8, k=14336, n=4096, dtype="bf16", out="bf16",
             trans=True),
        # an f32 product of ordinary size with ragged edges
        dict(name="matmul f32", op="matmul", m=999, k=4096, n=1000, dtype="f32", out="f32",
             trans=False),
        # the MLP's gate over a prompt of any length, activation fused
        dict(name="swiglu prompt", op="swiglu", m=3000, k=4096, n=14336, dtype="f16", out="f16",
             trans=False),
        # a batch of whole prompts: the largest call
        dict(name="prefill batch", op="prefill", batch=4, seq=4096, start=0, heads=32,
             kv_heads=32, head_dim=128, dtype="bf16"),
        # one chunk of a long prompt after what is cached already
        dict(name="prefill chunk", op="prefill", batch=1, seq=512, start=7680, heads=32,
             kv_heads=8, head_dim=128, dtype="bf16"),
        # the tile op's own type, a prompt of odd length
        dict(name="prefill f32", op="prefill", batch=1, seq=1001, start=0, heads=32, kv_heads=8,
             head_dim=128, dtype="f32"),
        # a decode step of many sequences
        dict(name="decode batch", op="decode", batch=64, seq=8192, heads=32, kv_heads=8,
             head_dim=128, dtype="bf16"),
        # a decode step of one long sequence
        dict(name="decode long", op="decode", batch=1, seq=32001, heads=32, kv_heads=8,
             head_dim=128, dtype="bf16"),
        # the tile op's own type, a few sequences
        dict(name="decode f32", op="decode", batch=8, seq=3000, heads=32, kv_heads=8,
             head_dim=128, dtype="f32"),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    op = rng.choice(["softmax", "rms_norm", "matmul", "matmul", "matmul f32", "swiglu", "prefill",
                     "prefill", "decode", "decode"])
    if op in ("softmax", "rms_norm"):
        dtype = rng.choice(["f32", "bf16", "f16"])
        cols = _log(rng, 128, 152064) if op == "softmax" else _log(rng, 512, 16384)
        if rng.random() < 0.6:   # most widths are whole vectors
            cols = max(64, cols // 64 * 64)
        return dict(op=op, rows=_log(rng, 1, min(16384, (1 << 26) // cols)), cols=cols,
                    dtype=dtype)
    if op == "matmul f32":
        size = lambda: _log(rng, 64, 4096)  # noqa: E731
        return dict(op="matmul", m=size(), k=size(), n=size(), dtype="f32", out="f32",
                    trans=rng.random() < 0.5)
    if op in ("matmul", "swiglu"):
        dtype = rng.choice(["bf16", "f16"])
        if rng.random() < 0.7:   # a model's projections
            k, n = rng.choice([(4096, 14336), (4096, 4096), (4096, 1024), (2048, 1024)]
                              + ([(14336, 4096)] if op == "matmul" else []))
        else:
            k, n = 8 * _log(rng, 32, 1024), 8 * _log(rng, 32, 1024)
        out = dtype if op == "swiglu" or rng.random() < 0.7 else "f32"
        return dict(op=op, m=_log(rng, 1, 4096), k=k, n=n, dtype=dtype, out=out,
                    trans=rng.random() < 0.5)
    heads, kv_heads = rng.choice([(32, 8), (32, 32), (16, 2), (8, 8)])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    head_dim = rng.choice([128, 128, 64])
    if op == "prefill":
        f32 = dtype == "f32"
        start = rng.choice([0, 0, _log(rng, 16, 1024 if f32 else 8192)])
        return dict(op=op, batch=1 if f32 else _log(rng, 1, 4),
                    seq=_log(rng, 16, 1024 if f32 else 4096 if start == 0 else 1024), start=start,
                    heads=heads, kv_heads=kv_heads, head_dim=head_dim, dtype=dtype)
    batch = _log(rng, 1, 64)
    most = (1 << 29) // (batch * kv_heads * head_dim * SIZE[dtype])   # 1 GiB of K and V
    return dict(op=op, batch=batch, seq=_log(rng, 64, max(64, min(32768, most))), heads=heads,
                kv_heads=kv_heads, head_dim=head_dim, dtype=dtype)


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, dtype=case["dtype"], std=1.0):
        x = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=g)
        return x.to(DTYPES[dtype][0])

    op = case["op"]
    if op in ("softmax", "rms_norm"):
        return dict(x=normal(case["rows"], case["cols"], std=2.0 if op == "softmax" else 1.0))
    if op in ("matmul", "swiglu"):
        m, k, n = case["m"], case["k"], case["n"]
        s = dict(a=normal(m, k), b=normal(*((n, k) if case["trans"] else (k, n)), std=0.02))
        if op == "swiglu":
            s["up"] = normal(m, n, dtype=case["out"])
        return s
    b, h, hk, d = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    if op == "prefill":
        rows = case["start"] + case["seq"]
        q = normal(b, case["seq"], h, d)
    else:
        rows = case["seq"]
        q = normal(b, h, d)
    return dict(q=q, k=normal(b, hk, rows, d), v=normal(b, hk, rows, d))


def prepare(case, seed):
    s = _inputs(case, seed)
    op = case["op"]
    if op in ("softmax", "rms_norm"):
        s["y"] = torch.empty_like(s["x"])
    elif op in ("matmul", "swiglu"):
        s["c"] = torch.empty(case["m"], case["n"], dtype=DTYPES[case["out"]][0], device="cuda")
    else:
        s["o"] = torch.empty_like(s["q"])
        if op == "decode":
            size = th.attention_decode_workspace_size(case["batch"], case["seq"],
                                                      case["head_dim"], case["heads"],
                                                      case["kv_heads"])
            s["ws"] = torch.empty(max(size, 16), dtype=torch.uint8, device="cuda")
            s["ws_size"] = size
    s["case"] = case
    return s


def run(s):
    c = s["case"]
    op, dt = c["op"], DTYPES[c["dtype"]][1]
    if op == "softmax":
        th.softmax(s["x"].data_ptr(), s["y"].data_ptr(), c["rows"], c["cols"], dt)
        return s["y"]
    if op == "rms_norm":
        th.rms_norm(s["x"].data_ptr(), s["y"].data_ptr(), c["rows"], c["cols"], EPS, dt)
        return s["y"]
    if op == "matmul":
        th.matmul(s["a"].data_ptr(), s["b"].data_ptr(), s["c"].data_ptr(), c["m"], c["k"], c["n"],
                  dt, DTYPES[c["out"]][1], c["trans"])
        return s["c"]
    if op == "swiglu":
        th.matmul_silu_mul(s["a"].data_ptr(), s["b"].data_ptr(), s["up"].data_ptr(),
                           s["c"].data_ptr(), c["m"], c["k"], c["n"], dt, DTYPES[c["out"]][1],
                           c["trans"])
        return s["c"]
    if op == "prefill":
        th.attention_prefill(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                             s["o"].data_ptr(), c["batch"], c["seq"], c["start"],
                             c["start"] + c["seq"], c["head_dim"], c["heads"], c["kv_heads"], dt)
        return s["o"]
    th.attention_decode(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                        s["o"].data_ptr(), c["batch"], c["seq"], c["seq"], c["head_dim"],
                        c["heads"], c["kv_heads"], dt, s["ws"].data_ptr(), s["ws_size"])
    return s["o"]


def work(case):
    op = case["op"]
    if op in ("softmax", "rms_norm"):
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * SIZE[case["dtype"]], "flops": 4 * n}
    if op in ("matmul", "swiglu"):
        m, k, n = case["m"], case["k"], case["n"]
        outs = 2 if op == "swiglu" else 1
        return {"bytes": (m * k + k * n) * SIZE[case["dtype"]] + outs * m * n * SIZE[case["out"]],
                "flops": 2 * m * k * n}
    b, h, hk, d = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    if op == "prefill":
        s, rows = case["seq"], case["start"] + case["seq"]
        pairs = s * case["start"] + s * (s + 1) // 2
    else:
        s, rows, pairs = 1, case["seq"], case["seq"]
    return {"bytes": (2 * b * s * h * d + 2 * b * hk * rows * d) * SIZE[case["dtype"]],
            "flops": 4 * b * h * pairs * d}


def tolerance(case):
    # four times the distance from 64 bits: f32 sums; one rounding of the result in f16 or
    # bf16; and in 16-bit attention the rounding of the probabilities as well
    out = case.get("out", case["dtype"])
    if out == "f32":
        return {"rel": 1e-5}
    return {"rel": 1e-3 if out == "f16" else 8e-3}


def exact(case, seed):
    s = {k: v.double() for k, v in _inputs(case, seed).items()}
    op = case["op"]
    if op == "softmax":
        return torch.softmax(s["x"], dim=-1)
    if op == "rms_norm":
        return s["x"] * torch.rsqrt(s["x"].square().mean(dim=-1, keepdim=True) + EPS)
    if op in ("matmul", "swiglu"):
        c = s["a"] @ (s["b"].t().contiguous() if case["trans"] else s["b"])
        return torch.nn.functional.silu(c) * s["up"] if op == "swiglu" else c
    q = s["q"].unsqueeze(1) if op == "decode" else s["q"]
    o = torch.empty_like(q)
    rows, queries = s["k"].shape[2], q.shape[1]
    hidden = torch.ones(queries, rows, dtype=torch.bool, device="cuda").triu(rows - queries + 1)
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            g = h // (case["heads"] // case["kv_heads"])
            score = q[b, :, h].contiguous() @ s["k"][b, g].t().contiguous()
            score = (score * case["head_dim"] ** -0.5).masked_fill_(hidden, float("-inf"))
            o[b, :, h] = torch.softmax(score, dim=-1) @ s["v"][b, g]
    return o[:, 0] if op == "decode" else o
