"""The work that users of this backend have it do, as measurable cases.

Every case is a Triton program launched as `kernel[grid](...)` with the backend active, over the range of sizes, types and
layouts such programs meet: the kernels of `triton_shared_amd.examples.kernels`, and two programs that are as common (a
flash-attention forward, and the weight and bias gradients of LayerNorm), written here against the same frontend.

`listed()` names one case per kind of work, `draw(rng)` takes more of the same kinds over their whole ranges.
"""
import math

import numpy as np
import torch

import triton_shared_amd as tsa
from triton_shared_amd.examples import kernels as K

triton, tl = K.triton, K.tl
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
ITEM = {"fp32": 4, "fp16": 2, "bf16": 2}


# ---- two programs of the tutorials that the package's examples do not hold -------------------------------------------
@triton.jit
def attention_fwd(Q, K, V, O, sm_scale, seq, stride_h, stride_s, BM: tl.constexpr, BN: tl.constexpr, D: tl.constexpr,
                  CAUSAL: tl.constexpr):
    """Flash-attention forward: one (query block, head) per program, an online softmax over blocks of keys."""
    pm = tl.program_id(0)
    ph = tl.program_id(1)
    rm = pm * BM + tl.arange(0, BM)
    rd = tl.arange(0, D)
    q = tl.load(Q + ph * stride_h + rm[:, None] * stride_s + rd[None, :], mask=rm[:, None] < seq, other=0.0)
    m_i = tl.zeros([BM], dtype=tl.float32) - float("inf")
    l_i = tl.zeros([BM], dtype=tl.float32)
    acc = tl.zeros([BM, D], dtype=tl.float32)
    last = seq
    if CAUSAL:
        last = tl.minimum(seq, (pm + 1) * BM)
    for start in range(0, last, BN):
        rn = start + tl.arange(0, BN)
        k = tl.load(K + ph * stride_h + rn[:, None] * stride_s + rd[None, :], mask=rn[:, None] < seq, other=0.0)
        v = tl.load(V + ph * stride_h + rn[:, None] * stride_s + rd[None, :], mask=rn[:, None] < seq, other=0.0)
        qk = tl.dot(q, tl.trans(k)) * sm_scale
        if CAUSAL:
            qk = tl.where((rn[None, :] < seq) & (rm[:, None] >= rn[None, :]), qk, -float("inf"))
        else:
            qk = tl.where(rn[None, :] < seq, qk, -float("inf"))
        m_new = tl.maximum(m_i, tl.max(qk, axis=1))
        p = tl.exp(qk - m_new[:, None])
        alpha = tl.exp(m_i - m_new)
        l_i = l_i * alpha + tl.sum(p, axis=1)
        acc = acc * alpha[:, None] + tl.dot(p.to(V.dtype.element_ty), v)
        m_i = m_new
    acc = acc / l_i[:, None]
    tl.store(O + ph * stride_h + rm[:, None] * stride_s + rd[None, :], acc.to(O.dtype.element_ty), mask=rm[:, None] < seq)


@triton.jit
def layer_norm_dwdb(dy_ptr, x_ptr, mean_ptr, rstd_ptr, dw_ptr, db_ptr, n_rows, n_cols, pitch, BR: tl.constexpr, BC: tl.constexpr):
    """The weight and bias gradients of LayerNorm: one block of columns per program, walked down the rows."""
    c = tl.program_id(0) * BC + tl.arange(0, BC)
    dw = tl.zeros((BR, BC), dtype=tl.float32)
    db = tl.zeros((BR, BC), dtype=tl.float32)
    for r0 in range(0, n_rows, BR):
        r = r0 + tl.arange(0, BR)
        m = (r[:, None] < n_rows) & (c[None, :] < n_cols)
        x = tl.load(x_ptr + r[:, None] * pitch + c[None, :], mask=m, other=0.0).to(tl.float32)
        dy = tl.load(dy_ptr + r[:, None] * pitch + c[None, :], mask=m, other=0.0).to(tl.float32)
        mean = tl.load(mean_ptr + r, mask=r < n_rows, other=0.0)
        rstd = tl.load(rstd_ptr + r, mask=r < n_rows, other=0.0)
        dw += dy * ((x - mean[:, None]) * rstd[:, None])
        db += dy
    tl.store(dw_ptr + c, tl.sum(dw, axis=0), mask=c < n_cols)
    tl.store(db_ptr + c, tl.sum(db, axis=0), mask=c < n_cols)


# ---- the cases ---------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call a program makes: the vector-add configuration at its literal size, where the launch is the cost
        {"name": "add_small", "kind": "add", "n": 98432},
        # attention scores or router logits of an odd width, one row per program
        {"name": "softmax_odd_rows", "kind": "softmax", "rows": 4096, "cols": 781, "dtype": "fp32"},
        # a normalisation layer in training: forward, input gradient, weight and bias gradients
        {"name": "layer_norm_train", "kind": "layer_norm", "rows": 4096, "cols": 8192, "dtype": "fp16"},
        # the large dense product of a training or prefill step
        {"name": "matmul_large", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096, "dtype": "bf16", "form": "tiles"},
        # the stock tutorial product (wrapped operands, fused activation) at sizes nothing divides
        {"name": "matmul_ragged_act", "kind": "matmul", "m": 1000, "n": 3001, "k": 1003, "dtype": "fp16", "form": "wrapped_act"},
        # the fp32 product of the reference's own benchmark, its largest size and its block sizes
        {"name": "matmul_fp32", "kind": "matmul", "m": 768, "n": 768, "k": 768, "dtype": "fp32", "form": "tiles"},
        # a projection of a batch of decoded tokens: far fewer rows than columns
        {"name": "matmul_skinny", "kind": "matmul", "m": 128, "n": 4096, "k": 4096, "dtype": "bf16", "form": "tiles"},
        # int8 weights in decode: 16 tokens against a feed-forward weight
        {"name": "w8a16_decode", "kind": "w8a16", "m": 16, "n": 28672, "k": 8192},
        # int8 weights in prefill or a big decode batch, a number of rows nothing divides
        {"name": "w8a16_prefill", "kind": "w8a16", "m": 300, "n": 28672, "k": 8192},
        # a mixture-of-experts layer: 2048 tokens, two of eight experts each, rows gathered and grouped by expert
        {"name": "experts", "kind": "experts", "tokens": 2048, "top": 2, "experts": 8, "k": 2048, "n": 2048},
        # causal self-attention over a whole prompt
        {"name": "attention_prefill", "kind": "attention", "heads": 32, "seq": 4096, "d": 128, "dtype": "bf16", "causal": True},
        # what stands between the products of a decoder layer: embedding rows, RMSNorm, rotary embedding, gated activation
        {"name": "decoder_rows", "kind": "rows", "tokens": 4000, "hidden": 4096, "inner": 14336, "half": 64, "vocab": 32000},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["add", "softmax", "layer_norm", "matmul", "matmul", "matmul", "w8a16", "w8a16", "experts", "attention", "attention", "rows"])
    if kind == "add":
        return {"kind": kind, "n": _log(rng, 1000, 1 << 27)}
    if kind == "softmax":
        cols = _log(rng, 50, 20000)
        return {"kind": kind, "rows": _log(rng, 64, min(65536, (1 << 27) // cols)), "cols": cols, "dtype": rng.choice(["fp32", "fp16", "bf16"])}
    if kind == "layer_norm":
        cols = rng.choice([_log(rng, 256, 8192), 256 * rng.randint(1, 32)])
        return {"kind": kind, "rows": _log(rng, 128, 8192), "cols": cols, "dtype": rng.choice(["fp16", "bf16", "fp32"])}
    if kind == "matmul":
        form = rng.choice(["tiles", "wrapped", "wrapped_act", "b_columns"])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        step = rng.choice([1, 8, 64, 64])  # nothing divides the size, 16-byte rows, whole tiles
        top = 1024 if dtype == "fp32" else 4096
        m, n, k = (max(step, _log(rng, low, top) // step * step) for low in (16, 128, 128))
        return {"kind": kind, "m": m, "n": n, "k": k, "dtype": dtype, "form": form}
    if kind == "w8a16":
        return {"kind": kind, "m": _log(rng, 1, 1024), "n": 128 * rng.randint(16, 224), "k": 128 * rng.randint(8, 64)}
    if kind == "experts":
        return {"kind": kind, "tokens": _log(rng, 64, 4096), "top": rng.choice([1, 2]), "experts": rng.choice([4, 8, 16]),
                "k": 64 * rng.randint(8, 40), "n": 64 * rng.randint(8, 40)}
    if kind == "attention":
        seq = _log(rng, 200, 4096)
        return {"kind": kind, "heads": rng.randint(1, 32), "seq": seq, "d": rng.choice([64, 128]), "dtype": rng.choice(["fp16", "bf16"]),
                "causal": rng.random() < 0.5 or seq > 2900}
    half = rng.choice([32, 64])
    return {"kind": "rows", "tokens": _log(rng, 1, 8192), "hidden": 2 * half * rng.randint(8, 4096 // half), "inner": 256 * rng.randint(8, 56),
            "half": half, "vocab": 32000}


def _slots(case):
    """Row slots of a mixture-of-experts product: every (token, expert) pair, each expert's rows filled up to whole blocks of 128."""
    return (case["tokens"] * case["top"] + 127) // 128 * 128 + case["experts"] * 128


def work(case):
    """Bytes and operations that one pass cannot do without: every input read once, every output written once."""
    kind = case["kind"]
    if kind == "add":
        return {"bytes": 12 * case["n"], "flops": case["n"]}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * ITEM[case["dtype"]], "flops": 5 * n}
    if kind == "layer_norm":
        rows, cols, item = case["rows"], case["cols"], ITEM[case["dtype"]]
        # x and dy read, y and dx written; weights and bias read, their gradients and the row statistics written
        return {"bytes": 4 * rows * cols * item + 2 * cols * item + 2 * cols * 4 + 2 * rows * 4, "flops": 24 * rows * cols}
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + k * n + m * n) * ITEM[case["dtype"]], "flops": 2 * m * n * k}
    if kind == "w8a16":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": k * n + 2 * m * k + 2 * n + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "experts":
        pairs, k, n = case["tokens"] * case["top"], case["k"], case["n"]
        return {"bytes": 2 * (case["tokens"] * k + case["experts"] * k * n + pairs * n), "flops": 2 * pairs * n * k}
    if kind == "attention":
        h, s, d = case["heads"], case["seq"], case["d"]
        return {"bytes": 4 * 2 * h * s * d, "flops": 4 * h * d * (s * (s + 1) // 2 if case["causal"] else s * s)}
    t, hidden, inner, half = case["tokens"], case["hidden"], case["inner"], case["half"]
    # the rows of the table that are named, the normalised rows, the rotated rows and the gated activation; the row that
    # goes from the gather to the normalisation is an output too (the residual stream), as is the normalised row
    return {"bytes": 2 * (4 * t * hidden + 3 * t * inner + hidden) + 8 * t * half + 4 * t, "flops": 20 * t * (hidden + inner)}


def tolerance(case):
    """Largest relative error another correct implementation at the same precision shows; see each line."""
    kind = case["kind"]
    if kind == "add":
        return "exact"  # one IEEE addition per element
    if kind == "softmax":
        # fp32: exponentials and sums of an ulp or two; 16-bit: results that round to the other neighbour
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "fp32" else {"rel": _ulp(case["dtype"]) / 2, "max": 2 * _ulp(case["dtype"])}
    if kind == "layer_norm":
        # fp32 sums in another order (means near zero are sums that cancel); 16-bit results that round to the other neighbour
        return {"rel": 1e-5, "max": 4e-4} if case["dtype"] == "fp32" else {"rel": _ulp(case["dtype"]) / 2, "max": 2 * _ulp(case["dtype"])}
    if kind == "matmul":
        # fp32 sums over K in another order; 16-bit results round once
        return {"rel": 4e-6, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": _ulp(case["dtype"]) / 2, "max": 2 * _ulp(case["dtype"])}
    if kind == "w8a16":
        return {"rel": 1e-3, "max": 8e-3}  # fp16 weights after the scale, fp16 results
    if kind == "experts":
        return {"rel": _ulp("bf16") / 2, "max": 2 * _ulp("bf16")}
    if kind == "attention":
        # probabilities are narrowed relative to a running maximum, whose history depends on the order of the key blocks
        return {"rel": _ulp(case["dtype"]), "max": 20 * _ulp(case["dtype"])}
    return {"rel": 1e-3, "max": 2 * _ulp("fp16")}


def _ulp(dtype):
    return 2.0 ** -10 if dtype == "fp16" else 2.0 ** -7


def _pow2(n):
    return 1 << max(0, n - 1).bit_length()


def prepare(case, seed):
    """Inputs, weights and result buffers, as a program that calls these kernels in a loop holds them."""
    tsa.activate()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, scale=1.0, mean=0.0, dtype=torch.float32):
        t = torch.empty(*shape, dtype=torch.float32, device="cuda")
        t.normal_(mean, scale, generator=g)
        return t.to(dtype)

    def out(*shape, dtype=torch.float32):
        return torch.zeros(*shape, dtype=dtype, device="cuda")

    kind, s = case["kind"], dict(case)
    if kind == "add":
        s.update(x=normal(case["n"]), y=normal(case["n"]), z=out(case["n"]))
    elif kind == "softmax":
        dt = DTYPES[case["dtype"]]
        s.update(x=normal(case["rows"], case["cols"], scale=3.0, dtype=dt), o=out(case["rows"], case["cols"], dtype=dt), block=max(16, _pow2(case["cols"])))
    elif kind == "layer_norm":
        rows, cols, dt = case["rows"], case["cols"], DTYPES[case["dtype"]]
        s.update(x=normal(rows, cols, mean=0.3, dtype=dt), dy=normal(rows, cols, mean=0.1, dtype=dt), w=normal(cols, scale=0.1, mean=1.0, dtype=dt), b=normal(cols, scale=0.1, dtype=dt),
                 y=out(rows, cols, dtype=dt), dx=out(rows, cols, dtype=dt), mean=out(rows), rstd=out(rows), dw=out(cols), db=out(cols), block=_pow2(cols))
    elif kind == "matmul":
        m, n, k, dt = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
        # activations of unit variance against weights whose products keep it
        a, c = normal(m, k, dtype=dt), out(m, n, dtype=dt)
        b = normal(n, k, scale=k ** -0.5, dtype=dt).t() if case["form"] == "b_columns" else normal(k, n, scale=k ** -0.5, dtype=dt)
        s.update(a=a, b=b, c=c, blocks=(32, 64, 16) if case["dtype"] == "fp32" else (128, 128, 64))
    elif kind == "w8a16":
        m, n, k = case["m"], case["n"], case["k"]
        w = torch.randint(-127, 128, (k, n), generator=g, dtype=torch.int8, device="cuda")
        s.update(a=normal(m, k, dtype=torch.float16), w=w, scales=normal(n, scale=1e-4, mean=8e-4).clamp_(min=1e-4).half(), c=out(m, n, dtype=torch.float16), bm=min(64, max(16, _pow2(m))))
    elif kind == "experts":
        t, top, e, k, n = (case[x] for x in ("tokens", "top", "experts", "k", "n"))
        rng = np.random.RandomState(seed % (1 << 32))
        chosen = np.argsort(rng.rand(t, e) + 0.3 * rng.rand(1, e), axis=1)[:, :top]  # experts are not equally popular
        rows, ids = [], []
        for x in range(e):
            mine = np.nonzero((chosen == x).any(axis=1))[0]
            blocks = -(-len(mine) // 128)
            rows.append(np.concatenate([mine, np.zeros(blocks * 128 - len(mine), mine.dtype)]))
            ids += [x] * blocks
        slots = _slots(case)
        rows = np.concatenate(rows)
        rows = np.concatenate([rows, np.zeros(slots - len(rows), rows.dtype)]).astype(np.int32)
        ids = np.array(ids + [-1] * (slots // 128 - len(ids)), np.int32)  # blocks past the last expert's have nothing to do
        s.update(a=normal(t, k, dtype=torch.bfloat16), b=normal(e, k, n, scale=k ** -0.5, dtype=torch.bfloat16), c=out(slots, n, dtype=torch.bfloat16),
                 rows=torch.from_numpy(rows).cuda(), ids=torch.from_numpy(ids).cuda(), slots=slots)
    elif kind == "attention":
        shape, dt = (case["heads"], case["seq"], case["d"]), DTYPES[case["dtype"]]
        s.update(q=normal(*shape, dtype=dt), k=normal(*shape, dtype=dt), v=normal(*shape, dtype=dt), o=out(*shape, dtype=dt))
    else:
        t, hidden, inner, half, vocab = (case[x] for x in ("tokens", "hidden", "inner", "half", "vocab"))
        angle = torch.arange(t, device="cuda", dtype=torch.float32)[:, None] * 10000.0 ** (-torch.arange(half, device="cuda", dtype=torch.float32) / half)
        s.update(table=normal(vocab, hidden, dtype=torch.float16), tokens_in=torch.randint(0, vocab, (t,), generator=g, dtype=torch.int32, device="cuda"),
                 w=normal(hidden, scale=0.1, mean=1.0, dtype=torch.float16), cos=torch.cos(angle), sin=torch.sin(angle),
                 gate=normal(t, inner, dtype=torch.float16), up=normal(t, inner, dtype=torch.float16), x=out(t, hidden, dtype=torch.float16),
                 normed=out(t, hidden, dtype=torch.float16), rotated=out(t, hidden, dtype=torch.float16), act=out(t, inner, dtype=torch.float16), block=_pow2(hidden))
    return s


def run(s):
    kind = s["kind"]
    if kind == "add":
        K.vec_add[(triton.cdiv(s["n"], 1024),)](s["x"], s["y"], s["z"], s["n"], BLOCK=1024)
        return s["z"]
    if kind == "softmax":
        x, o = s["x"], s["o"]
        K.row_softmax[(s["rows"],)](o, x, x.stride(0), o.stride(0), s["cols"], BLOCK=s["block"])
        return o
    if kind == "layer_norm":
        rows, cols, x = s["rows"], s["cols"], s["x"]
        K.layer_norm_fwd[(rows,)](x, s["y"], s["w"], s["b"], s["mean"], s["rstd"], x.stride(0), cols, 1e-5, BLOCK=1024)
        K.layer_norm_dx_rows[(rows,)](s["dx"], s["dy"], x, s["w"], s["mean"], s["rstd"], x.stride(0), cols, BLOCK=s["block"])
        layer_norm_dwdb[(triton.cdiv(cols, 128),)](s["dy"], x, s["mean"], s["rstd"], s["dw"], s["db"], rows, cols, x.stride(0), BR=32, BC=128)
        return {"y": s["y"], "mean": s["mean"], "rstd": s["rstd"], "dx": s["dx"], "dw": s["dw"], "db": s["db"]}
    if kind == "matmul":
        a, b, c, (bm, bn, bk) = s["a"], s["b"], s["c"], s["blocks"]
        m, n, k = s["m"], s["n"], s["k"]
        grid = (triton.cdiv(m, bm) * triton.cdiv(n, bn),)
        strides = (a.stride(0), a.stride(1), b.stride(0), b.stride(1), c.stride(0), c.stride(1))
        if s["form"] in ("wrapped", "wrapped_act"):
            K.matmul_wrapped[grid](a, b, c, m, n, k, *strides, BM=bm, BN=bn, BK=bk, GROUP_M=8, ACTIVATION="leaky_relu" if s["form"] == "wrapped_act" else "")
        else:
            K.matmul_tiles[grid](a, b, c, m, n, k, *strides, BM=bm, BN=bn, BK=bk, GROUP_M=8)
        return c
    if kind == "w8a16":
        a, w, c, bm = s["a"], s["w"], s["c"], s["bm"]
        m, n, k = s["m"], s["n"], s["k"]
        K.w8a16_matmul[(triton.cdiv(m, bm), triton.cdiv(n, 128))](a, w, s["scales"], c, m, n, k, k, 1, n, 1, n, 1, BM=bm, BN=128, BK=128)
        return c
    if kind == "experts":
        k, n = s["k"], s["n"]
        K.expert_rows_matmul[(s["slots"] // 128, triton.cdiv(n, 128))](s["a"], s["b"], s["c"], s["rows"], s["ids"], s["slots"], k, n, k, k * n, n, n, BM=128, BN=128, BK=64)
        return s["c"]
    if kind == "attention":
        q, seq, d = s["q"], s["seq"], s["d"]
        bm = 128 if d == 64 else 64
        attention_fwd[(triton.cdiv(seq, bm), s["heads"])](q, s["k"], s["v"], s["o"], d ** -0.5, seq, q.stride(0), q.stride(1), BM=bm, BN=64, D=d, CAUSAL=s["causal"])
        return s["o"]
    t, hidden, half = s["tokens"], s["hidden"], s["half"]
    x = s["x"]
    K.take_rows[(triton.cdiv(t, 4),)](s["table"], s["tokens_in"], x, t, hidden, hidden, hidden, BR=4, BC=s["block"])
    K.rms_norm_rows[(t,)](x, s["w"], s["normed"], hidden, hidden, 1e-6, BLOCK=s["block"])
    K.rotary_embedding[(t, hidden // (2 * half))](s["normed"], s["cos"], s["sin"], s["rotated"], hidden, HALF=half)
    n = t * s["inner"]
    K.silu_mul_f16[(triton.cdiv(n, 1024),)](s["gate"], s["up"], s["act"], n, BLOCK=1024)
    return {"x": x, "normed": s["normed"], "rotated": s["rotated"], "act": s["act"]}
