"""The work a user of this package has it do, as timed cases: the attention layers of the column, row and
ICL stages (inference and training), the query-time column and row stages and the whole cached-KV query.

listed() names the cases; draw(rng) gives another one of the same ranges; prepare / run / exact / work /
tolerance take a case. Inputs come from torch's device generator and the seed alone. exact() restates a
case in float64 torch, with none of the package's code.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tabiclv2-torchtpu-v5p-benchmark_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tabicl_mi355_attn as pk  # noqa: E402
import tabicl_mi355_icl as icl  # noqa: E402
import tabicl_mi355_query as query  # noqa: E402

H = 8                # heads of every stage
E, HD = 128, 16      # column / row stage: width, head dim
W, ID = 512, 64      # ICL stage: width, head dim
NI = 128             # inducing points of a column block
C = 4                # CLS tokens of a row
NCLS = 10            # classes of the decoder
SKIP = -100.0        # the column stage's skip value
LAYER_SCALE = HD ** -0.5
DT = {"bf16": torch.bfloat16, "fp32": torch.float32}


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed() -> list:
    return [
        # one block's attention of a cached query: a few test rows of a small table, 8 estimators (latency)
        {"name": "icl_query_small", "kind": "icl_query", "est": 8, "test": 40, "train": 700, "cap": 1024},
        # the same at the headline workload: 5,000 test rows over 45,000 cached train rows
        {"name": "icl_query_large", "kind": "icl_query", "est": 8, "test": 5000, "train": 45000, "cap": 45000},
        # dataset-wise attention of a training step: 8 tables, 1,024 test rows over 16,384 train rows
        {"name": "icl_train", "kind": "icl_train", "est": 8, "test": 1024, "train": 16384},
        # column stage at fit time, first attention: 128 inducing points over the 45,000 train rows of
        # 100 columns x 8 estimators, padded to 50,000
        {"name": "isab1_bf16", "kind": "isab1", "dtype": "bf16", "seqs": 800, "rows": 50000, "valid": 45000},
        # second attention of the same block: every row over the 128 inducing points
        {"name": "isab2_bf16", "kind": "isab2", "dtype": "bf16", "seqs": 800, "rows": 50000},
        # the first attention again in the fp32 of the default (no autocast) column stage, 1,024 rows
        {"name": "isab1_fp32", "kind": "isab1", "dtype": "fp32", "seqs": 400, "rows": 1024, "valid": 1024},
        # row stage self-attention with RoPE: 16,384 rows of 100 features + 4 CLS tokens
        {"name": "row_bf16", "kind": "row", "dtype": "bf16", "rows": 16384, "tokens": 104, "live": 104},
        # the same layer in the default fp32 for a narrow table: 21 features padded to 24
        {"name": "row_fp32_narrow", "kind": "row", "dtype": "fp32", "rows": 20000, "tokens": 28, "live": 25},
        # the same layer at 104 tokens in a training step (4,096 rows), forward and backward
        {"name": "row_train", "kind": "row_train", "rows": 4096, "tokens": 104},
        # second column attention in a training step (416 columns x 1,024 rows), forward and backward
        {"name": "column_train", "kind": "column_train", "seqs": 416, "queries": 1024, "keys": 128},
        # column embedder of the headline cached query, fp32 as the default knobs run it
        {"name": "column_stage", "kind": "column_stage", "dtype": "fp32", "est": 8, "test": 5000, "features": 100,
         "real": 100},
        # a whole cached query for a small table, as a service answers it (logits)
        {"name": "query_small", "kind": "query", "dtype": "fp32", "est": 8, "test": 60, "features": 24, "real": 21,
         "train": 700, "blocks": 12},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["icl_query", "icl_train", "isab1", "isab2", "row", "row_train", "column_train",
                       "column_stage", "row_stage", "query"])
    dtype = rng.choice(["bf16", "fp32"])
    if kind == "icl_query":
        est = rng.choice([1, 2, 4, 8])
        train = _log(rng, 64, 50000)
        test = _log(rng, 1, max(1, min(8192, 1800000000 // (est * train))))
        return {"kind": kind, "est": est, "test": test, "train": train, "cap": train + rng.choice([0, 0, train // 9])}
    if kind == "icl_train":
        est = rng.choice([1, 2, 4, 8])
        train = _log(rng, 64, 16384)
        return {"kind": kind, "est": est, "test": _log(rng, 32, max(32, min(4096, 134217728 // (est * train)))),
                "train": train}
    if kind in ("isab1", "isab2"):
        seqs = _log(rng, 4, 800)
        rows = _log(rng, 100, max(100, min(50000, (40000000 if dtype == "bf16" else 4000000) // seqs)))
        case = {"kind": kind, "dtype": dtype, "seqs": seqs, "rows": rows}
        if kind == "isab1":
            case["valid"] = rng.choice([rows, max(1, int(rows * rng.uniform(0.55, 1.0)))])
        return case
    if kind in ("row", "row_train"):
        tokens = rng.randint(8, 260)  # 4 CLS tokens + 4 to 256 features
        rows = _log(rng, 16, max(16, min(40000, (1700000 if kind == "row" else 420000) // tokens)))
        if kind == "row_train":
            return {"kind": kind, "rows": rows, "tokens": tokens}
        return {"kind": kind, "dtype": dtype, "rows": rows, "tokens": tokens,
                "live": rng.choice([tokens, max(5, tokens - rng.randint(1, 7))])}
    if kind == "column_train":
        queries, keys = rng.choice([(128, _log(rng, 100, 2000)), (_log(rng, 100, 2000), 128)])
        return {"kind": kind, "seqs": _log(rng, 8, max(8, min(416, 430000 // max(queries, keys)))), "queries": queries,
                "keys": keys}
    est = rng.choice([1, 4, 8])
    features = rng.randint(4, 120)
    real = max(3, features - rng.choice([0, 0, rng.randint(1, 7)]))
    if kind == "query":
        train = _log(rng, 100, 8000)
        return {"kind": kind, "dtype": dtype, "est": est, "test": _log(rng, 1, 400), "features": features,
                "real": real, "train": train, "blocks": 12}
    test = _log(rng, 16, max(16, min(5000, 4000000 // (est * (features + C)))))
    return {"kind": kind, "dtype": dtype, "est": est, "test": test, "features": features, "real": real}


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
class Rope:
    """The row stage's rotary embedding (upstream's RotaryEmbedding surface: halves form, base 100000)."""
    interleaved = False

    def __init__(self):
        self.freqs = 100000.0 ** (-torch.arange(0, HD, 2, dtype=torch.float32) / HD)

    def get_seq_pos(self, n, device=None, dtype=torch.float32):
        return torch.arange(n, device=device, dtype=dtype)


def _gen(seed: int):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(1000003 * (seed + 1))

    def randn(*shape, dtype=torch.float32, scale=1.0):
        if math.prod(shape) > 1 << 28:  # in the target dtype at once: no fp32 copy of a large tensor
            return torch.randn(*shape, generator=g, device=dev, dtype=dtype).mul_(scale)
        return (torch.randn(*shape, generator=g, device=dev) * scale).to(dtype)

    return dev, randn


def _linear(randn, o: int, i: int, dt):
    return randn(o, i, dtype=dt, scale=i ** -0.5), randn(o, dtype=dt, scale=0.02)


def _block(randn, width: int, dt):
    """One pre-norm encoder layer: LayerNorms in fp32, GEMM weights in dt, feed-forward factor 2."""
    def norm():
        return 1 + randn(width, scale=0.05), randn(width, scale=0.05)

    return icl.IclBlockWeights(*norm(), *_linear(randn, 3 * width, width, dt), *_linear(randn, width, width, dt), *norm(),
                               *_linear(randn, 2 * width, width, dt), *_linear(randn, width, 2 * width, dt))


def _column(case: dict, randn):
    """Test rows, column weights and the hidden states [B, columns, 128, E] that the caches project."""
    dt, B, HC = DT[case["dtype"]], case["est"], case["features"] + C
    weights = query.ColumnWeights(*_linear(randn, E, 3, dt), [_block(randn, E, dt) for _ in range(3)], reserve_cls=C)
    X = randn(B, case["test"], case["features"])
    hidden = [randn(B, HC, NI, E, dtype=dt) for _ in range(3)]
    real = torch.full((B,), case["real"], dtype=torch.int64, device=X.device)
    return X, real, weights, hidden


def _row(case: dict, randn):
    dt = DT[case["dtype"]]
    return query.RowWeights(randn(C, E, dtype=dt, scale=0.5), [_block(randn, E, dt) for _ in range(3)],
                            1 + randn(E, scale=0.05), randn(E, scale=0.05))


def _inputs(case: dict, seed: int) -> dict:
    dev, randn = _gen(seed)
    kind = case["kind"]
    if kind in ("icl_query", "icl_train"):
        n, tq, tk = case["est"], case["test"], case["train"]
        s = {"q": randn(n, H, tq, ID, dtype=torch.bfloat16, scale=2.0), "k": randn(n, H, tk, ID, dtype=torch.bfloat16),
             "v": randn(n, H, tk, ID, dtype=torch.bfloat16)}
        if kind == "icl_train":
            s["do"] = randn(n, H, tq, ID, dtype=torch.bfloat16)
        return s
    if kind == "isab1":
        dt = DT[case["dtype"]]
        return {"q": randn(case["seqs"], NI, E, dtype=dt, scale=LAYER_SCALE),  # hxq takes pre-scaled queries
                "kv": randn(case["seqs"], case["rows"], 2 * E, dtype=dt),
                "valid": torch.tensor([case["valid"]], dtype=torch.int32, device=dev)}
    if kind == "isab2":
        dt = DT[case["dtype"]]
        return {"q": randn(case["seqs"], case["rows"], E, dtype=dt), "kv": randn(case["seqs"], NI, 2 * E, dtype=dt)}
    if kind == "row":
        kb = torch.zeros(1, case["tokens"], device=dev)
        kb[:, case["live"]:] = torch.finfo(torch.float32).min  # the padded feature slots' key mask
        return {"qkv": randn(case["rows"], case["tokens"], 3 * E, dtype=DT[case["dtype"]]),
                "kb": kb if case["live"] < case["tokens"] else None, "rope": Rope()}
    if kind == "row_train":
        return {"qkv": randn(case["rows"], case["tokens"], 3 * E, dtype=torch.bfloat16),
                "do": randn(case["rows"], case["tokens"], E, dtype=torch.bfloat16), "rope": Rope()}
    if kind == "column_train":
        B, lq, lk = case["seqs"], case["queries"], case["keys"]
        return {"q": randn(B, lq, E, dtype=torch.bfloat16, scale=LAYER_SCALE),
                "k": randn(B, lk, E, dtype=torch.bfloat16), "v": randn(B, lk, E, dtype=torch.bfloat16),
                "do": randn(B, lq, E, dtype=torch.bfloat16)}
    if kind == "row_stage":
        return {"src": randn(case["est"], case["features"] + C, case["test"], E, dtype=DT[case["dtype"]]),
                "real": torch.full((case["est"],), case["real"], dtype=torch.int64, device=dev),
                "row": _row(case, randn), "rope": Rope()}
    X, real, column, hidden = _column(case, randn)
    s = {"X": X, "real": real, "column": column, "hidden": hidden}
    if kind == "query":
        B, n = case["est"], case["train"]
        s.update(row=_row(case, randn), rope=Rope(),
                 blocks=[_block(randn, W, torch.bfloat16) for _ in range(case["blocks"])],
                 decoder=query.DecoderWeights(1 + randn(W, scale=0.05), randn(W, scale=0.05),
                                              *_linear(randn, 2 * W, W, torch.bfloat16),
                                              *_linear(randn, NCLS, 2 * W, torch.bfloat16)),
                 k=[randn(B, H, n, ID, dtype=torch.bfloat16) for _ in range(case["blocks"])],
                 v=[randn(B, H, n, ID, dtype=torch.bfloat16) for _ in range(case["blocks"])],
                 valid=torch.tensor([n], dtype=torch.int32, device=dev))
    return s


def prepare(case: dict, seed: int) -> dict:
    """The inputs and the fit-time caches a program keeps between its queries."""
    s = _inputs(case, seed)
    s["kind"] = kind = case["kind"]
    if kind == "icl_query":
        cache = icl.IclKVCache(case["est"], 1, H, case["cap"], ID, torch.bfloat16, s["q"].device)
        cache.append(0, s.pop("k"), s.pop("v"))
        s["cache"] = cache
    elif kind in ("icl_train", "column_train"):
        s["leaves"] = [s[n].requires_grad_() for n in ("q", "k", "v")]
    elif kind == "row_train":
        s["leaves"] = [s["qkv"].requires_grad_()]
    elif kind in ("column_stage", "query"):
        with torch.no_grad():
            hidden = s.pop("hidden")
            cache = query.ColumnKVCache(3, case["est"], case["features"] + C, NI, E, DT[case["dtype"]], s["X"].device)
            for b in range(3):
                cache.append_projected(b, hidden[b], s["column"].blocks[b])
        s["cache"] = cache
        if kind == "query":
            kv = icl.IclKVCache(case["est"], case["blocks"], H, case["train"], ID, torch.bfloat16, s["X"].device)
            for b, (k, v) in enumerate(zip(s.pop("k"), s.pop("v"))):
                kv.append(b, k, v)
            s["icl"] = kv
            s["weights"] = query.QueryWeights(s["column"], s["row"], s["blocks"], s["decoder"])
    return s


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def run(s: dict):
    kind = s["kind"]
    if kind == "icl_train":
        out = icl.icl_sdpa(s["q"], s["k"], s["v"])
        return [out.detach(), *torch.autograd.grad(out, s["leaves"], s["do"])]
    if kind == "column_train":
        out = pk.hx_attention(s["q"], s["k"], s["v"], H)
        return [out.detach(), *torch.autograd.grad(out, s["leaves"], s["do"])]
    if kind == "row_train":
        out = pk.pk_self_attention(s["qkv"], H, None, s["rope"], LAYER_SCALE)
        return [out.detach(), *torch.autograd.grad(out, s["leaves"], s["do"])]
    with torch.no_grad():
        if kind == "icl_query":
            return s["cache"].query(0, s["q"])
        if kind == "isab1":
            return pk.hxq_attention(s["q"], s["kv"], s["valid"], H)
        if kind == "isab2":
            return pk.pk_cross_attention(s["q"], s["kv"], H, None, None, LAYER_SCALE)
        if kind == "row":
            return pk.pk_self_attention(s["qkv"], H, s["kb"], s["rope"], LAYER_SCALE)
        if kind == "column_stage":
            return query.column_stage(s["X"], s["real"], s["cache"], s["column"])
        if kind == "row_stage":
            return query.row_stage(s["src"], s["real"], s["row"], s["rope"])
        return query.cached_query(s["X"], s["real"], s["cache"], s["icl"], s["weights"], s["valid"], s["rope"])


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _layer_flops(rows: float, width: int, keys: float) -> float:
    """One encoder layer over `rows` rows without its K|V projection: q and out projections, attention over
    `keys` keys, feed-forward of factor 2."""
    return rows * (2 * 2.0 * width * width + 4.0 * keys * width + 2 * 4.0 * width * width)


def work(case: dict) -> dict:
    kind = case["kind"]
    size = 4 if case.get("dtype") == "fp32" else 2
    if kind in ("icl_query", "icl_train"):
        n, tq, tk = case["est"] * H, case["test"], case["train"]
        fl = 4.0 * n * tq * tk * ID
        by = 2.0 * n * ID * (2 * tq + 2 * tk)
        if kind == "icl_train":  # five products backward; reads dO, writes dq, dk, dv
            fl *= 3.5
            by += 2.0 * n * ID * (2 * tq + 2 * tk)
        return {"bytes": by, "flops": fl}
    if kind in ("isab1", "isab2"):
        lq, lk = (NI, case["valid"]) if kind == "isab1" else (case["rows"], NI)
        return {"bytes": float(size * case["seqs"] * E * (2 * lq + 2 * lk)), "flops": 4.0 * case["seqs"] * lq * lk * E}
    if kind in ("row", "row_train"):
        B, n = case["rows"], case["tokens"]
        fl, by = 4.0 * B * n * n * E, float(size * B * n * E * 4)
        return {"bytes": by * 2, "flops": fl * 3.5} if kind == "row_train" else {"bytes": by, "flops": fl}
    if kind == "column_train":
        B, lq, lk = case["seqs"], case["queries"], case["keys"]
        return {"bytes": 2.0 * 2.0 * B * E * (2 * lq + 2 * lk), "flops": 3.5 * 4.0 * B * lq * lk * E}
    B, T, n = case["est"], case["test"], case["features"] + C
    wts = 8.0 * E * E * size  # one layer's weights
    col = {"bytes": B * T * case["features"] * 4.0 + size * (float(B) * n * T * E + 3.0 * B * n * NI * 2 * E) + 3 * wts,
           "flops": B * T * n * 6.0 * E + 3 * _layer_flops(float(B) * T * n, E, NI)}
    # row stage: two self-attention layers with their K|V projection, the CLS layer over all tokens' K|V
    row = {"bytes": size * (float(B) * n * T * E + float(B) * T * C * E) + 3 * wts,
           "flops": 2 * _layer_flops(float(B) * T * n, E, n) + 3 * B * T * n * 4.0 * E * E
           + _layer_flops(float(B) * T * C, E, n)}
    if kind == "column_stage":
        return col
    if kind == "row_stage":
        return row
    nb, train = case["blocks"], case["train"]
    # the tensors between the stages need not exist in memory
    return {"bytes": col["bytes"] - size * float(B) * n * T * E + 3 * wts + nb * (8.0 * W * W * 2
                                                                                + 2.0 * 2 * B * H * train * ID)
            + 2.0 * 2 * W * W + 4.0 * B * T * NCLS,
            "flops": col["flops"] + row["flops"] + nb * _layer_flops(float(B) * T, W, train)
            + B * T * (4.0 * W * W + 4.0 * W * NCLS)}


def tolerance(case: dict) -> dict:
    """About four times the largest distance from exact() measured over the ranges (in brackets)."""
    return TOLERANCES[case["kind"], case.get("dtype", "bf16")]


TOLERANCES = {
    ("icl_query", "bf16"): {"rel": 9e-3},  # [2.3e-3]
    ("icl_train", "bf16"): {"rel": 1.1e-2},  # [2.8e-3]
    ("isab1", "bf16"): {"rel": 9e-3},  # [2.4e-3]
    ("isab1", "fp32"): {"rel": 1e-5},  # [1.2e-6 at 8,000 rows, growing with their square root]
    ("isab2", "bf16"): {"rel": 9e-3},  # [2.3e-3]
    ("isab2", "fp32"): {"rel": 1e-6},  # [2.3e-7]
    ("row", "bf16"): {"rel": 1.5e-2},  # [3.6e-3]
    ("row", "fp32"): {"rel": 1e-6},  # [2.0e-7]
    ("row_train", "bf16"): {"rel": 1.6e-2},  # [4.0e-3]
    ("column_train", "bf16"): {"rel": 1.1e-2},  # [2.6e-3]
    # the reserved columns' skip value (-100) carries most of the result's norm
    ("column_stage", "bf16"): {"rel": 1.6e-3},  # [3.8e-4]
    ("column_stage", "fp32"): {"rel": 1.2e-7},  # [3.0e-8]
    ("row_stage", "bf16"): {"rel": 2.8e-2},  # [6.7e-3]
    ("row_stage", "fp32"): {"rel": 2e-6},  # [5.1e-7]
    # 12 bf16 ICL blocks deep
    ("query", "bf16"): {"rel": 4.5e-2},  # [1.1e-2]
    ("query", "fp32"): {"rel": 4e-2},  # [8.2e-3]
}


# ---------------------------------------------------------------------------------------------
# float64 restatement
# ---------------------------------------------------------------------------------------------
def _heads(x, h: int = H):
    return x.double().unflatten(-1, (h, x.shape[-1] // h)).transpose(-3, -2).contiguous()


def _merge(x):
    return x.transpose(-3, -2).flatten(-2)


def _attend(q, k, v, scale: float, mask=None):
    """softmax(q k^T scale + mask) v over [..., T, d] in float64, in slices of the leading dim and of the queries."""
    out = torch.empty(*q.shape[:-1], v.shape[-1], dtype=torch.float64, device=q.device)
    lead, tq, tk = max(1, q[0, ..., 0, 0].numel()), q.shape[-2], k.shape[-2]
    budget = 1 << 28  # scores held at once
    nq = max(1, min(tq, budget // (lead * tk)))
    nb = max(1, budget // (lead * nq * tk))
    for b in range(0, q.shape[0], nb):
        kt, vb = k[b:b + nb].double().transpose(-1, -2).contiguous(), v[b:b + nb].double()
        for t in range(0, tq, nq):
            s = torch.matmul(q[b:b + nb, ..., t:t + nq, :].double(), kt).mul_(scale)
            if mask is not None:
                s += mask.double()
            s -= s.amax(dim=-1, keepdim=True)
            s.exp_()
            out[b:b + nb, ..., t:t + nq, :] = torch.matmul(s, vb) / s.sum(dim=-1, keepdim=True)
    return out


def _attend_grad(q, k, v, do, scale: float):
    """(out, dq, dk, dv) of softmax(q k^T scale) v for leading-dim slices, float64."""
    outs = []
    for b in range(q.shape[0]):
        qb, kb, vb, db = (t[b].double() for t in (q, k, v, do))
        p = torch.softmax(torch.matmul(qb, kb.transpose(-1, -2).contiguous()) * scale, dim=-1)
        o = torch.matmul(p, vb)
        dp = torch.matmul(db, vb.transpose(-1, -2).contiguous())
        ds = p * (dp - (db * o).sum(dim=-1, keepdim=True)) * scale
        outs.append((o, torch.matmul(ds, kb), torch.matmul(ds.transpose(-1, -2).contiguous(), qb),
                     torch.matmul(p.transpose(-1, -2).contiguous(), db)))
    return [torch.stack(t) for t in zip(*outs)]


def _rotate(x, freqs, sign: float = 1.0):
    """RoPE (halves form) of [..., T, HD] at positions 0..T-1; sign -1 is its transpose."""
    ang = torch.outer(torch.arange(x.shape[-2], device=x.device, dtype=torch.float32),
                      freqs.to(x.device)).double().repeat(1, 2)
    a, b = x.chunk(2, dim=-1)
    return x * ang.cos() + sign * torch.cat([-b, a], dim=-1) * ang.sin()


def _ln(x, w, b, eps):
    return F.layer_norm(x, (x.shape[-1],), w.double(), b.double(), eps)


def _lin(x, w, b):
    return F.linear(x, w.double(), b.double())


def _ffn(x, blk):
    h = _lin(_ln(x, blk.ln2_w, blk.ln2_b, blk.eps), blk.ff1_w, blk.ff1_b)
    return x + _lin(F.gelu(h), blk.ff2_w, blk.ff2_b)


def _exact_column(X, real: int, w, hidden):
    """Column stage of one estimator: X [T, features], hidden three [columns, 128, E] -> [columns, T, E]."""
    T, nf = X.shape
    j = torch.arange(nf, device=X.device) % real
    x = torch.stack([X[:, (j + 2 ** i) % real] for i in range(3)], dim=-1)
    # rounded to the stage's dtype like any input of it
    x = x.transpose(0, 1).to(w.in_w.dtype).double()
    src = _lin(x, w.in_w, w.in_b)
    for blk, hid in zip(w.blocks, hidden):
        q = _heads(_lin(_ln(src, blk.ln1_w, blk.ln1_b, blk.eps), blk.in_w[:E], blk.in_b[:E]))
        kv = _lin(_ln(hid[C:].double(), blk.ln1_w, blk.ln1_b, blk.eps), blk.in_w[E:], blk.in_b[E:])
        a = _merge(_attend(q, _heads(kv[..., :E]), _heads(kv[..., E:]), LAYER_SCALE))
        src = _ffn(src + _lin(a, blk.out_w, blk.out_b), blk)
    skip = torch.full((C, T, E), SKIP, dtype=torch.float64, device=X.device)  # the reserved slots stay untouched
    return torch.cat([skip, src])


def _exact_row(src, real: int, w, rope):
    """Row stage of one estimator: src [tokens, T, E] -> [T, C E]."""
    x = src.double().transpose(0, 1)
    x = torch.cat([w.cls_tokens.double().expand(x.shape[0], C, E), x[:, C:]], dim=1)
    mask = torch.zeros(x.shape[1], dtype=torch.float64, device=x.device)
    mask[real + C:] = torch.finfo(torch.float32).min
    for i, blk in enumerate(w.blocks):
        last = i == len(w.blocks) - 1
        q, k, v = (_heads(t) for t in _lin(_ln(x, blk.ln1_w, blk.ln1_b, blk.eps), blk.in_w, blk.in_b).split(E, dim=-1))
        if last:  # the CLS rows alone
            q, x = q[..., :C, :], x[:, :C]
        a = _merge(_attend(_rotate(q, rope.freqs), _rotate(k, rope.freqs), v, LAYER_SCALE, mask))
        x = _ffn(x + _lin(a, blk.out_w, blk.out_b), blk)
    return _ln(x, w.out_ln_w, w.out_ln_b, w.eps).flatten(-2)


def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "icl_query":
        return _attend(s["q"], s["k"], s["v"], ID ** -0.5)
    if kind == "icl_train":
        return _attend_grad(s["q"], s["k"], s["v"], s["do"], ID ** -0.5)
    if kind in ("isab1", "isab2"):
        kv, scale = (s["kv"][:, :case["valid"]], 1.0) if kind == "isab1" else (s["kv"], LAYER_SCALE)
        out = torch.empty(s["q"].shape, dtype=torch.float64, device=kv.device)
        for b in range(0, kv.shape[0], 8):
            out[b:b + 8] = _merge(_attend(_heads(s["q"][b:b + 8]), _heads(kv[b:b + 8, :, :E]),
                                          _heads(kv[b:b + 8, :, E:]), scale))
        return out
    if kind == "column_train":
        out = _attend_grad(*(_heads(s[n]) for n in ("q", "k", "v", "do")), 1.0)
        return [_merge(t) for t in out]
    if kind in ("row", "row_train"):
        f, parts = s["rope"].freqs, []
        for x, d in zip(s["qkv"].split(512), s["do"].split(512) if kind == "row_train" else s["qkv"].split(512)):
            q, k, v = (_heads(t) for t in x.split(E, dim=-1))
            q, k = _rotate(q, f), _rotate(k, f)
            if kind == "row":
                parts.append((_merge(_attend(q, k, v, LAYER_SCALE, s["kb"])),))
                continue
            o, dq, dk, dv = _attend_grad(q, k, v, _heads(d), LAYER_SCALE)
            parts.append((_merge(o), torch.cat([_merge(_rotate(dq, f, -1.0)), _merge(_rotate(dk, f, -1.0)),
                                                _merge(dv)], dim=-1)))
        out = [torch.cat(p) for p in zip(*parts)]
        return out if kind == "row_train" else out[0]
    if kind == "row_stage":
        return torch.stack([torch.cat([_exact_row(t, case["real"], s["row"], s["rope"]) for t in src.split(512, dim=1)])
                            for src in s["src"]])
    B = case["est"]
    src = [_exact_column(s["X"][b], case["real"], s["column"], [h[b] for h in s["hidden"]]) for b in range(B)]
    if kind == "column_stage":
        return torch.stack(src)
    x = torch.stack([_exact_row(t, case["real"], s["row"], s["rope"]) for t in src])
    for blk, k, v in zip(s["blocks"], s["k"], s["v"]):
        q = _heads(_lin(_ln(x, blk.ln1_w, blk.ln1_b, blk.eps), blk.in_w[:W], blk.in_b[:W]))
        x = _ffn(x + _lin(_merge(_attend(q, k, v, ID ** -0.5)), blk.out_w, blk.out_b), blk)
    d = s["decoder"]
    return _lin(F.gelu(_lin(_ln(x, d.ln_w, d.ln_b, d.eps), d.w1, d.b1)), d.w2, d.b2)
