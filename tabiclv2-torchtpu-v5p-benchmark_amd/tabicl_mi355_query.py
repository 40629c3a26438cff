"""The whole cached-KV query of TabICLv2 on MI355X: test rows through the column blocks over their
cached inducing-point K/V, the row interactor, the cached ICL blocks and the decoder, every attention
on the HIP kernels of libtabicl_attn.so.

This is the body of the reference runner's query function (`_make_query_fn`,
scripts/tabicl_tpu_bucketed.py:768-834), the step its published 938.49 ms cached-KV query times
(results/inference/best_model_forward_and_e2e.jsonl:2):
  * column stage (:777-797): circular feature grouping of the test rows (group size 3, the reference's
    restatement at :362-372), `reserve_cls_tokens` leading feature slots filled with the skip value -100,
    the in-linear (a group of 3 values -> width 128; rows whose inputs are all the skip value stay the
    skip value), then per column block the block's second attention `multihead_attn2(src,
    cached_kv=...)` (a pre-norm encoder layer whose attention reads the cached K/V of the 128 inducing
    points) with the skip-column refill of results/tpu_patch.diff:1749-1757;
  * row interactor (`_train_forward`, diff:1276-1307 and :169-190): the CLS tokens replace the reserved
    slots, an additive key mask hides the padded feature slots (finfo.min past d + num_cls), every
    block but the last is RoPE self-attention over the row's tokens, the last block computes the CLS
    rows only (4 queries over all tokens, RoPE), then the out-LayerNorm (SafeLayerNorm) and the CLS rows
    flattened into the row representation [B, T, num_cls width];
  * ICL stage (:803-823): the cached ICL blocks (tabicl_mi355_icl.IclKVCache.query_blocks), the final
    LayerNorm (norm_first) and the decoder MLP.
Upstream tabicl (2.2.0) is not in the reference tree; the layers around the attention are restated from
these call sites. The weights are the caller's (random in the benchmark and tests: no checkpoint is
available); upstream's SSMax and RoPE modules come in as the caller's q transforms and rope object.

Attention kernels per stage: column blocks `pk_cross` over 128 cached keys (fp32: sx_resident_kernel; bf16:
sh_resident_kernel), row blocks `pk_self` with in-kernel RoPE and the key mask (sh_persist_kernel for
104 tokens in bf16), the CLS block `pk_cross` with RoPE, ICL `icl_pipe_kernel`. The rest of the
column and row layers (norms, projections, feed-forward, residuals, skip refill) runs on two fused kernels
(layer.hip: tabicl_layer_proj, tabicl_layer_tail) where _layer_native takes the layer, the column stage's
input on tabicl_column_embed, ICL blocks of up to 8192 rows on tabicl_ln_linear and tabicl_icl_block_tail, the
decoder's norm and first layer on tabicl_ln_linear; the others on torch GEMMs (hipBLASLt) and elementwise kernels. Precision follows the weights:
the reference runs the column and row stages in fp32 and the ICL stage under bf16 autocast (its
headline knobs, best_model_forward_and_e2e.jsonl:2: no column / row autocast)."""
from __future__ import annotations

from dataclasses import dataclass
from typing import Callable, Optional, Union

import torch
import torch.nn.functional as F
from torch import Tensor

import tabicl_mi355_attn as _pk
import tabicl_mi355_icl as _icl
import tabicl_mi355_native as _nat

BlockWeights = _icl.IclBlockWeights  # one pre-norm encoder layer (norms, packed in-projection, out-projection, FFN)
SKIP_VALUE = -100.0  # the column stage's skip value (scripts/tabicl_tpu_bucketed.py:708, 780)


@dataclass
class ColumnWeights:
    """Column embedder at query time: the in-linear [width, group] + bias, and for every column block the
    weights of its second attention layer (`multihead_attn2`; the first one only runs at fit time)."""
    in_w: Tensor
    in_b: Optional[Tensor]
    blocks: list
    heads: int = 8
    reserve_cls: int = 4


@dataclass
class RowWeights:
    """Row interactor: the CLS tokens [num_cls, width], the tf_row blocks (the last one computes the CLS
    rows only) and the out-LayerNorm."""
    cls_tokens: Tensor
    blocks: list
    out_ln_w: Tensor
    out_ln_b: Optional[Tensor]
    heads: int = 8
    eps: float = 1e-5


@dataclass
class DecoderWeights:
    """The ICL predictor's final LayerNorm (norm_first) and decoder MLP width -> ff -> classes."""
    ln_w: Tensor
    ln_b: Optional[Tensor]
    w1: Tensor
    b1: Optional[Tensor]
    w2: Tensor
    b2: Optional[Tensor]
    eps: float = 1e-5


def _ln(x: Tensor, w: Tensor, b: Optional[Tensor], eps: float, out_dtype: torch.dtype) -> Tensor:
    return _icl._safe_layer_norm(x, w, b, eps, out_dtype)


def _layer_native(x: Tensor, blk, activation) -> bool:  # noqa: ANN001
    """Whether the library's layer kernels (tabicl_layer_proj, tabicl_layer_tail) take a layer: rows of width
    128 and feed-forward width 256 with the erf GELU, x and the GEMM weights of one dtype (bf16 / fp32),
    contiguous and 16-byte aligned, fp32 LayerNorm parameters, no gradient."""
    E = x.shape[-1]
    if activation is not F.gelu or x.device.type != "cuda" or E != 128 or not blk.eps > 0.0 \
            or x.dtype not in (torch.bfloat16, torch.float32) or x.numel() // E > 0xffffffff:
        return False
    if blk.ln1_w is None or blk.ln2_w is None or not _nat.direct(x):
        return False
    dev, grad, dt = x.get_device(), torch.is_grad_enabled(), x.dtype
    for t, n, k in ((blk.in_w, 384, 128), (blk.out_w, 128, 128), (blk.ff1_w, 256, 128), (blk.ff2_w, 128, 256)):
        if not _nat.plain(t, n * k, dt, dev, grad) or t.shape != (n, k) or t.data_ptr() % 16:
            return False
    for t, n in ((blk.in_b, 384), (blk.out_b, 128), (blk.ff1_b, 256), (blk.ff2_b, 128)):
        if t is not None and (t.dim() != 1 or not _nat.plain(t, n, dt, dev, grad)):
            return False
    return all(t is None or _nat.plain(t, 128, torch.float32, dev, grad)
               for t in (blk.ln1_w, blk.ln1_b, blk.ln2_w, blk.ln2_b))


def _rows128(x: Tensor) -> bool:
    """x is rows of 128 the layer kernels read in place: contiguous and 16-byte aligned."""
    return x.is_contiguous() and x.data_ptr() % 16 == 0


def _layer_ws(n_out: int, rows: int, x: Tensor):
    """(scratch tensor or None, its bytes) of one layer-kernel call, from torch's caching allocator."""
    code = _nat.dtype_code(x.dtype)
    n = int(_nat.load().tabicl_layer_workspace_bytes(n_out, rows, code)) if code == _nat.DTYPE_F32 else 0
    return (torch.empty(n, dtype=torch.uint8, device=x.device), n) if n else (None, 0)


def _layer_proj(x: Tensor, blk, lo: int, hi: int, live: Optional[Tensor] = None, group_rows: int = 1,  # noqa: ANN001
                skip: float = 0.0) -> Tensor:
    """LN1(x) W[lo:hi]^T + b[lo:hi] of the packed in-projection in one kernel; live: see tabicl_layer_proj."""
    E, es = x.shape[-1], x.element_size()
    out = torch.empty(*x.shape[:-1], hi - lo, dtype=x.dtype, device=x.device)
    ws, nws = _layer_ws(hi - lo, x.numel() // E, x)
    _nat.call("tabicl_layer_proj", x.data_ptr(), blk.ln1_w.data_ptr(), _nat.ptr(blk.ln1_b), float(blk.eps),
              blk.in_w.data_ptr() + lo * E * es, None if blk.in_b is None else blk.in_b.data_ptr() + lo * es,
              out.data_ptr(), x.numel() // E, hi - lo, _nat.dtype_code(x.dtype),
              _nat.ptr(live), group_rows, skip, _nat.ptr(ws), nws, _nat.stream_of(x))
    return out


def _layer_tail(a: Tensor, x: Tensor, blk, live: Optional[Tensor] = None, group_rows: int = 1,  # noqa: ANN001
                skip: float = 0.0) -> Tensor:
    """x + a Wo^T + bo, then + FFN(LN2(.)): the rest of a layer after its attention a, in one kernel."""
    out = torch.empty_like(x)
    ws, nws = _layer_ws(0, x.numel() // x.shape[-1], x)
    _nat.call("tabicl_layer_tail", a.data_ptr(), x.data_ptr(), blk.out_w.data_ptr(), _nat.ptr(blk.out_b),
              blk.ln2_w.data_ptr(), _nat.ptr(blk.ln2_b), float(blk.eps), blk.ff1_w.data_ptr(), _nat.ptr(blk.ff1_b),
              blk.ff2_w.data_ptr(), _nat.ptr(blk.ff2_b), out.data_ptr(), x.numel() // x.shape[-1],
              _nat.dtype_code(x.dtype), _nat.ptr(live), group_rows, skip, _nat.ptr(ws), nws, _nat.stream_of(x))
    return out


def _after_attention(a: Tensor, x: Tensor, blk, activation) -> Tensor:  # noqa: ANN001
    """The layer's output from its residual stream x and its attention a (before the out-projection)."""
    if _layer_native(x, blk, activation) and a.dtype == x.dtype and a.shape == x.shape and _rows128(x) \
            and _rows128(a) and _nat.direct(a):
        return _layer_tail(a, x, blk)
    return _ffn(x, blk, activation, F.linear(a, blk.out_w, blk.out_b))


def _pre_projection(x: Tensor, blk, activation, lo: int, hi: int) -> Tensor:  # noqa: ANN001
    """LN1(x) through rows [lo, hi) of the packed in-projection."""
    if _layer_native(x, blk, activation) and _rows128(x):
        return _layer_proj(x, blk, lo, hi)
    return F.linear(_ln(x, blk.ln1_w, blk.ln1_b, blk.eps, blk.in_w.dtype), blk.in_w[lo:hi],
                    None if blk.in_b is None else blk.in_b[lo:hi])


def _ffn(x: Tensor, blk, activation, delta: Optional[Tensor] = None) -> Tensor:  # noqa: ANN001
    """x + W2 act(W1 LN2(x) + b1) + b2 (the feed-forward half of a pre-norm encoder layer); with delta
    (the attention half's output) x + delta first, fused with LN2."""
    if delta is None:
        h = _ln(x, blk.ln2_w, blk.ln2_b, blk.eps, blk.ff1_w.dtype)
    else:
        x, h = _icl.add_layer_norm(x, delta.to(x.dtype), blk.ln2_w, blk.ln2_b, blk.eps, blk.ff1_w.dtype)
    return x + F.linear(activation(F.linear(h, blk.ff1_w, blk.ff1_b)), blk.ff2_w, blk.ff2_b).to(x.dtype)


def feature_grouping(X: Tensor, real_features: Optional[Tensor] = None, group_size: int = 3) -> Tensor:
    """Circular feature grouping ("same" mode) of X [B, T, H]: slot j of the result holds the values of
    features (j mod rf + 2^i) mod rf for i < group_size, rf = the table's real feature count
    (real_features [B], default H): [B, T, H, group_size]. The reference's restatement of upstream's
    grouping, indices computed once per table (scripts/tabicl_tpu_bucketed.py:362-372)."""
    B, T, H = X.shape
    idx = torch.arange(H, dtype=torch.long, device=X.device).view(1, 1, H)
    rf = torch.full((B, 1, 1), H, dtype=torch.long, device=X.device) if real_features is None \
        else real_features.to(device=X.device, dtype=torch.long).view(B, 1, 1)
    base = idx % rf
    return torch.stack([torch.gather(X, 2, ((base + 2 ** i) % rf).expand(B, T, H)) for i in range(group_size)],
                       dim=-1)


class ColumnKVCache:
    """Fit-time K|V of every column block's second attention: [blocks, B, columns, inducing, 2 width],
    the packed rows (K columns [0, width), V [width, 2 width)) that pk_cross reads, so the query makes no
    copy. Upstream's need_kv returns the same K/V head-split (diff:1569-1575, cached at
    scripts/tabicl_tpu_bucketed.py:719-724); the dispatch route for that form merges them per call."""

    def __init__(self, blocks: int, batch: int, columns: int, inducing: int, width: int,
                 dtype: torch.dtype = torch.float32, device: Union[str, torch.device] = "cuda"):
        self.kv = torch.empty(blocks, batch, columns, inducing, 2 * width, dtype=dtype, device=device)
        self.width = width
        self.filled = [False] * blocks

    def append_projected(self, block: int, hidden: Tensor, blk) -> None:  # noqa: ANN001
        """K|V of block `block` from the first attention's output hidden [B, columns, inducing, width]:
        the layer's pre-norm (norm1 normalises the keys too, diff:505-508), then the K|V thirds of its
        packed in-projection (one GEMM)."""
        E = self.width
        if tuple(hidden.shape) != tuple(self.kv.shape[1:-1]) + (E,):
            raise ValueError(f"hidden must be {tuple(self.kv.shape[1:-1]) + (E,)}, got {tuple(hidden.shape)}")
        h = _ln(hidden, blk.ln1_w, blk.ln1_b, blk.eps, blk.in_w.dtype)
        self.kv[block] = F.linear(h, blk.in_w[E:], None if blk.in_b is None else blk.in_b[E:]).to(self.kv.dtype)
        self.filled[block] = True


def _skippable_linear(x: Tensor, w: Tensor, b: Optional[Tensor], skip: float) -> Tensor:
    """x W^T + b, with rows whose inputs all equal the skip value left at the skip value."""
    out = F.linear(x, w, b)
    return torch.where((x == skip).all(dim=-1, keepdim=True), torch.full((), skip, dtype=out.dtype, device=out.device),
                       out)


def _embed_native(X: Tensor, real_features: Optional[Tensor], w: ColumnWeights, group_size: int) -> bool:
    """Whether tabicl_column_embed takes the stage's input: fp32 rows in groups of three, in-linear
    [128, 3] in bf16 / fp32, real feature counts as int64 on the GPU, no gradient."""
    if group_size != 3 or X.dim() != 3 or X.dtype != torch.float32 or X.numel() == 0 or not X.is_contiguous() \
            or tuple(w.in_w.shape) != (128, 3) or w.in_w.dtype not in (torch.bfloat16, torch.float32) \
            or X.shape[0] * (X.shape[2] + w.reserve_cls) > 65535 or w.reserve_cls < 0:
        return False
    vecs = ((w.in_w, 384, w.in_w.dtype), (w.in_b, 128, w.in_w.dtype), (real_features, X.shape[0], torch.int64))
    return _nat.direct(X, w.in_w, w.in_b, real_features) and (w.in_b is None or w.in_b.dim() == 1) and all(
        t is None or (t.numel() == n and t.dtype == dt and t.is_contiguous() and t.device == X.device)
        for t, n, dt in vecs)


def _column_embed(X: Tensor, real_features: Optional[Tensor], w: ColumnWeights) -> Tensor:
    """[B, H + reserve, T, 128]: feature_grouping, the reserved columns and the skippable in-linear in one
    kernel."""
    B, T, H = X.shape
    out = torch.empty(B, H + w.reserve_cls, T, 128, dtype=w.in_w.dtype, device=X.device)
    _nat.call("tabicl_column_embed", X.data_ptr(), _nat.ptr(real_features), w.in_w.data_ptr(), _nat.ptr(w.in_b),
              out.data_ptr(), B, T, H, w.reserve_cls, SKIP_VALUE, _nat.dtype_code(w.in_w.dtype), _nat.stream_of(X))
    return out


def column_stage(X: Tensor, real_features: Optional[Tensor], cache: ColumnKVCache, w: ColumnWeights,
                 group_size: int = 3, activation: Callable[[Tensor], Tensor] = F.gelu,
                 q_transform: Optional[Callable[[int, Tensor], Tensor]] = None) -> Tensor:
    """Test rows X [B, T, H] through the column embedder with cached K/V: [B, H + reserve, T, width]
    in the weights' dtype (scripts/tabicl_tpu_bucketed.py:777-792). Each block:
        x = x + out_proj(pk_cross(LN1(x) W_q^T + b_q, cached K|V)),  x = x + FFN(LN2(x)),
    then columns whose input was all skip value are refilled with it. q_transform(block, q) stands for a
    module applied to the block's q (none in upstream's second attention)."""
    _nat.require_device(X, cache.kv)
    E, h = cache.width, w.heads
    dt = w.in_w.dtype
    if _embed_native(X, real_features, w, group_size):
        src = _column_embed(X, real_features, w)
    else:
        x = feature_grouping(X, real_features, group_size)
        if w.reserve_cls:
            x = F.pad(x, (0, 0, w.reserve_cls, 0), value=SKIP_VALUE)
        src = _skippable_linear(x.transpose(1, 2).to(dt), w.in_w, w.in_b, SKIP_VALUE)  # [B, HC, T, E]
    skip = torch.full((), SKIP_VALUE, dtype=src.dtype, device=src.device)
    T = src.shape[2]
    native = [_layer_native(src, blk, activation) and _rows128(src) and T > 0 for blk in w.blocks]
    # per block and column: nonzero once the column is seen to hold anything but the skip value
    live = torch.zeros(len(w.blocks), src.shape[0] * src.shape[1], dtype=torch.int32, device=src.device) \
        if any(native) else None
    for b, blk in enumerate(w.blocks):
        if not cache.filled[b]:
            raise ValueError(f"column block {b} of the cache was never filled")
        if native[b]:
            q = _layer_proj(src, blk, 0, E, live[b], T, SKIP_VALUE)
        else:
            skip_mask = (src == skip).all(dim=-1, keepdim=True).all(dim=-2, keepdim=True)
            q = F.linear(_ln(src, blk.ln1_w, blk.ln1_b, blk.eps, blk.in_w.dtype), blk.in_w[:E],
                         None if blk.in_b is None else blk.in_b[:E])
        if q_transform is not None:
            q = q_transform(b, q)
        kv = cache.kv[b]
        if kv.dtype != q.dtype:
            kv = kv.to(q.dtype)
        a = _pk.pk_cross_attention(q, kv, h, None, None, (E // h) ** -0.5)
        if native[b] and a.dtype == src.dtype and a.shape == src.shape and _rows128(a) and _nat.direct(a):
            src = _layer_tail(a, src, blk, live[b], T, SKIP_VALUE)
            continue
        if native[b]:
            skip_mask = (live[b] == 0).view(src.shape[0], src.shape[1], 1, 1)
        src = torch.where(skip_mask, skip, _ffn(src, blk, activation, F.linear(a, blk.out_w, blk.out_b)))
    return src


def feature_key_mask(B: int, HC: int, real_features: Optional[Tensor], num_cls: int, device,  # noqa: ANN001
                     dtype: torch.dtype) -> Optional[Tensor]:
    """Additive key mask [B, 1, HC] over a row's tokens: 0 for the CLS slots and the table's real
    features (token index < d + num_cls), finfo(dtype).min after (diff:172-190); None without d."""
    if real_features is None:
        return None
    cond = torch.arange(HC, device=device).view(1, 1, HC) < (real_features.to(device).view(B, 1, 1) + num_cls)
    return torch.where(cond, torch.zeros((), dtype=dtype, device=device),
                       torch.full((), torch.finfo(dtype).min, dtype=dtype, device=device))


def row_stage(src: Tensor, real_features: Optional[Tensor], w: RowWeights, rope,  # noqa: ANN001
              activation: Callable[[Tensor], Tensor] = F.gelu) -> Tensor:
    """The column output src [B, HC, T, width] as rows of HC tokens through the row interactor:
    [B, T, num_cls width] (diff:1276-1307). Every block but the last: x = x + out_proj(pk_self(LN1(x)
    W^T + b, RoPE, key mask)), x = x + FFN(LN2(x)); the last block takes the CLS rows as queries over
    all tokens (keys normalised by the same norm1), pk_cross with RoPE on both sides; then the
    out-LayerNorm and the CLS rows flattened."""
    B, HC, T, E = src.shape
    C, h = w.cls_tokens.shape[0], w.heads
    x = src.transpose(1, 2)  # [B, T, HC, E]
    x = torch.cat([w.cls_tokens.to(device=x.device, dtype=x.dtype).expand(B, T, C, E), x[:, :, C:]], dim=2)
    kb = feature_key_mask(B, HC, real_features, C, x.device, x.dtype)
    kb = None if kb is None else kb.view(B, 1, HC).float()
    scale = (E // h) ** -0.5
    for blk in w.blocks[:-1]:
        qkv = _pre_projection(x, blk, activation, 0, 3 * E)
        x = _after_attention(_pk.pk_self_attention(qkv, h, kb, rope, scale), x, blk, activation)
    blk = w.blocks[-1]
    cls = x[:, :, :C].contiguous()
    q = _pre_projection(cls, blk, activation, 0, E)
    kv = _pre_projection(x, blk, activation, E, 3 * E)
    cls = _after_attention(_pk.pk_cross_attention(q, kv, h, kb, rope, scale), cls, blk, activation)
    cls = _ln(cls, w.out_ln_w, w.out_ln_b, w.eps, cls.dtype)
    return cls.flatten(-2)


def decode(x: Tensor, w: DecoderWeights, activation: Callable[[Tensor], Tensor] = F.gelu) -> Tensor:
    """Final LayerNorm and decoder MLP of the ICL predictor, logits in fp32 (scripts/tabicl_tpu_bucketed.py
    :819-823)."""
    if activation is F.gelu and _icl._ln_linear_native(x, w.ln_w, w.ln_b, w.eps, w.w1, w.b1):
        h = _icl._ln_linear(x, w.ln_w, w.ln_b, w.eps, w.w1, w.b1, True)
    else:
        h = activation(F.linear(_ln(x, w.ln_w, w.ln_b, w.eps, w.w1.dtype), w.w1, w.b1))
    return F.linear(h, w.w2, w.b2).float()


@dataclass
class QueryWeights:
    column: ColumnWeights
    row: RowWeights
    icl_blocks: list
    decoder: DecoderWeights


def cached_query(X: Tensor, real_features: Optional[Tensor], col_cache: ColumnKVCache, icl_cache,  # noqa: ANN001
                 w: QueryWeights, train_size: Union[int, Tensor], rope,
                 icl_q_transform: Optional[Callable[[Tensor], Tensor]] = None,
                 activation: Callable[[Tensor], Tensor] = F.gelu) -> Tensor:
    """Logits [B, T, classes] of test rows X [B, T, H] (B = estimators) from the fit-time caches: column
    stage, row interactor, the ICL blocks over the cached train rows (keys >= train_size masked) and the
    decoder (scripts/tabicl_tpu_bucketed.py:768-834). The ICL stage's GEMMs run in its weights' dtype
    (bf16: the reference's autocast of that stage) around an fp32 residual stream (the row representation
    in fp32)."""
    src = column_stage(X, real_features, col_cache, w.column, activation=activation)
    reprs = row_stage(src, real_features, w.row, rope, activation)
    x = icl_cache.query_blocks(reprs.float(), w.icl_blocks, train_size, icl_q_transform, activation)
    return decode(x, w.decoder, activation)
