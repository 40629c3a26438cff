"""Edges of the small-head kernels' key ranges, fp32 (resident, LDS and streaming forms) and bf16 with RoPE or
a mask, against the CPU oracle: lengths on both sides of every tile and dispatch line, masks, valid lengths,
non-finite inputs. Bars: tests/parity.py; fp32 results also in the 2-norm (2e-6: the kernels sit at 2e-7 to 6e-7 at these
lengths, with RoPE up to 1.6e-6 at 800 positions, where the fp32 angles of the tables count; with scores from splits
without their low plane they would be off by 4.3e-6)."""
import numpy as np
import pytest
import torch

from oracle import attention as O
from parity import check, check_norm
from test_gpu_smallhead import E, H, _attn, _gen, _Rope, _rope_np

pytestmark = pytest.mark.gpu
FMIN = torch.finfo(torch.float32).min
F32, BF16 = torch.float32, torch.bfloat16


def _check(out, want, dtype, what):
    check(out, want, dtype, what)
    if dtype == F32:
        check_norm(out, want, what)


def _self(dev, B, L, dtype, rope, kb, seed):
    x = torch.randn(B, L, 3 * E, generator=_gen(seed)).to(dtype)
    print(f"[edges] B={B} L={L} {dtype} rope={rope is not None} mask={kb is not None}", flush=True)
    out = _attn().pk_self_attention(x.to(dev), H, None if kb is None else kb.to(dev), rope, 16 ** -0.5)
    torch.cuda.synchronize()
    _check(out, O.pk_self_ref(x, H, kb, None if rope is None else _rope_np(rope, L), 16 ** -0.5), dtype, "self")


@pytest.mark.parametrize("dtype,lengths,dims", [
    (F32, (1, 12, 15, 16, 17, 32, 33, 112, 113, 128, 129, 192, 193, 384, 385), None),
    (F32, (1, 16, 17, 128, 129, 192, 193, 384, 385, 768, 769), 16),
    (F32, (17, 128, 200, 800), 8),
    (BF16, (129, 160, 161, 192, 193, 384, 385, 768, 769), 16),
    (BF16, (1, 12, 17, 32, 33, 104, 128, 129, 400), 8),
])
@pytest.mark.parametrize("masked", [False, True])
def test_self_lengths(dev, dtype, lengths, dims, masked):
    # masked: finite biases, keys shut out by the lowest value at scattered places (not a prefix mask)
    for L in lengths:
        kb = None
        if masked:
            g = _gen(L)
            kb = torch.randn(2, L, generator=g)
            kb[torch.rand(2, L, generator=g) < 0.3] = FMIN
            kb[:, L // 2] = 0.0
        _self(dev, 2, L, dtype, None if dims is None else _Rope(dim=dims, interleaved=L % 2 == 1), kb, L)


@pytest.mark.parametrize("Lk", [16, 40, 150, 300, 600, 2100])
def test_fp32_valid_lengths(dev, Lk):
    # valid lengths 0 (zeros), 1, around a 16-key group and full; the rows past them hold NaN
    valid = [0, 1, 15, 16, Lk - 1, Lk]
    g = _gen(Lk)
    q = torch.randn(len(valid), 37, E, generator=g) * 0.25
    kv = torch.randn(len(valid), Lk, 2 * E, generator=g)
    want = O.hxq_ref(q, kv, np.array(valid), H)
    for b, v in enumerate(valid):
        kv[b, v:] = float("nan")
    print(f"[edges] valid lengths Lk={Lk}", flush=True)
    out = _attn().hxq_attention(q.to(dev), kv.to(dev), torch.tensor(valid).to(dev), H)
    torch.cuda.synchronize()
    assert bool((out[0] == 0).all())
    _check(out[1:], want[1:], F32, "valid")


@pytest.mark.parametrize("dtype,L,rope", [(F32, 20, False), (F32, 128, True), (F32, 150, False), (F32, 300, True),
                                          (F32, 900, False), (BF16, 129, True), (BF16, 300, True), (BF16, 768, True)])
def test_all_keys_at_the_lowest_value(dev, dtype, L, rope):
    # every score becomes the same lowest value: uniform weights
    x = torch.randn(2, L, 3 * E, generator=_gen(L)).to(dtype)
    kb = torch.full((2, L), FMIN)
    print(f"[edges] all masked {dtype} {L}", flush=True)
    out = _attn().pk_self_attention(x.to(dev), H, kb.to(dev), _Rope() if rope else None, 16 ** -0.5)
    torch.cuda.synchronize()
    _check(out, x[..., 2 * E:].double().mean(dim=1, keepdim=True).expand(2, L, E), dtype, "uniform")


@pytest.mark.parametrize("dtype,L,rope", [(F32, 20, False), (F32, 128, True), (F32, 150, False), (F32, 300, True),
                                          (F32, 900, False), (BF16, 150, True), (BF16, 500, True)])
def test_non_finite_values(dev, dtype, L, rope):
    # an infinite value reaches its own head's dim alone, with its sign; a NaN key its own head and batch
    # element alone
    x = torch.randn(2, L, 3 * E, generator=_gen(L)).to(dtype)
    ro = _Rope() if rope else None
    want = O.pk_self_ref(x, H, None, None if ro is None else _rope_np(ro, L), 16 ** -0.5)
    want = torch.as_tensor(np.asarray(want))
    x[0, 3, 2 * E + 5] = float("-inf")
    x[1, 4, E + 40] = float("nan")
    print(f"[edges] non-finite {dtype} {L}", flush=True)
    out = _attn().pk_self_attention(x.to(dev), H, None, ro, 16 ** -0.5).cpu()
    assert bool((out[0, :, 5] == float("-inf")).all()) and bool(out[1, :, 32:48].isnan().all())
    keep = torch.ones(2, L, E, dtype=torch.bool)
    keep[0, :, 5] = False
    keep[1, :, 32:48] = False
    _check(out[keep], want[keep], dtype, "finite part")


@pytest.mark.parametrize("B,Lq,Lk", [(64, 128, 400), (64, 128, 1024), (40, 128, 2500), (2, 128, 2100), (3, 17, 900)])
def test_fp32_mask_over_whole_parts_keeps_the_fast_pass(dev, B, Lq, Lk):
    # fp32 keys beyond the LDS form are split over the waves of a workgroup. Keys shut out by a mask give whole parts
    # without weight; the row must not go through the exact pass for that (5 times the time). A bias of -300 leaves
    # such a part trusted by itself and its weight zero (exp2 of -430 and less), so both calls are the same sums of the
    # same products: equal bits. The exact pass sums on other matrix units, with other bits.
    g = _gen(Lk)
    q = (torch.randn(B, Lq, E, generator=g) * 0.25).to(dev)
    kv = torch.randn(B, Lk, 2 * E, generator=g).to(dev)
    n, outs = Lk * 3 // 10, []
    for low in (-1e30, -300.0):
        kb = torch.full((1, Lk), low)
        kb[:, :n] = 0.0
        print(f"[edges] masked parts B={B} Lq={Lq} Lk={Lk} {low}", flush=True)
        outs.append(_attn().hxq_attention(q, kv, torch.tensor([Lk]), H, key_bias=kb.to(dev)).cpu())
    assert torch.equal(outs[0], outs[1])
    _check(outs[0][:1], O.hxq_ref(q[:1].cpu(), kv[:1, :n].cpu(), np.array([n]), H), F32, "prefix")
    kb = torch.full((1, Lk), -1e30)
    kb[:, Lk - n:] = 0.0
    out = _attn().hxq_attention(q, kv, torch.tensor([Lk]), H, key_bias=kb.to(dev)).cpu()
    _check(out[:1], O.hxq_ref(q[:1].cpu(), kv[:1, Lk - n:].cpu(), np.array([n]), H), F32, "suffix")


@pytest.mark.parametrize("Lk,low", [(900, -60.0), (2100, -60.0), (2100, -1e30)])
def test_fp32_parts_without_weight_beside_low_scores(dev, Lk, low):
    # one live key group in the second half, far below zero: parts whose keys are all masked may not be left out on
    # the strength of that row's sum; with low = -1e30 every key is masked and the weights are uniform over the row
    g = _gen(Lk)
    q, kv = torch.randn(2, 40, E, generator=g) * 0.25, torch.randn(2, Lk, 2 * E, generator=g)
    kb = torch.full((2, Lk), -1e30)
    kb[:, Lk - 40:Lk - 10] = low
    print(f"[edges] low scores Lk={Lk} {low}", flush=True)
    out = _attn().hxq_attention(q.to(dev), kv.to(dev), torch.tensor([Lk]), H, key_bias=kb.to(dev)).cpu()
    if low == -60.0:
        want = O.hxq_ref(q, kv[:, Lk - 40:Lk - 10].contiguous(), np.array([30, 30]), H)
    else:
        want = kv[..., E:].double().mean(dim=1, keepdim=True).expand(2, 40, E)
    check(out, want, F32, "low scores")  # scores of -86 in log2 units: a rounding of one is 4e-6 of its weight


@pytest.mark.parametrize("L,dims,shut", [(12, 8, 0), (28, 8, 0), (104, 8, 0), (129, 16, 0), (200, 16, 0), (260, 16, 0),
                                         (129, 16, 64), (200, 16, 128), (140, None, 70)])
def test_bf16_rows_are_as_close_as_fp32_softmax_with_bf16_weights(dev, L, dims, shut):
    # bf16 with RoPE: besides its operands q' and k' (rounded in the oracle too) the kernel rounds the weights and the
    # result. The error of a softmax in float64 whose weights, the largest of the first 64 keys 1, and result are
    # rounded to bf16 and whose row sums are not: 1.95e-3 (12 keys) to 2.28e-3 of the result's 2-norm. The kernel may
    # not be further off (half a percent: a few fp32 roundings fall on the other side of a bf16 tie).
    # shut: that many leading keys masked; the reference is then the first 64-key tile's with a live key.
    B, ro = 24, None if dims is None else _Rope(dim=dims)
    x = torch.randn(B, L, 3 * E, generator=_gen(L)).to(BF16)
    kb = torch.zeros(1, L)
    kb[:, :shut] = FMIN
    tab = None if ro is None else _rope_np(ro, L)
    want = torch.as_tensor(np.asarray(O.pk_self_ref(x, H, kb if shut else None, tab, 16 ** -0.5, cast=BF16)))
    heads = lambda t: torch.as_tensor(t).unflatten(-1, (H, 16)).transpose(1, 2)  # noqa: E731
    rope = lambda t: t if tab is None else O.rope_merged_ref(t, tab[0], tab[1], H, *tab[2:])  # noqa: E731
    q, k = (heads(O._cast(rope(x[..., lo:lo + E].double().numpy()) * s, BF16)) for lo, s in ((0, 16 ** -0.5), (E, 1.0)))
    s = q @ k.transpose(-1, -2) + kb.double().clamp_min(-1e30)
    p = torch.exp(s - s[..., shut // 64 * 64:][..., :64].amax(-1, keepdim=True))
    ref = (p.to(BF16).double() @ heads(x[..., 2 * E:].double())) / p.sum(-1, keepdim=True)
    ref = ref.transpose(1, 2).flatten(-2).to(BF16).double()
    print(f"[edges] bf16 rows L={L} dims={dims} shut={shut}", flush=True)
    out = _attn().pk_self_attention(x.to(dev), H, kb.to(dev) if shut else None, ro, 16 ** -0.5).cpu().double()
    err, bar = float((out - want).norm() / want.norm()), float((ref - want).norm() / want.norm())
    assert err <= 1.005 * bar, (err, bar)


@pytest.mark.parametrize("dtype,L,dims", [(F32, 33, None), (F32, 97, None), (F32, 97, 16), (F32, 200, None), (F32, 500, 16),
                                          (F32, 900, None), (F32, 2100, None), (BF16, 33, 8), (BF16, 129, 16),
                                          (BF16, 700, 16)])
def test_values_near_the_largest_float(dev, dtype, L, dims):
    # one key with high scores and a value of 3e38: weights are at most 1, so the weighted sum is finite, also where the
    # key's score lies above the reference of the first keys and the exact pass takes the row
    x = torch.randn(2, L, 3 * E, generator=_gen(L))
    x[1, L - 2, E:2 * E] *= 3
    x[1, L - 2, 2 * E:] = 3e38
    x = x.to(dtype)
    ro = None if dims is None else _Rope(dim=dims)
    want = torch.as_tensor(np.asarray(O.pk_self_ref(x, H, None, None if ro is None else _rope_np(ro, L), 16 ** -0.5)))
    print(f"[edges] large values {dtype} {L}", flush=True)
    out = _attn().pk_self_attention(x.to(dev), H, None, ro, 16 ** -0.5).cpu().double()
    assert bool(out.isfinite().all())
    assert float((out - want)[1].abs().max()) <= (2e-2 if dtype == BF16 else 1e-4) * float(want[1].abs().max())


@pytest.mark.parametrize("dtype,dims,B,L", [(BF16, 8, 4300000, 2), (F32, None, 8500000, 1), (F32, 16, 600000, 3)])
def test_many_sequences(dev, dtype, dims, B, L):
    # more sequences than one grid's 2^32 threads take: launched in slices, each of which must be whole, with its own
    # masks. Against calls of a few sequences (the same kernel, the same bits) at the slices' ends.
    x = torch.empty(B, L, 3 * E, dtype=dtype, device=dev).normal_()
    kb = torch.zeros(B, L, device=dev)
    kb[1::2, L - 1] = -1.5
    ro = None if dims is None else _Rope(dim=dims)
    print(f"[edges] {B} sequences of {L} {dtype}", flush=True)
    out = _attn().pk_self_attention(x, H, kb, ro, 16 ** -0.5)
    for i in (0, (1 << 18) - 2, 2 * (1 << 18) - 2, (B >> 18 << 18) - 2, B - 4):
        few = _attn().pk_self_attention(x[i:i + 4].clone(), H, kb[i:i + 4].clone(), ro, 16 ** -0.5)
        assert torch.equal(out[i:i + 4], few), i
