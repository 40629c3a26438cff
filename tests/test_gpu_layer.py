"""GPU parity of the encoder-layer kernels around the small-head attention (tabicl_layer_proj,
tabicl_layer_tail) against the same layer in float64 on the same (dtype-rounded) inputs.

Bars: fp32 max abs error <= 1e-4 and <= 1e-3 x max |ref| (tests/parity.py), and 2e-6 in the 2-norm relative to the
result (tests/parity.py: the kernels sit at 2e-7; splits without their low plane are off by 3.4e-6). bf16: products of
bf16 operands with fp32 sums; the operands LN(.), GELU(.) and the output are rounded to bf16 (relative 2^-9 each), so an
output of scale S is off by a few 2^-9 S: 2e-2 x max |ref|. Row counts: one row, around a wave's 32 and a
workgroup's 128 rows, enough tiles that the projection is not split over workgroups.
"""
import pytest
import torch
import torch.nn.functional as F

from parity import check, check_norm
from query_ref import block_weights

pytestmark = pytest.mark.gpu
E = 128


def _block(dtype, seed, bias=True):
    g = torch.Generator().manual_seed(seed)
    w = block_weights(E, 2 * E, g, dtype)
    if not bias:
        w.ln1_b = w.in_b = w.out_b = w.ln2_b = w.ff1_b = w.ff2_b = None
    return w, g


def _ln64(x, w, b, eps):
    return F.layer_norm(x.double(), (E,), w.double(), None if b is None else b.double(), eps)


def _lin64(x, w, b):
    return F.linear(x, w.double(), None if b is None else b.double())


def _tail64(a, x, w):
    s = x.double() + _lin64(a.double(), w.out_w, w.out_b)
    return s + _lin64(F.gelu(_lin64(_ln64(s, w.ln2_w, w.ln2_b, w.eps), w.ff1_w, w.ff1_b)), w.ff2_w, w.ff2_b)


def _check(out, ref, dtype, what):
    scale = max(1.0, float(ref.abs().max()))
    check(out, ref, dtype, what, abs_tol=(1e-4 if dtype == torch.float32 else 2e-2) * scale)
    if dtype == torch.float32:
        check_norm(out, ref, what)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,bias", [(1, True), (31, True), (33, False), (128, True), (129, True), (4099, False),
                                       (70001, True)])
def test_projection_and_tail(dev, dtype, rows, bias):
    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(dtype, rows, bias)
    x = (torch.randn(rows, E, generator=g) * 2 + 0.5).to(dtype)
    a = torch.randn(rows, E, generator=g).to(dtype)
    wd, xd, ad = to_device(w, dev), x.to(dev), a.to(dev)
    assert Q._layer_native(xd, wd, F.gelu)
    print(f"[layer] rows={rows} {dtype}", flush=True)
    for lo, hi in ((0, E), (E, 3 * E), (0, 3 * E)):
        out = Q._layer_proj(xd, wd, lo, hi)
        torch.cuda.synchronize()
        ref = _lin64(_ln64(x, w.ln1_w, w.ln1_b, w.eps), w.in_w[lo:hi], None if w.in_b is None else w.in_b[lo:hi])
        _check(out, ref, dtype, f"proj {lo}:{hi}")
    out = Q._layer_tail(ad, xd, wd)
    torch.cuda.synchronize()
    _check(out, _tail64(a, x, w), dtype, "tail")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 50, 128, 300, 4700])  # 4700: the fp32 projection on splits (32,768 rows on)
def test_skip_groups(dev, dtype, T):
    # groups of T rows: 0, 3 and 4 hold the skip value throughout, group 2 in all rows but one value
    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(dtype, T)
    x = torch.randn(7, T, E, generator=g).to(dtype)
    x[0] = x[3] = x[4] = -100.0
    x[2] = -100.0
    x[2, T - 1, E - 1] = 1.0
    a = torch.randn(7, T, E, generator=g).to(dtype)
    wd, xd = to_device(w, dev), x.to(dev)
    live = torch.zeros(7, dtype=torch.int32, device=dev)
    Q._layer_proj(xd, wd, 0, E, live, T, -100.0)
    out = Q._layer_tail(a.to(dev), xd, wd, live, T, -100.0)
    torch.cuda.synchronize()
    assert (live.cpu() != 0).tolist() == [False, True, True, False, False, True, True]
    dead = torch.tensor([0, 3, 4])
    assert torch.equal(out.cpu()[dead], x[dead])
    keep = torch.tensor([1, 2, 5, 6])
    _check(out.cpu()[keep], _tail64(a, x, w)[keep], dtype, f"live groups T={T}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gelu_range(dev, dtype):
    # feed-forward inputs from -40 to 40 and beyond float range: W1 = 0, so gelu sees b1 alone
    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(dtype, 5)
    w.ff1_w = torch.zeros_like(w.ff1_w)
    w.ff1_b = torch.linspace(-40.0, 40.0, 2 * E).to(dtype)
    w.ff1_b[:4] = torch.tensor([3e38, 1e20, -1e20, -3e38])
    w.ff2_w = torch.eye(E, 2 * E).roll(0, 1).to(dtype) + torch.eye(2 * E)[E:].to(dtype)
    w.ff2_w[:, :4] = 0  # the four extremes meet zero weights: finite results
    w.ff2_b = torch.zeros_like(w.ff2_b)
    x = torch.randn(40, E, generator=g).to(dtype)
    a = torch.zeros_like(x)
    out = Q._layer_tail(a.to(dev), x.to(dev), to_device(w, dev))
    torch.cuda.synchronize()
    _check(out, _tail64(a, x, w), dtype, "gelu range")


def test_route_conditions(dev):
    # what the kernels do not take keeps the general path: another activation, width, dtype mix, a gradient,
    # a misaligned weight view
    import dataclasses

    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(torch.float32, 1)
    wd = to_device(w, dev)
    x = torch.randn(10, E, generator=g).to(dev)
    assert Q._layer_native(x, wd, F.gelu)
    assert not Q._layer_native(x, wd, F.relu)
    assert not Q._layer_native(x.bfloat16(), wd, F.gelu)
    assert not Q._layer_native(x, dataclasses.replace(wd, ff1_w=wd.ff1_w[:200], ff1_b=wd.ff1_b[:200]), F.gelu)
    odd = torch.empty(E * E + 1, device=dev)[1:].view(E, E)
    assert not Q._layer_native(x, dataclasses.replace(wd, out_w=odd), F.gelu)
    grad = dataclasses.replace(wd, ff2_w=wd.ff2_w.clone().requires_grad_())
    assert not Q._layer_native(x, grad, F.gelu)
    with torch.no_grad():
        assert Q._layer_native(x, grad, F.gelu)


def test_biases_of_another_shape_keep_the_general_path(dev):
    # a bias of as many values in a column is torch's to refuse or to broadcast
    import dataclasses

    import tabicl_mi355_icl as icl
    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(torch.float32, 1)
    wd, wi = to_device(w, dev), to_device(block_weights(512, 1024, g, torch.bfloat16), dev)
    x, xi = torch.randn(10, E, device=dev), torch.randn(10, 512, device=dev)
    X, cw = torch.randn(2, 9, 5, device=dev), Q.ColumnWeights(torch.randn(E, 3, device=dev), torch.randn(E, device=dev), [])
    assert Q._layer_native(x, wd, F.gelu) and icl._linear_native(xi, wi, F.gelu) and Q._embed_native(X, None, cw, 3)
    for name in ("in_b", "out_b", "ff1_b", "ff2_b"):
        column = lambda blk: dataclasses.replace(blk, **{name: getattr(blk, name)[:, None]})  # noqa: E731
        assert not Q._layer_native(x, column(wd), F.gelu) and not icl._linear_native(xi, column(wi), F.gelu)
    assert not Q._embed_native(X, None, dataclasses.replace(cw, in_b=cw.in_b[:, None]), 3)


@pytest.mark.parametrize("rows,bias", [(1, True), (31, False), (32, True), (33, True), (480, True), (2001, False)])
def test_icl_linear_layers(dev, rows, bias):
    # the ICL block's fused linear layers against float64 on the same bf16 / fp32 inputs. Bars: bf16 results
    # (and bf16-rounded LN / GELU operands) 2e-2 x max |ref|; the fp32 residual form rounds nothing but its
    # inputs: 1e-4, 1e-3 x max |ref| and 2e-6 in the 2-norm.
    import tabicl_mi355_icl as icl
    g = torch.Generator().manual_seed(rows)
    w = block_weights(512, 1024, g, torch.bfloat16)
    x = torch.randn(rows, 512, generator=g) * 2 + 0.3
    bq, b1, bo, b2 = (w.in_b[:512], w.ff1_b, w.out_b, w.ff2_b) if bias else (None,) * 4
    a, h = torch.randn(rows, 512, generator=g).bfloat16(), torch.randn(rows, 1024, generator=g).bfloat16()
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    print(f"[icl layer] rows={rows}", flush=True)
    n64 = F.layer_norm(x.double(), (512,), w.ln1_w.double(), w.ln1_b.double(), w.eps)
    for wt, b, gelu in ((w.in_w[:512], bq, False), (w.ff1_w, b1, True)):
        out = icl._ln_linear(d(x), d(w.ln1_w), d(w.ln1_b), w.eps, d(wt), d(b), gelu)
        torch.cuda.synchronize()
        ref = _lin64(n64, wt, b)
        _check(out, F.gelu(ref) if gelu else ref, torch.bfloat16, f"ln_linear gelu={gelu}")
    for src, wt, b in ((a, w.out_w, bo), (h, w.ff2_w, b2)):
        out = icl._linear_residual(d(src), d(wt), d(b), d(x))
        torch.cuda.synchronize()
        _check(out, x.double() + _lin64(src.double(), wt, b), torch.float32, f"linear_residual k={src.shape[1]}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,H,reserve", [(1, 1, 3, 4), (2, 17, 5, 4), (2, 300, 11, 0), (3, 256, 24, 4)])
def test_column_embed(dev, dtype, B, T, H, reserve):
    # against feature_grouping, the padding and the skippable linear run by torch; the same three products
    # and fp32 sums: fp32 2^-22 of the terms' scale, bf16 one rounding step
    import tabicl_mi355_query as Q
    g = torch.Generator().manual_seed(T + H)
    X = torch.randn(B, T, H, generator=g)
    X[0, 0] = -100.0  # every group of this row is skipped
    X[-1, -1, : H // 2] = -100.0
    rf = torch.tensor([H, max(1, H - 2), 1][:B])
    w = Q.ColumnWeights((torch.randn(E, 3, generator=g) * 0.5).to(dtype), (0.1 * torch.randn(E, generator=g)).to(dtype), [],
                        reserve_cls=reserve)
    wd = Q.ColumnWeights(w.in_w.to(dev), w.in_b.to(dev), [], reserve_cls=reserve)
    for real in (rf, None):
        rd = None if real is None else real.to(dev)
        assert Q._embed_native(X.to(dev), rd, wd, 3)
        print(f"[embed] {B} {T} {H} {dtype}", flush=True)
        out = Q._column_embed(X.to(dev), rd, wd)
        torch.cuda.synchronize()
        x = Q.feature_grouping(X, real, 3)
        x = F.pad(x, (0, 0, reserve, 0), value=-100.0).transpose(1, 2).to(dtype)
        ref = F.linear(x.double(), w.in_w.double(), w.in_b.double())
        skip = (x == -100.0).all(-1, keepdim=True)
        assert torch.equal(out.cpu()[skip.expand_as(ref)], torch.full((int(skip.sum()) * E,), -100.0, dtype=dtype))
        err = (out.cpu().double() - ref)[~skip.expand_as(ref)].abs().max() if (~skip).any() else torch.zeros(())
        scale = float((x.double().abs() @ w.in_w.double().abs().T)[~skip.expand_as(ref)].max()) if (~skip).any() else 1.0
        assert float(err) <= (2.0 ** -22 if dtype == torch.float32 else 2.0 ** -8) * max(1.0, scale)


def test_column_embed_bad_count(dev):
    # a count outside [1, H] names no features: NaN in that table's slots only
    import tabicl_mi355_query as Q
    X = torch.randn(3, 5, 4, device=dev)
    w = Q.ColumnWeights(torch.randn(E, 3, device=dev), None, [], reserve_cls=2)
    out = Q._column_embed(X, torch.tensor([0, 4, 5], device=dev), w).cpu()
    assert out[[0, 2], 2:].isnan().all() and out[1].isfinite().all() and (out[:, :2] == -100.0).all()


@pytest.mark.parametrize("amp", [torch.bfloat16, torch.float16])
def test_autocast_keeps_the_general_path(dev, amp):
    # autocast casts the operands of torch's linear layers; the layer kernels, launched on raw pointers,
    # would run in the tensors' own types and return another dtype
    import tabicl_mi355_icl as icl
    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(torch.float32, 3)
    wd = to_device(w, dev)
    wi = to_device(block_weights(512, 1024, g, torch.bfloat16), dev)
    x, xi = torch.randn(2, 9, E, generator=g).to(dev), torch.randn(9, 512, generator=g).to(dev)
    X, cw = torch.randn(2, 9, 5, device=dev), Q.ColumnWeights(torch.randn(E, 3, device=dev), None, [])
    on = lambda: (Q._layer_native(x, wd, F.gelu), icl._linear_native(xi, wi, F.gelu), Q._embed_native(X, None, cw, 3))  # noqa: E731
    assert on() == (True, True, True)
    with torch.autocast("cuda", dtype=amp):
        assert on() == (False, False, False)
        out = Q._after_attention(x, x, wd, F.gelu)
        assert torch.equal(out, Q._ffn(x, wd, F.gelu, F.linear(x, wd.out_w, wd.out_b)))
    assert on() == (True, True, True)


@pytest.mark.parametrize("ff,classes", [(1024, 10), (128, 3), (1000, 10)])
@pytest.mark.parametrize("lead", [(1, 1), (8, 60), (3, 33)])
def test_decoder(dev, lead, ff, classes):
    # decode on the fused LayerNorm + linear + GELU kernel (ff a multiple of 128) and on the general path
    # against float64 on the same weights. Operands rounded to bf16 (LN, GELU, logits): 2e-2 x max |ref|.
    import tabicl_mi355_icl as icl
    import tabicl_mi355_query as Q
    g = torch.Generator().manual_seed(ff + lead[1])
    mat = lambda o, i: (torch.randn(o, i, generator=g) * i ** -0.5).bfloat16()  # noqa: E731
    w = Q.DecoderWeights(1 + 0.1 * torch.randn(512, generator=g), 0.1 * torch.randn(512, generator=g), mat(ff, 512),
                         (0.1 * torch.randn(ff, generator=g)).bfloat16(), mat(classes, ff), None)
    x = torch.randn(*lead, 512, generator=g) * 2 + 0.3
    wd = Q.DecoderWeights(*(None if t is None else t.to(dev) for t in (w.ln_w, w.ln_b, w.w1, w.b1, w.w2, w.b2)))
    xd = x.to(dev)
    assert icl._ln_linear_native(xd, wd.ln_w, wd.ln_b, wd.eps, wd.w1, wd.b1) == (ff % 128 == 0)
    print(f"[decode] {lead} ff={ff}", flush=True)
    out = Q.decode(xd, wd)
    torch.cuda.synchronize()
    n64 = F.layer_norm(x.double(), (512,), w.ln_w.double(), w.ln_b.double(), w.eps)
    assert out.dtype == torch.float32 and out.shape == (*lead, classes)
    _check(out, _lin64(F.gelu(_lin64(n64, w.w1, w.b1)), w.w2, None), torch.bfloat16, f"decode {lead} {ff}")


@pytest.mark.parametrize("rows,bias", [(1, True), (33, False), (480, True), (2001, True)])
def test_icl_block_tail(dev, rows, bias):
    # the three launches in one call (the second residual in place) against the same three by themselves: the
    # same kernels on the same values, so the same bits
    import tabicl_mi355_icl as icl
    import tabicl_mi355_native as nat
    g = torch.Generator().manual_seed(rows)
    w = block_weights(512, 1024, g, torch.bfloat16)
    x = (torch.randn(rows, 512, generator=g) * 2 + 0.3).to(dev)
    a = torch.randn(rows, 512, generator=g).bfloat16().to(dev)
    d = lambda t: t.to(dev) if t.dim() == 2 or bias else None  # noqa: E731
    ow, ob, lb, w1, b1, w2, b2 = (d(t) for t in (w.out_w, w.out_b, w.ln2_b, w.ff1_w, w.ff1_b, w.ff2_w, w.ff2_b))
    lw, before = w.ln2_w.to(dev), x.clone()
    out, h = torch.empty_like(x), torch.empty(rows, 1024, dtype=torch.bfloat16, device=dev)
    print(f"[icl tail] rows={rows}", flush=True)
    nat.call("tabicl_icl_block_tail", a.data_ptr(), x.data_ptr(), ow.data_ptr(), nat.ptr(ob), lw.data_ptr(), nat.ptr(lb),
             w.eps, w1.data_ptr(), nat.ptr(b1), w2.data_ptr(), nat.ptr(b2), h.data_ptr(), out.data_ptr(), rows,
             nat.stream_of(x))
    x1 = icl._linear_residual(a, ow, ob, x)
    ref = icl._linear_residual(icl._ln_linear(x1, lw, lb, w.eps, w1, b1, True), w2, b2, x1)
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and torch.equal(x, before)
    with pytest.raises(nat.UnsupportedShapeError):
        nat.call("tabicl_icl_block_tail", a.data_ptr(), x.data_ptr(), ow.data_ptr(), nat.ptr(ob), lw.data_ptr(),
                 nat.ptr(lb), w.eps, w1.data_ptr(), nat.ptr(b1), w2.data_ptr(), nat.ptr(b2), h.data_ptr(), x.data_ptr(),
                 rows, nat.stream_of(x))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("value", [7.3, 99.9, 12345.678, 1e19])
def test_constant_rows(dev, dtype, value):
    # the LayerNorm of a constant row is its bias: the mean of equal values must be exact, or the rounding of the sum is
    # normalised to order 1 (deviations of 1e-3 against sqrt(eps) = 3e-3)
    import tabicl_mi355_icl as icl
    import tabicl_mi355_query as Q
    from query_ref import to_device
    w, g = _block(dtype, 9)
    w.out_b = torch.zeros_like(w.out_b)
    x = torch.randn(40, E, generator=g).to(dtype)
    x[3], x[39] = value, -value
    a, wd, xd = torch.zeros(40, E, dtype=dtype), to_device(w, dev), x.to(dev)
    ref = _lin64(_ln64(x, w.ln1_w, w.ln1_b, w.eps), w.in_w, w.in_b)
    _check(Q._layer_proj(xd, wd, 0, 3 * E), ref, dtype, "projection")
    if dtype == torch.float32:
        if value < 1e5:  # the feed-forward part, to the rounding of the sum that holds it (2^-24 of 1.2e4: 7e-4)
            out, ref = Q._layer_tail(a.to(dev), xd, wd).cpu(), _tail64(a, x, w)
            assert float((out.double() - ref)[[3, 39]].abs().max()) <= 1.5e-3
        wi = block_weights(512, 1024, g, torch.bfloat16)
        xi = torch.randn(40, 512, generator=g)
        xi[3], xi[39] = value, -value
        d = to_device(wi, dev)
        n64 = F.layer_norm(xi.double(), (512,), wi.ln1_w.double(), wi.ln1_b.double(), wi.eps)
        out = icl._ln_linear(xi.to(dev), d.ln1_w, d.ln1_b, d.eps, d.in_w, d.in_b, False)
        _check(out, _lin64(n64, wi.in_w, wi.in_b), torch.bfloat16, "ln_linear")
