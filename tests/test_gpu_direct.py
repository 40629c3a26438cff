"""The wrappers' direct launches (tabicl_mi355_native.direct): taken for plain GPU tensors, left to the
torch.library op wherever something watches or transforms op calls, with the same bits either way."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


class _Seen(TorchDispatchMode):
    """Records the op calls it sees."""

    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _calls(dev):
    import tabicl_mi355_attn as pk
    import tabicl_mi355_icl as icl
    from query_ref import Rope
    g = torch.Generator(device=dev).manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    q, kv, qkv, x, ind = r(3, 40, 128), r(3, 200, 256), r(3, 24, 384), r(3, 300, 128), r(16, 128)
    kb = torch.zeros(24, device=dev)
    kb[20:] = -1e30
    iq, ik, iv = r(2, 8, 30, 64), r(2, 8, 100, 64), r(2, 8, 100, 64)
    rope = Rope()
    valid = torch.tensor(150, device=dev)
    return {
        "hx_fwd": lambda: pk.hx_attention(q, kv[..., :128], kv[..., 128:], 8),
        "hxq_fwd": lambda: pk.hxq_attention(q, kv, valid, 8),
        "pk_self_fwd": lambda: pk.pk_self_attention(qkv, 8, kb, rope, 0.25),
        "pk_cross_fwd": lambda: pk.pk_cross_attention(q, kv, 8, None, None, 0.25),
        "hxf_fwd": lambda: pk.hxf_attention(ind, x, 250),
        "icl_cached_attn": lambda: icl.icl_sdpa(iq, ik, iv, 90),
    }


def test_direct_equals_op_and_modes_see_the_op(dev):
    for name, call in _calls(dev).items():
        print(f"[direct] {name}", flush=True)
        out = call()
        with _Seen() as seen:
            want = call()
        torch.cuda.synchronize()
        assert any(name in n for n in seen.names), (name, seen.names)
        assert torch.equal(out, want), name


def test_direct_conditions(dev):
    import tabicl_mi355_native as nat
    t = torch.zeros(2, device=dev)
    w = torch.zeros(2, device=dev, requires_grad=True)
    assert nat.direct(t, None)
    assert not nat.direct(t, w)
    assert not nat.direct(t, torch.zeros(2))
    with torch.no_grad():
        assert nat.direct(t, w)
    seen = []
    torch.func.vmap(lambda a: (seen.append(nat.direct(a)), a)[1])(t)
    torch.func.grad(lambda a: (seen.append(nat.direct(a)), a.sum())[1])(t)
    with torch.autograd.forward_ad.dual_level():
        seen.append(nat.direct(t))
    with torch.device("cuda"):  # a function mode
        seen.append(nat.direct(t))
    torch.jit.trace(lambda a: (seen.append(nat.direct(a)), a + 1)[1], t, check_trace=False)
    assert seen and not any(seen), seen
    assert nat.direct(t)


def test_query_out_bumps_version(dev):
    # the direct launch writes `out` as the op does: autograd's version check sees it
    import tabicl_mi355_icl as icl
    cache = icl.IclKVCache(1, 1, 8, 64, 64, torch.bfloat16, dev)
    k = torch.randn(1, 8, 64, 64, device=dev).to(torch.bfloat16)
    cache.append(0, k, k)
    out = torch.empty(1, 8, 10, 64, dtype=torch.bfloat16, device=dev)
    v0 = out._version
    with torch.no_grad():
        cache.query(0, k[:, :, :10], out=out)
    torch.cuda.synchronize()
    assert out._version > v0
