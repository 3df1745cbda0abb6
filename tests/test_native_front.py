"""The native front of the step-wise operators: it answers None to every form it does not take, and what it takes comes
out as on the general way, bit for bit."""
import sys

import pytest
import torch

import neuralattentionsearch_amd
from neuralattentionsearch_amd import ops
from tests.gpu_util import say


class NoFront:
    """The general way: every operator of the front declines."""

    def __init__(self, front):
        self.front = front

    def __getattr__(self, name):
        if name in ("cache_append", "evict_plan", "evict_apply_inplace", "matvec_takes"):
            return getattr(self.front, name)
        return lambda *a: None


def test_declines_what_is_not_plain():
    t = torch.zeros(1, 2, 1, 32)  # (not on a GPU)
    v = torch.zeros(1, 2, 8, dtype=torch.uint8)
    f = ops._front
    assert f.decode(t, t, t, v, 1, None, None, None) is None
    assert f.decode(None, 1, "x", t, 1.5, None, None, None) is None
    assert f.decode(t) is None
    assert f.prefill(t, t, t, v, 8, 8, None) is None
    assert f.roles_from_logits(t, 0.1, True, False, True) is None
    assert f.rope_append(*[t] * 7, v, None, 0, 0, -1) is None
    assert f.matvec(t, t, False) is None
    assert f.matvec_takes(t, t, 32) is False
    assert f.step_project(t, (t,), 1, None, True, None, None, 0.1, False) is None
    assert f.step_project(t, [t], 1, None, True, None, None, 0.1, False) is None
    with pytest.raises(TypeError):
        f.cache_append(1, 2)
    with pytest.raises(ValueError):  # (and the operator says why)
        ops.decode_attention(t, t, t, v, 1)


def both(monkeypatch, call, taken=True):
    """The results of `call` with the front and on the general way; `taken`: the front has answered all its calls, or none."""
    real, answers = ops._front, []

    class Watched:
        def __getattr__(self, name):
            return lambda *a: answers.append(getattr(real, name)(*a)) or answers[-1]

    with monkeypatch.context() as m:
        m.setattr(ops, "_front", Watched())
        got = call()
    assert answers and all((a is not None) == taken for a in answers)
    with monkeypatch.context() as m:
        m.setattr(ops, "_front", NoFront(ops._front))
        want = call()
    return got, want


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layout", ["plain", "strided", "single"])
def test_equals_the_general_way(dtype, layout, monkeypatch):
    say("native front", dtype, layout)
    g = torch.Generator(device="cuda").manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    B, Hq, Hkv, D, N = (1, 4, 1, 64, 300) if layout == "single" else (3, 8, 4, 64, 300)
    taken = []
    real = ops._front.decode

    # decode: caches that are slices of larger buffers, bool and uint8 valid rows, q that is a transposed view
    k, v = (rn(B, Hkv, N + 84, D)[:, :, :N + 20] if layout == "strided" else rn(B, Hkv, N, D) for _ in range(2))
    valid = torch.rand(B, Hkv, k.shape[2], generator=g, device="cuda") < 0.7
    q = rn(B, 1, Hq, D).transpose(1, 2) if layout == "strided" else rn(B, Hq, 1, D)
    end = torch.full((B, Hkv), 200, device="cuda")
    for args in ((q, k, v, valid, N), (q, k, v, valid.to(torch.uint8), N - 7, 0.3), (q, k, v, valid, N, None, end, 290),
                 (q, k, v, valid, N, None, end.t().contiguous().t(), 290)):
        plain = len(args) < 7 or args[6].is_contiguous()
        a, b = both(monkeypatch, lambda: ops.decode_attention(*args), taken=plain)
        assert a.shape == b.shape == (B, Hq, 1, D) and torch.equal(a, b)
    # prefill and roles
    L, C, W = 77, 16, 32
    logits = rn(B, -(-L // C), Hkv, 3)
    if layout == "strided":
        logits = rn(B, Hkv, -(-L // C), 3).transpose(1, 2)
    (r1, h1), (r2, h2) = both(monkeypatch, lambda: ops.roles_from_logits(logits, 0.1, True, True), taken=logits.is_contiguous())
    assert torch.equal(r1, r2) and torch.equal(h1, h2) and ops.roles_from_one_hot(h1) is r1
    pq, pk, pv = ((rn(B, L, h, D).transpose(1, 2) if layout == "strided" else rn(B, h, L, D)) for h in (Hq, Hkv, Hkv))
    a, b = both(monkeypatch, lambda: ops.prefill_attention(pq, pk, pv, r1, C, W, 0.2))
    assert torch.equal(a, b)
    # rotary embedding with the append
    cos, sin = rn(B, 1, D), rn(B, 1, D)
    qkv = rn(B, 1, Hq + 2 * Hkv, D).transpose(1, 2)

    def append():
        ck, cv = torch.zeros(B, Hkv, 16, D, dtype=dtype, device="cuda"), torch.zeros(B, Hkv, 16, D, dtype=dtype, device="cuda")
        val, pos = torch.ones(B, Hkv, 16, dtype=torch.uint8, device="cuda"), torch.zeros(B, Hkv, 16, dtype=torch.int32, device="cuda")
        out = ops.rope_append(qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:], cos, sin, ck, cv, val, pos, 5, 9, 2)
        return torch.cat([t.flatten().double() for t in (out, ck, cv, val, pos)])

    a, b = both(monkeypatch, append)
    assert torch.equal(a, b)
    # rows and matrices
    x, w = rn(B, 1, 256), torch.nn.Parameter(rn(64, 256), requires_grad=False)
    for gate in (False, True):
        a, b = both(monkeypatch, lambda: ops.matvec(x, w, gate))
        assert torch.equal(a, b)

    # a call with new scratch needs takes the operator's own table
    monkeypatch.setattr(ops._front, "decode", lambda *a: taken.append(real(*a)) or taken[-1], raising=False)
    ops._workspaces.clear()
    ops.decode_attention(rn(B, Hq, 1, D), k, v, valid, N)
    assert taken[-1] is not None and len(ops._workspaces) == 1


@pytest.fixture
def without(monkeypatch):
    """The package as it is where _nats_host.so has not been built, or was built for another torch."""
    def take_away(how):
        if how == "missing":
            monkeypatch.delattr(neuralattentionsearch_amd, "_nats_host", raising=False)
            monkeypatch.setitem(sys.modules, "neuralattentionsearch_amd._nats_host", None)
        else:
            from neuralattentionsearch_amd import _nats_host
            monkeypatch.setattr(_nats_host, "built_for", "0.0")
        monkeypatch.setattr(ops, "_front", ops._NativeFront())
    return take_away


@pytest.mark.parametrize("how", ["missing", "other torch"])
def test_without_the_native_front_operators_go_the_general_way(without, how):
    without(how)
    t, v = torch.zeros(1, 2, 1, 32), torch.zeros(1, 2, 8, dtype=torch.uint8)
    with pytest.warns(RuntimeWarning, match="native front"):
        assert ops._front.decode(t, t, t, v, 1, None, None, None) is None
    with pytest.raises(ValueError, match="CPU tensor"):
        ops.decode_attention(t, t, t, v, 1)
    with pytest.raises(ValueError, match="CPU tensor"):
        ops.prefill_attention(t, t, t, v, 8, 8)
    assert ops.matvec_takes(t, t[0, 0], 32) is False
    assert ops._front.cache_append(*[None] * 6, *[0] * 7, *[None] * 4, 0, None) < 0  # (the library's error code)
    assert ops._front.cache_append(*[None] * 6, *[0] * 7, *[None] * 4, 0, *[None] * 5, 0, None, None, None) < 0
    assert ops._front.evict_plan(*[None] * 5, 0, None, None, None) < 0
    assert ops._front.evict_apply_inplace(*[None] * 10, 0, None, None, None) < 0
    with pytest.raises(AttributeError):
        ops._front.no_such_function


def test_without_the_library_arguments_are_checked_first(monkeypatch):
    from neuralattentionsearch_amd import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libnats_hip.so")
    monkeypatch.setattr(ops, "_front", ops._NativeFront())
    t, v = torch.zeros(1, 2, 1, 32), torch.zeros(1, 2, 8, dtype=torch.uint8)
    with pytest.raises(ValueError, match="CPU tensor"):
        ops.decode_attention(t, t, t, v, 1)
    with pytest.raises(ImportError, match="build it"):
        ops._front.cache_append()


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:the native front")
def test_without_the_native_front_everything_runs(without):
    """A layer's conversation (prompt, one-token steps, segment, streamed evictions) and a cache filled piece by piece."""
    from neuralattentionsearch_amd.attention import LlamaNAtSChunkAttentionLayer
    from neuralattentionsearch_amd.cache import NAtSCache, NAtSChunkLayerCache
    from neuralattentionsearch_amd.llama import rotary_tables
    say("without the native front")
    torch.manual_seed(5)
    mod = LlamaNAtSChunkAttentionLayer(dim=256, n_heads=4, n_kv_heads=2, chunk_size=8, local_seq_max_length=16)
    mod = mod.cuda().bfloat16().eval().requires_grad_(False)
    x = torch.randn(1, 60, 256, device="cuda").bfloat16()
    k, v = (torch.randn(2, 4, 96, 64, device="cuda").bfloat16() for _ in range(2))
    roles = torch.randint(0, 3, (2, 4, 12), device="cuda", dtype=torch.uint8)
    roles[:, :, 0] = 0

    def run():
        outs, at, cache = [], 0, NAtSCache(16, 8)
        for n in [20] + [1] * 18 + [13] + [1] * 9:
            emb = rotary_tables(torch.arange(at, at + n, device="cuda")[None], 64, 10000.0, torch.bfloat16)
            with torch.no_grad():
                outs.append(mod(x[:, at:at + n], emb, None, start_pos=at, cache=cache))
            at += n
        layer = NAtSChunkLayerCache(2, 4, 16, chunk_size=8, device="cuda", track_positions=True)
        for i in range(12):
            layer.update(k[:, :, 8 * i:8 * i + 8], v[:, :, 8 * i:8 * i + 8], None, roles=roles[:, :, i:i + 1])
            layer.post_update(8)
        return torch.cat(outs, dim=1), [layer.cache_k, layer.cache_v, layer.valid_tokens, layer.token_positions]

    want, rows = run()
    without("missing")
    got, got_rows = run()
    # (the products of a one-token step sum in another order: one rounding to bf16, carried through the layer)
    assert ((got - want).float().norm() / want.float().norm()).item() <= 4 * 2.0 ** -8
    assert all(torch.equal(a, b) for a, b in zip(got_rows, rows))
