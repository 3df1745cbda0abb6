"""GPU: the one-launch projections, chunk statistic and roles of a one-token step, and the attention modules' one-token
path that is built on them, against the separate torch ops."""
import pytest
import torch

from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,k,ns,H,C,hs", [(1, 4096, (4096, 1024, 1024), 8, 64, 1), (4, 512, (129, 3, 70, 1), 5, 12, 16),
                                              (3, 8, (1,), 1, 1, 16), (2, 2056, (4, 5), 2, 16, 1)])
def test_step_project(dtype, rows, k, ns, H, C, hs):
    from neuralattentionsearch_amd import ops
    say("step_project", dtype, rows, k, ns, H, C, hs)
    g = torch.Generator().manual_seed(rows * k)
    x = torch.randn(rows, 1, k, generator=g).to(dtype).cuda()
    w = [(torch.randn(n, k, generator=g) / k ** 0.5).to(dtype).cuda() for n in ns]
    wr = (torch.randn(3 * H, k, generator=g) * (C / k) ** 0.5).to(dtype).cuda()
    carry = torch.randn(rows, 1, k, generator=g).to(dtype).cuda()
    for c_in in (None, carry):
        buf = torch.full((rows, H, hs), 7, dtype=torch.uint8, device="cuda")
        y, stat = ops.step_project(x, w, C, c_in, with_carry=True, role_weight=wr, roles_out=buf[:, :, :1])
        # elementwise steps equal the torch ops bit for bit (components/cache/dyn_cache.py:101-104)
        want = x / C if c_in is None else c_in + x / C
        assert torch.equal(stat, want)
        # products: fp32 sums in another order, one rounding (2^-8 of the value in bf16) at the end
        exact = torch.cat([x.double() @ m.double().T for m in w], dim=-1)
        err = ((y.double() - exact).abs() / exact.abs().clamp_min(1.0)).max().item()
        assert err <= (2.0 ** -8 if dtype == torch.bfloat16 else 2e-6), err
        # roles: the argmax of the rounded logits, wherever no logit of the sums in 64 bits is that close to another
        lg = (want.double() @ wr.double().T).view(rows, H, 3)
        ulp = (lg.abs().max().item() + 0.2) * (2.0 ** -7 if dtype == torch.bfloat16 else 2e-6)
        lg[..., 0] += 0.1
        top = lg.topk(2, dim=-1).values
        sure = top[..., 0] - top[..., 1] > 2 * ulp
        assert torch.equal(buf[:, :, 0][sure], lg.argmax(-1).to(torch.uint8)[sure])
        assert bool((buf[:, :, 1:] == 7).all())
    roles = torch.empty(rows, H, 1, dtype=torch.uint8, device="cuda")
    y2, none = ops.step_project(x, w, C, role_weight=wr, roles_out=roles, force_first_global=True)
    assert none is None and torch.equal(y2, y) and not roles.any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,C,W,lens", [(1, 16, 32, [50] + [1] * 40 + [20] + [1] * 20), (4, 1, 32, [40] + [1] * 40 + [7] + [1] * 9),
                                        (2, 12, 36, [5] + [1] * 30), (3, 1, 16, [1] * 40)])
def test_module_step_equals_the_general_way(dtype, B, C, W, lens):
    """The fast step and the general forward (forced by a hook) on the same hidden states: the same roles and rows."""
    from neuralattentionsearch_amd.attention import LlamaNAtSAttentionLayer, LlamaNAtSChunkAttentionLayer
    from neuralattentionsearch_amd.cache import NAtSCache
    from neuralattentionsearch_amd.llama import rotary_tables
    say("module step", dtype, B, C, W)
    torch.manual_seed(3)
    kw = dict(dim=512, n_heads=8, n_kv_heads=4, layer_id=0, local_seq_max_length=W)
    mod = LlamaNAtSAttentionLayer(**kw) if C == 1 else LlamaNAtSChunkAttentionLayer(chunk_size=C, **kw)
    mod = mod.cuda().to(dtype).eval().requires_grad_(False)
    mod.proj_layer.weight.mul_(8.0)
    fast, slow = NAtSCache(W, C), NAtSCache(W, C)
    taken = []
    general = type(mod)._one_token_step
    at = 0
    tol = 4 * 2.0 ** -8 if dtype == torch.bfloat16 else 2e-5
    with torch.no_grad():
        for n in lens:
            x = torch.randn(B, n, 512, device="cuda").to(dtype)
            pos = torch.arange(at, at + n, device="cuda")[None].expand(B, -1)
            emb = rotary_tables(pos, 64, 10000.0, dtype)
            if n == 1:
                taken.append(general(mod, x, emb, at, None) is None)  # (no cache: the general way)
            got = mod(x, emb, None, start_pos=at, cache=fast)
            hook = mod.wv.register_forward_hook(lambda m, i, o: None)
            want = mod(x, emb, None, start_pos=at, cache=slow)
            hook.remove()
            at += n
            err = ((got - want).float().norm() / want.float().norm()).item()
            assert err <= tol, (at, err)
            a, b = fast.cache_model[0], slow.cache_model[0]
            assert a.n_ctx_data == b.n_ctx_data and torch.equal(a.valid_tokens, b.valid_tokens), at
            assert torch.equal(a.size_global_kv, b.size_global_kv) and torch.equal(a.size_local_kv, b.size_local_kv), at
    assert all(taken)


def test_module_step_leaves_watched_modules_to_the_general_way():
    """Hooks, wrapped projections, autograd and overridden methods see every call."""
    from neuralattentionsearch_amd.attention import LlamaNAtSChunkAttentionLayer
    from neuralattentionsearch_amd.cache import NAtSCache
    from neuralattentionsearch_amd.llama import rotary_tables

    class Scaled(LlamaNAtSChunkAttentionLayer):
        calls = 0

        def add_rotary_emb(self, xq, xk, pos_emb):
            Scaled.calls += 1
            return super().add_rotary_emb(xq, xk, pos_emb)

    kw = dict(dim=256, n_heads=4, n_kv_heads=2, layer_id=0, local_seq_max_length=16, chunk_size=8)
    x = torch.randn(1, 1, 256, device="cuda")

    def step(mod):
        cache = NAtSCache(16, 8)
        with torch.no_grad():
            emb = rotary_tables(torch.arange(20, device="cuda")[None], 64, 10000.0, torch.float32)
            mod(torch.randn(1, 20, 256, device="cuda"), emb, None, start_pos=0, cache=cache)
        emb = rotary_tables(torch.full((1, 1), 20, device="cuda"), 64, 10000.0, torch.float32)
        return mod._one_token_step(x, emb, 20, cache), cache, emb

    mod = LlamaNAtSChunkAttentionLayer(**kw).cuda().eval()
    assert step(mod)[0] is None  # (autograd records the projections)
    mod.requires_grad_(False)
    out, cache, emb = step(mod)
    assert out is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert mod._one_token_step(x, emb, 21, cache) is None
    assert step(Scaled(**kw).cuda().eval().requires_grad_(False))[0] is None
    mod.wo.register_forward_hook(lambda m, i, o: o)
    assert step(mod)[0] is None


@pytest.mark.parametrize("C", [1, 8])
@pytest.mark.parametrize("where", ["class", "instance", "subclass"])
def test_model_step_calls_a_replaced_append(C, where, monkeypatch):
    """`append_rotated` of a layer cache is the hand-over of the model's one-token step, also where it is replaced."""
    from neuralattentionsearch_amd import cache as cm
    from neuralattentionsearch_amd.llama import NAtSLlamaConfig, NAtSLlamaForCausalLM
    say("model step, replaced append", C, where)
    cfg = NAtSLlamaConfig(vocab_size=64, hidden_size=128, intermediate_size=128, num_hidden_layers=2, num_attention_heads=4,
                          num_key_value_heads=2, chunk_size=C, local_seq_max_length=16, fused_role_step=True)
    model = NAtSLlamaForCausalLM.random_init(cfg, device="cuda", dtype=torch.bfloat16, seed=1)
    ids = torch.randint(0, 64, (1, 24), generator=torch.Generator().manual_seed(2)).cuda()
    cls = cm.NAtSLayerCache if C == 1 else cm.NAtSChunkLayerCache

    def run(replace):
        cache = model.new_cache()
        out = [model(ids[:, :20], 0, cache)]
        if replace:
            replace(cache)
        out += [model(ids[:, i:i + 1], i, cache) for i in range(20, 24)]
        return torch.stack(out, dim=1)

    want = run(None)
    calls = []

    class Counting(cls):
        def append_rotated(self, *a, **kw):
            calls.append(1)
            return super().append_rotated(*a, **kw)

    def replace(cache):
        layer = cache.cache_model[0]
        if where == "subclass":
            layer.__class__ = Counting
        elif where == "instance":
            old = layer.append_rotated
            layer.append_rotated = lambda *a, **kw: calls.append(1) or old(*a, **kw)
        else:
            old_fn = cls.append_rotated
            monkeypatch.setattr(cls, "append_rotated", lambda *a, **kw: calls.append(1) or old_fn(*a, **kw))

    got = run(replace)
    assert len(calls) == (8 if where == "class" else 4)
    assert torch.equal(got, want)


@pytest.mark.parametrize("name", ["rotate_half", "apply_rotary_pos_emb"])
def test_segment_calls_a_replaced_rotary_embedding(name, monkeypatch):
    """The rotary functions of the module, replaced by a program, rotate a segment of several tokens."""
    from neuralattentionsearch_amd import attention
    from neuralattentionsearch_amd.llama import rotary_tables
    say("segment, replaced rotary embedding", name)
    mod = attention.LlamaNAtSAttentionLayer(dim=256, n_heads=4, n_kv_heads=2).cuda().eval().requires_grad_(False)
    q, k = torch.randn(1, 4, 20, 64, device="cuda"), torch.randn(1, 2, 20, 64, device="cuda")
    emb = rotary_tables(torch.arange(20, device="cuda")[None], 64, 10000.0, torch.float32)
    want = mod.add_rotary_emb(q, k, emb)
    calls, old = [], getattr(attention, name)
    monkeypatch.setattr(attention, name, lambda *a, **kw: calls.append(1) or old(*a, **kw))
    got = mod.add_rotary_emb(q, k, emb)
    assert calls and all(torch.equal(a, b) for a, b in zip(got, want))


def _targets():
    from neuralattentionsearch_amd import attention, cache, ops
    base, chunk = attention.BaseNAtSAttentionLayer, attention.BaseNAtSChunkAttentionLayer
    return {"prepare_x_values": base, "prepare_kv": base, "multi_head_attention": base, "role_logits": base,
            "_sample_for_token_info_values_inference": chunk, "add_rotary_emb": attention.AttentionLayer,
            "repeat_kv_values": attention.AttentionLayer, "apply_rotary_pos_emb": attention, "rotate_half": attention,
            "NAtSCache.update": cache.NAtSCache, "update_nats_cached_x_in_chunk": cache.NAtSCache,
            "update_nats_cached_x_across_chunk": cache.NAtSCache, "merge_new_x_values_in_chunk": cache.NAtSCache,
            "NAtSChunkLayerCache.update": cache.NAtSChunkLayerCache, "valid_tokens": cache.NAtSChunkLayerCache,
            "roles_from_logits": ops, "roles_from_one_hot": ops, "Linear.forward": torch.nn.Linear,
            "linear": torch.nn.functional, "Module.__call__": torch.nn.Module}


def _counted(owner, name, monkeypatch):
    """Replaces owner.name by one that counts its calls."""
    calls = []
    name = name.split(".")[-1]
    old = owner.__dict__[name] if isinstance(owner, type) else getattr(owner, name)
    if isinstance(old, property):
        new = property(lambda self: calls.append(1) or old.fget(self))
    elif isinstance(old, staticmethod):
        new = staticmethod(lambda *a, **kw: calls.append(1) or old.__func__(*a, **kw))
    else:
        def new(*a, **kw):
            calls.append(1)
            return old(*a, **kw)
    monkeypatch.setattr(owner, name, new)
    return calls


@pytest.mark.parametrize("name", list(_targets()))
@pytest.mark.parametrize("where", ["class", "instance"])
def test_module_step_calls_what_was_replaced(name, where, monkeypatch):
    """A method, a function or a cache update that a program replaces is called by one-token steps as by any other."""
    from neuralattentionsearch_amd.attention import LlamaNAtSChunkAttentionLayer
    from neuralattentionsearch_amd.cache import NAtSCache
    from neuralattentionsearch_amd.llama import rotary_tables
    say("module step, replaced", name, where)
    owner = _targets()[name]
    kw = dict(dim=256, n_heads=4, n_kv_heads=2, layer_id=0, local_seq_max_length=16, chunk_size=8)
    mod = LlamaNAtSChunkAttentionLayer(**kw).cuda().eval().requires_grad_(False)
    cache = NAtSCache(16, 8)
    calls, at = None, 0
    for n in [20] + [1] * 9:  # (through the open chunk and the step that completes it)
        if n == 1 and calls is None:
            if where == "instance":
                short = name.split(".")[-1]
                owner = next((o for o in (mod, cache, cache.cache_model[0]) if isinstance(owner, type) and isinstance(o, owner)), None)
                if owner is None or short in ("valid_tokens", "__call__", "forward", "merge_new_x_values_in_chunk"):
                    pytest.skip("nothing that an instance can replace")
                calls, old = [], getattr(owner, short)
                monkeypatch.setattr(owner, short, lambda *a, _old=old, **kws: calls.append(1) or _old(*a, **kws), raising=False)
            else:
                calls = _counted(owner, name, monkeypatch)
        emb = rotary_tables(torch.arange(at, at + n, device="cuda")[None], 64, 10000.0, torch.float32)
        with torch.no_grad():
            mod(torch.randn(1, n, 256, device="cuda"), emb, None, start_pos=at, cache=cache)
        at += n
    assert len(calls) > (9 if name == "Module.__call__" else 0), name  # (9: the module itself)
