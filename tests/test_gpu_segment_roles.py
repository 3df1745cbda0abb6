"""The role step of a multi-token segment in one launch (attention modules) against the torch ops it stands in for: roles, the
statistic of the open chunk, and the general way wherever something of it is replaced.

The statistic is the same ops with the same rounding points and a power-of-two divisor; only the order of its fp32 sums may
differ (bf16: one unit in the last place, 2^-8 of the value; fp32: 64 terms of 6e-8).  Roles are compared where the best two logits
of the general way differ by more than the two products can (bf16 logits of order one: 2^-6)."""
import pytest
import torch

from neuralattentionsearch_amd import ops
from neuralattentionsearch_amd.attention import LlamaNAtSChunkAttentionLayer
from neuralattentionsearch_amd.cache import NAtSCache
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


def build(dtype, dim, C, seed=0):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        m = LlamaNAtSChunkAttentionLayer(dim=dim, n_heads=8, n_kv_heads=4, layer_id=0, local_seq_max_length=2 * C, chunk_size=C)
    return m.to(dtype).eval().requires_grad_(False)


def roles_of(m, x, fill, general, monkeypatch, heads=4):
    """One hot roles and carry of a segment behind `fill` tokens of an open chunk; which way it went."""
    C = m.chunk_size
    cache = NAtSCache(2 * C, C)
    calls = []
    role_step = ops.role_step
    with monkeypatch.context() as mp:
        mp.setattr(ops, "role_step", lambda *a, **k: calls.append(1) or role_step(*a, **k))
        if general:
            mp.setattr(LlamaNAtSChunkAttentionLayer, "_segment_roles", lambda *a: None)
        with torch.no_grad():
            if fill:
                k = torch.zeros(x.shape[0], heads, fill, m.head_dim, device="cuda", dtype=x.dtype)
                m._sample_for_token_info_values_inference(x[:, :fill], 0, cache)
                cache.update(k, k, 0, {"token_states_info": m.one_hot_values.to(x).reshape(1, 1, 1, -1).expand(x.shape[0], heads, 1, -1)})
                cache.post_update(0, fill)
            out = m._sample_for_token_info_values_inference(x[:, fill:], fill, cache)
    return out, cache.get_nats_cached_x_in_chunk(0), bool(calls)


@pytest.mark.parametrize("dtype,dim,C,B,fill,L", [
    (torch.bfloat16, 1024, 64, 2, 0, 64), (torch.bfloat16, 4096, 64, 1, 13, 301), (torch.bfloat16, 512, 8, 3, 5, 3),
    (torch.bfloat16, 72, 16, 2, 15, 1 + 16 * 40), (torch.float32, 1000, 32, 2, 31, 70), (torch.float32, 64, 128, 1, 0, 129),
])
def test_agrees_with_the_torch_ops(monkeypatch, dtype, dim, C, B, fill, L):
    say("segment roles", dtype, dim, C, B, fill, L)
    m = build(dtype, dim, C)
    x = torch.randn(B, fill + L, dim, device="cuda", dtype=dtype)
    got, carry, fused = roles_of(m, x, fill, False, monkeypatch)
    want, carry_want, general = roles_of(m, x, fill, True, monkeypatch)
    assert fused and not general
    assert got.dtype == want.dtype and got.shape == want.shape and got.device == want.device
    assert torch.equal(ops.roles_from_one_hot(got), got.argmax(-1).to(torch.uint8))
    pooled = torch.nn.functional.pad(x.float(), (0, 0, 0, -(fill + L) % C)).unflatten(1, (-1, C)).mean(2)
    top = (m.proj_layer.weight.float() @ pooled.transpose(1, 2)).transpose(1, 2).unflatten(-1, (4, 3))
    top = (top + torch.tensor([0.1, 0.0, 0.0], device="cuda")).topk(2, dim=-1).values
    clear = (top[..., 0] - top[..., 1] > 2 ** -6).transpose(1, 2)
    assert torch.equal(got.argmax(-1)[clear], want.argmax(-1)[clear])
    assert (carry is None) == (carry_want is None)
    if carry is not None:
        assert carry.shape == carry_want.shape
        tol = 2 ** -8 if dtype == torch.bfloat16 else 64 * 6e-8
        assert ((carry.float() - carry_want.float()).abs() <= tol * carry_want.float().abs().clamp_min(2 ** -6)).all()


@pytest.mark.parametrize("dtype,dim,heads,C,B,L,shift,fused", [
    (torch.bfloat16, 1024, 32, 8, 1, 8 * 32, 0, True), (torch.bfloat16, 4096, 32, 32, 1, 32 * 30, 0, False),    # up to 32 chunks
    (torch.bfloat16, 4096, 8, 8, 3, 8 * 11, 0, True), (torch.bfloat16, 4096, 32, 8, 3, 8 * 11, 0, False),       # 33 chunks
    (torch.bfloat16, 4096, 8, 8, 1, 8 * 600, 0, True), (torch.bfloat16, 4096, 32, 8, 1, 8 * 600, 0, False),     # many
    (torch.float32, 4096, 16, 8, 1, 8 * 300, 0, True), (torch.float32, 4096, 32, 8, 1, 8 * 300, 0, False),
    (torch.bfloat16, 1024, 8, 8, 1, 100, 1, False), (torch.float32, 1024, 8, 8, 1, 100, 1, False),              # rows off 16 bytes
    (torch.bfloat16, 1028, 4, 8, 1, 100, 0, False),
])
def test_where_the_kernel_pays(monkeypatch, dtype, dim, heads, C, B, L, shift, fused):
    say("segment roles pay", dtype, dim, heads, C, B, L, shift)
    with torch.device("cuda"):
        m = LlamaNAtSChunkAttentionLayer(dim=dim, n_heads=heads, n_kv_heads=heads, layer_id=0, local_seq_max_length=2 * C, chunk_size=C)
    m = m.to(dtype).eval().requires_grad_(False)
    x = torch.randn(B * L * dim + shift, device="cuda", dtype=dtype)[shift:].view(B, L, dim)
    got, _, went = roles_of(m, x, 0, False, monkeypatch, heads)
    assert went == fused and got.shape == (B, heads, -(-L // C), 3)


@pytest.mark.parametrize("C", [8, 64, 512])
@pytest.mark.parametrize("offset", [0.0, 1.0])
def test_fp32_statistic_is_no_further_from_the_exact_one(monkeypatch, C, offset):
    """The open chunk's mean against 64 bits, as a share of what the torch ops are off by: one rounding of an fp64 sum is at most
    2^-24 and 3.5e-8 in the mean over normal values, which any fp32 sum ends with as well."""
    say("fp32 statistic", C, offset)
    m = build(torch.float32, 1024, C)
    torch.manual_seed(C)
    x = torch.randn(2, 3 * C - 1, 1024, device="cuda") + offset
    exact = x[:, 2 * C:].double().sum(1, keepdim=True) / C
    _, got, fused = roles_of(m, x, 0, False, monkeypatch)
    _, want, general = roles_of(m, x, 0, True, monkeypatch)
    assert fused and not general
    off = [((c.double() - exact).norm() / exact.norm()).item() for c in (got, want)]
    assert off[0] <= 1.01 * off[1]  # (1 %: where both are the rounding alone)


@pytest.mark.parametrize("what", ["role_logits", "hook", "merge", "pool", "max", "grad"])
def test_what_is_replaced_is_called(monkeypatch, what):
    m = build(torch.bfloat16, 256, 8)
    x = torch.randn(1, 50, 256, device="cuda", dtype=torch.bfloat16)
    seen = []
    if what == "role_logits":
        m.role_logits = lambda p: seen.append(1) or type(m).role_logits(m, p)
    elif what == "hook":
        m.proj_layer.register_forward_hook(lambda *a: seen.append(1))
    elif what == "merge":
        f = NAtSCache.merge_new_x_values_in_chunk
        monkeypatch.setattr(NAtSCache, "merge_new_x_values_in_chunk", staticmethod(lambda *a, **k: seen.append(1) or f(*a, **k)))
    elif what == "pool":
        from neuralattentionsearch_amd import cache as cm
        f2 = cm.pool_chunks
        monkeypatch.setattr(cm, "pool_chunks", lambda *a, **k: seen.append(1) or f2(*a, **k))
    elif what == "max":
        from neuralattentionsearch_amd.cache import ChunkMergeType
        m.chunk_merge_method = ChunkMergeType.MAX
        seen.append(1)
    elif what == "grad":
        m.proj_layer.requires_grad_(True)
        calls = []
        role_step = ops.role_step
        monkeypatch.setattr(ops, "role_step", lambda *a, **k: calls.append(1) or role_step(*a, **k))
        m._sample_for_token_info_values_inference(x, 0, NAtSCache(16, 8))
        assert not calls
        return
    _, _, fused = roles_of(m, x, 3, False, monkeypatch)
    assert seen and not fused
