"""GPU: prefill launches of one to four rounds of workgroups whose streams differ in how much is visible (the map that
starts the heavy streams first), against fp32 attention under the oracle's mask."""
import math

import numpy as np
import pytest
import torch

from oracle import nats_oracle as orc
from tests.gpu_util import draw_roles, say

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["1", None], ids=["looks", "rule"])
def balance(request, monkeypatch):
    """The look at the streams in every launch of such a size, and where the rule has it."""
    if request.param:
        monkeypatch.setenv("NATS_PREFILL_BALANCE", request.param)
        monkeypatch.setenv("NATS_PREFILL_SPLIT", "0")


@pytest.mark.parametrize("B,Hq,Hkv,D,L,C,W,heavy", [
    (1, 32, 8, 128, 2100, 64, 128, [0]),          # one heavy stream of eight, 33 query tiles
    (2, 32, 4, 128, 2050, 64, 128, [5]),          # two head groups per kv head
    (3, 12, 3, 32, 1900, 64, 64, [8, 0]),         # nine streams, one XCD has two
    (1, 4, 1, 32, 20000, 64, 64, [0]),            # a single stream: the plain map
    (2, 32, 8, 64, 1100, 64, 64, []),             # no heavy stream
    (2, 32, 8, 64, 1100, 64, 64, list(range(16))),
    (1, 32, 8, 64, 4200, 64, 64, [3]),            # head dim 64: from two rounds of workgroups on
])
def test_prefill_with_streams_of_unequal_weight(balance, B, Hq, Hkv, D, L, C, W, heavy):
    from neuralattentionsearch_amd import ops
    say("balance", B, Hq, Hkv, D, L, C, W, heavy)
    S = math.ceil(L / C)
    roles = draw_roles(L + D, B, Hkv, S, p=(0.02, 0.05, 0.93))
    for s in heavy:
        roles[s // Hkv, s % Hkv] = 0
    roles[:, :, -1] = 0
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(B, h, L, D, generator=g).bfloat16().cuda() for h in (Hq, Hkv, Hkv))
    got = ops.prefill_attention(q, k, v, torch.from_numpy(roles).cuda(), C, W)
    n_rep = Hq // Hkv
    for b in range(B):
        for h in range(Hkv):
            for lo in range(0, L, 4096):  # (rows at a time: the masks of a long stream are large)
                hi = min(lo + 4096, L)
                mask = torch.from_numpy(np.ascontiguousarray(orc_rows(roles[b:b + 1, h:h + 1], L, C, W, lo, hi))).cuda()
                for r in range(n_rep):
                    sc = q[b, h * n_rep + r, lo:hi].float() @ k[b, h].float().T / math.sqrt(D)
                    want = torch.softmax(sc.masked_fill(~mask, -math.inf), -1) @ v[b, h].float()
                    err = (got[b, h * n_rep + r, lo:hi].float() - want).abs().max().item()
                    # bf16 probabilities and output: 2^-8 of values of order one, twice
                    assert err <= 2e-2, (b, h, r, lo, err)


def orc_rows(roles, L, C, W, lo, hi):
    """Rows [lo, hi) of the oracle's mask of one stream, from its slot limits."""
    if L <= 4096:
        return orc.prefill_mask(roles, L, C, W)[0, 0, lo:hi]
    S = roles.shape[-1]
    r = roles[0, 0]
    nxt = np.empty(S, dtype=np.int64)
    e = S - 1
    for n in range(S - 1, -1, -1):
        e = n if r[n] == 0 else e
        nxt[n] = e
    lim = np.where(r == 0, S, np.where(r == 2, np.arange(S) + W // C, nxt))
    keys, qs = np.arange(L), np.arange(lo, hi)[:, None]
    return (keys[None] <= qs) & (qs // C <= lim[keys // C][None])


@pytest.mark.parametrize("Hq,Hkv,D,first,L,C,W,heavy", [
    (32, 8, 128, 1500, 2100, 64, 128, [0]),
    (32, 8, 64, 1000, 2112, 16, 64, [7, 3]),  # packed tiles
    (32, 8, 32, 600, 2070, 4, 32, [1]),       # gathered rows
    (12, 3, 64, 300, 6000, 32, 64, [2]),      # three streams on eight XCDs
    (12, 3, 64, 1500, 6000, 64, 64, [2]),     # over enough rows: a stream twice as heavy as the mean
])
def test_segment_with_streams_of_unequal_weight(balance, Hq, Hkv, D, first, L, C, W, heavy):
    from neuralattentionsearch_amd.cache import NAtSChunkLayerCache
    say("balance, filled cache", Hq, Hkv, D, first, L, C, W, heavy)
    roles = draw_roles(L, 1, Hkv, -(-(first + L) // C) + 1, p=(0.02, 0.05, 0.93))
    roles[0, heavy] = 0
    cache = NAtSChunkLayerCache(1, Hkv, W, chunk_size=C, device="cuda")
    g = torch.Generator().manual_seed(L)
    for n in (first, L):
        k, v = (torch.randn(1, Hkv, n, D, generator=g).bfloat16().cuda() for _ in range(2))
        S = -(-(cache.chunk_fill_size + n) // C)
        r = torch.from_numpy(roles[:, :, :S].copy())
        if (cache.chunk_fill_size + n) % C:
            r[:, :, -1] = 0
        keys, values = cache.update(k, v, None, roles=r.cuda())
        if n == L:
            q = torch.randn(1, Hq, L, D, generator=g).bfloat16().cuda()
            got = cache.segment_attention(q)
            mask = cache.generate_mask(L)  # (pinned against the oracle elsewhere)
            for hq in range(Hq):
                h = hq // (Hq // Hkv)
                sc = q[0, hq].float() @ keys[0, h].float().T / math.sqrt(D)
                want = torch.softmax(sc.masked_fill(~mask[0, h], -math.inf), -1) @ values[0, h].float()
                err = (got[0, hq].float() - want).abs().max().item()
                assert err <= 2e-2, (hq, err)  # (as above)
        cache.post_update(n)
