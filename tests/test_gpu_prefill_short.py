"""GPU: short prompts from an empty cache (one launch, limits from the roles inside it) against the oracle."""
import math

import pytest
import torch

from oracle import nats_oracle as orc
from tests.gpu_util import draw_roles, say, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("L,C,W", [(1, 1, 1), (1, 64, 64), (31, 1, 4), (32, 8, 16), (33, 64, 64), (63, 3, 9), (64, 64, 256), (65, 1, 0),
                                   (127, 16, 16), (129, 2048, 2048), (173, 64, 256), (257, 5, 50), (300, 1, 64), (511, 32, 64),
                                   (513, 128, 128), (1000, 7, 70), (1023, 1, 256), (1024, 64, 128), (2047, 32, 96),
                                   (2048, 1, 512)])
def test_short_prompts(D, L, C, W):
    from neuralattentionsearch_amd import ops
    B, Hq, Hkv = (2, 3, 1) if L % 2 else (1, 8, 4)
    say("short", D, L, C, W)
    g = torch.Generator().manual_seed(L * D)
    S = math.ceil(L / C)
    for p in ((0.05, 0.15, 0.8), (0.01, 0.95, 0.04), (1.0, 0.0, 0.0)):
        roles = draw_roles(L + D, B, Hkv, S, p=p)
        q, k, v = (torch.randn(B, L, h, D, generator=g).bfloat16().transpose(1, 2) for h in (Hq, Hkv, Hkv))
        want = orc.masked_attention(q.float(), k.float(), v.float(), orc.prefill_mask(roles, L, C, W))
        got = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), to_dev(roles), C, W).cpu().float()
        # probabilities and output in bf16: 2^-9 of values up to 4, each
        err = (got - want).abs().max().item()
        assert err <= 2e-2, (p, err)


@pytest.mark.parametrize("Hq,Hkv,D,C,lens", [
    (16, 4, 64, 64, (1536, 1537)), (16, 16, 64, 64, (2048,)),  # three / four workgroups per compute unit
    (40, 10, 64, 64, (768, 769)), (32, 8, 64, 64, (896, 897)), (64, 16, 64, 64, (512, 513)),
    (32, 8, 64, 1, (1024, 1025)),
    (8, 8, 128, 64, (2047, 2049)), (12, 4, 128, 64, (1344, 1345)),
    (8, 8, 64, 1, (1792, 1793)), (8, 8, 128, 3, (1792, 1793)), (8, 8, 128, 4, (1793,)),  # chunks of a few tokens
])
def test_both_sides_of_the_line(Hq, Hkv, D, C, lens):
    from neuralattentionsearch_amd import ops
    for L in lens:
        say("short, line", Hq, Hkv, D, C, L)
        g = torch.Generator().manual_seed(L)
        roles = draw_roles(L, 1, Hkv, math.ceil(L / C), p=(0.05, 0.15, 0.8))
        q, k, v = (torch.randn(1, h, L, D, generator=g).bfloat16() for h in (Hq, Hkv, Hkv))
        want = orc.masked_attention(q.float(), k.float(), v.float(), orc.prefill_mask(roles, L, C, 192 // C * C))
        got = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), to_dev(roles), C, 192 // C * C).cpu().float()
        assert (got - want).abs().max().item() <= 2e-2, L  # (as above)


def test_short_prompt_into_strided_output_at_other_scales():
    from neuralattentionsearch_amd import ops
    g = torch.Generator().manual_seed(9)
    B, Hq, Hkv, L, D, C, W = 3, 8, 2, 200, 64, 16, 32
    roles = draw_roles(1, B, Hkv, math.ceil(L / C))
    q, k, v = (torch.randn(B, h, L, D, generator=g).bfloat16() for h in (Hq, Hkv, Hkv))
    mask = orc.prefill_mask(roles, L, C, W)
    for scale in (0.0, -0.2, 1.5):
        out = torch.full((B, L, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda").transpose(1, 2)
        ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), to_dev(roles), C, W, scale, out=out)
        want = orc.masked_attention(q.float() * (scale * math.sqrt(D)), k.float(), v.float(), mask)
        assert (out.cpu().float() - want).abs().max().item() <= 2e-2, scale
