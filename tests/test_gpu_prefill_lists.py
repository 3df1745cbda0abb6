"""Visit lists of the bf16 prefill at the edges of how they are read and built (entries are held 64 at a time, granules of up to
4096 rows are listed in one trip) and streams whose rows reach beyond 32-bit byte offsets, against the oracle and each other.

Tolerance 2e-2 as for every bf16 prefill; the two layouts of one input hold the same rows, so their outputs are the same bytes."""
import math

import numpy as np
import pytest
import torch

from oracle import nats_oracle as orc
from tests.gpu_util import draw_roles, say, to_dev
from tests.test_gpu_prefill import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,D,C,W,p", [
    (4095, 128, 64, 256, (0.96, 0.02, 0.02)),   # 61 entries of whole tiles
    (4161, 128, 64, 256, (0.96, 0.02, 0.02)),   # 65
    (8300, 64, 64, 128, (0.97, 0.01, 0.02)),    # 126
    (4096, 128, 32, 256, (0.4, 0.3, 0.3)),      # the last query group walks 256 granules: the early list
    (4112, 128, 32, 256, (0.4, 0.3, 0.3)),      # 257: tile summaries first
    (4300, 32, 16, 32, (0.9, 0.05, 0.05)),      # 62 and 63 packed entries
    (4200, 128, 1, 16, (0.5, 0.25, 0.25)),      # gathered tiles, more than the five known ahead
    (700, 128, 1, 256, (0.1, 0.5, 0.4)),        # fewer
])
@pytest.mark.parametrize("heads", [(4, 1), (1, 1)])
def test_list_edges(monkeypatch, heads, L, D, C, W, p):
    monkeypatch.setenv("NATS_PREFILL_SPLIT", "0")  # one workgroup walks a whole list
    run_case(1, heads[0], heads[1], L, D, C, W, torch.bfloat16, seed=L, p=p)


def list_entries(rows, packed):
    """Entries of the list of a query group, from its rows of the mask [queries, keys]: whole tiles somebody sees, or 16-row granules in
    fours, those that nobody masks among themselves."""
    step = 16 if packed else 64
    parts = np.pad(rows, ((0, 0), (0, -rows.shape[1] % step))).reshape(len(rows), -1, step)
    seen = parts.any((0, 2))
    if not packed:
        return int(seen.sum())
    plain = int(parts.all((0, 2)).sum())
    return plain // 4 + -(-(int(seen.sum()) - plain // 4 * 4) // 4)


@pytest.mark.parametrize("L,D,C,heads,p,entries", [
    (64 * 64, 128, 64, (4, 1), (1.0, 0.0, 0.0), 64), (64 * 66, 64, 64, (4, 1), (1.0, 0.0, 0.0), 66),  # the second group of 64 opened for nothing, for two
    (8711, 32, 64, (4, 1), (0.97, 0.01, 0.02), 135),
    (64 * 64, 128, 16, (4, 1), (1.0, 0.0, 0.0), 64), (64 * 65, 64, 16, (4, 1), (1.0, 0.0, 0.0), 65),
    (9000, 32, 16, (4, 1), (0.96, 0.02, 0.02), 136), (9000, 128, 16, (4, 1), (0.96, 0.02, 0.02), 136),
    (4800, 128, 32, (4, 1), (0.95, 0.03, 0.02), 72), (9000, 64, 64, (1, 1), (0.97, 0.01, 0.02), 138),
])
def test_long_lists(monkeypatch, L, D, C, heads, p, entries):
    """The last query group walks a list of a known length, on both sides of 64 and 128 entries (fp32 reference of its rows)."""
    from neuralattentionsearch_amd import ops
    say("long lists", L, D, C, heads, entries)
    monkeypatch.setenv("NATS_PREFILL_SPLIT", "0")
    roles = draw_roles(L, 1, 1, -(-L // C), p=p)
    tiles = 4 if heads == (1, 1) else 1  # query tiles of a group
    first = (L - 1) // 64 // tiles * tiles * 64
    rows = orc.prefill_mask(roles, L, C, 2 * C)[0, 0, first:]
    assert list_entries(rows, C < 64 or tiles > 1) == entries
    g = torch.Generator(device="cuda").manual_seed(L)
    q = torch.randn(1, heads[0], L, D, generator=g, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(1, 1, L, D, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    got = ops.prefill_attention(q, k, v, to_dev(roles), C, 2 * C)[:, :, first:].float()
    scores = (q[:, :, first:].float() @ k.float().transpose(-1, -2)) / math.sqrt(D)
    want = scores.masked_fill(~to_dev(rows), float("-inf")).softmax(-1) @ v.float()
    assert (got - want).abs().max().item() <= 2e-2


@pytest.mark.parametrize("D,C,W,Hq,Hkv", [(128, 32, 256, 4, 1), (64, 16, 64, 8, 2), (32, 32, 64, 2, 1), (128, 64, 128, 1, 1)])
def test_lists_of_either_kind_hold_the_same_order(monkeypatch, D, C, W, Hq, Hkv):
    """A prompt alone (its granules are listed in one trip) and behind 4096 tokens that slide out of the window (they are not:
    tile summaries first): the same keys in the same order, so the same bytes, for the queries that no longer see the others."""
    from neuralattentionsearch_amd import ops
    say("lists of either kind", D, C, W, Hq, Hkv)
    monkeypatch.setenv("NATS_PREFILL_SPLIT", "0")
    monkeypatch.setenv("NATS_PREFILL_SHORT", "0")
    L, P = 3000, 4096
    g = torch.Generator(device="cuda").manual_seed(D + C)
    q = torch.randn(1, Hq, P + L, D, generator=g, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(1, Hkv, P + L, D, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    roles = to_dev(draw_roles(C, 1, Hkv, math.ceil((P + L) / C)))
    roles[:, :, :P // C] = 2  # sliding window
    both = ops.prefill_attention(q, k, v, roles, C, W)
    alone = ops.prefill_attention(q[:, :, P:], k[:, :, P:], v[:, :, P:], roles[:, :, P // C:].contiguous(), C, W)
    first = -(-(W + C) // 256) * 256  # (a workgroup's query tiles share one list)
    assert torch.equal(both[:, :, P + first:], alone[:, :, first:])


@pytest.mark.parametrize("stride,D,Hq,Hkv,C", [
    (720000, 128, 4, 1, 64), (720000, 128, 4, 1, 32), (720000, 128, 4, 1, 1), (720000, 64, 2, 1, 64), (720000, 32, 4, 1, 8),
    (720000, 128, 32, 8, 64),                                                            # streams in the order of their length
    (400000, 128, 4, 1, 64), (400000, 128, 4, 1, 32), (400000, 128, 4, 1, 1), (400000, 64, 4, 1, 8),
])
def test_rows_beyond_32_bit_offsets(stride, D, Hq, Hkv, C):
    """K and V as every 720000th element group of a 4.5 GB buffer, where row 2983 on lies beyond 2^32 bytes, and of one of 2.5 GB, where
    the offsets do not fit 31 bits: every stream's keys are visited in the same order, so the outputs are the same bytes."""
    from neuralattentionsearch_amd import ops
    say("rows beyond 32-bit offsets", stride, D, Hq, Hkv, C)
    L, W = 3100, 256
    g = torch.Generator(device="cuda").manual_seed(C)
    q = torch.randn(1, Hq, L, D, generator=g, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(1, Hkv, L, D, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    roles = to_dev(draw_roles(C, 1, Hkv, math.ceil(L / C)))
    want = ops.prefill_attention(q, k, v, roles, C, W)
    wide = torch.empty(L * stride, device="cuda", dtype=torch.bfloat16)
    spread = []
    for i, x in enumerate((k, v)):
        view = wide.as_strided((1, Hkv, L, D), (L * stride, 2 * D, stride, 1), storage_offset=i * D)
        view.copy_(x)
        spread.append(view)
    got = ops.prefill_attention(q, spread[0], spread[1], roles, C, W)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype,D,C,L", [
    (torch.bfloat16, 128, 64, 3073), (torch.bfloat16, 128, 64, 3135), (torch.bfloat16, 128, 32, 3001), (torch.bfloat16, 128, 1, 3001),
    (torch.bfloat16, 64, 64, 3100), (torch.bfloat16, 32, 64, 4097), (torch.bfloat16, 64, 8, 3001),
    (torch.bfloat16, 256, 64, 65), (torch.bfloat16, 256, 64, 111), (torch.bfloat16, 256, 8, 273),
    (torch.bfloat16, 128, 64, 33), (torch.bfloat16, 64, 64, 173), (torch.bfloat16, 32, 16, 70),
    (torch.float32, 32, 64, 33), (torch.float32, 64, 64, 173), (torch.float32, 128, 8, 1001),
])
def test_rows_behind_the_last_one_are_not_read(dtype, D, C, L):
    """K and V as the first L rows of longer streams: whatever lies behind them (here: NaN, which a probability of zero would
    pass on) is the same to the result as zeros."""
    from neuralattentionsearch_amd import ops
    say("rows behind the last one", dtype, D, C, L)
    g = torch.Generator(device="cuda").manual_seed(L)
    q = torch.randn(1, 8, L, D, generator=g, device="cuda", dtype=dtype)
    longer = torch.randn(2, 1, 2, L + 128, D, generator=g, device="cuda", dtype=dtype)
    roles = to_dev(draw_roles(C, 1, 2, math.ceil(L / C)))
    outs = []
    for tail in (0.0, float("nan")):
        longer[:, :, :, L:] = tail
        outs.append(ops.prefill_attention(q, longer[0, :, :, :L], longer[1, :, :, :L], roles, C, 256))
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])
