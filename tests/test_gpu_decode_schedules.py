"""The decode schedules (several workgroups per head, one of eight or of four wavefronts per head, the balanced one) on both
sides of the lines between them, with unequal heads and invalid rows that hold NaN, against the oracle.  Scores are peaked
and the error is held against a row's own size (tests/test_gpu_decode.py): a partial result that is lost or wrongly scaled shows."""
import math

import pytest
import torch

from oracle import nats_oracle as orc
from tests.gpu_util import say
from tests.test_gpu_decode import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,D,W,C,chunks,fill", [
    (1, 4, 1, 128, 16, 16, 1, 0), (1, 4, 1, 128, 32, 32, 1, 31), (2, 6, 2, 64, 8, 8, 13, 6),     # a tile or two per head
    (1, 4, 1, 128, 64, 64, 30, 5), (1, 8, 1, 64, 64, 64, 127, 63), (1, 4, 1, 256, 64, 64, 60, 3),  # 64 (32) workgroups per head, edges of a share
    (1, 16, 1, 32, 64, 64, 200, 0),
    (16, 16, 8, 64, 64, 64, 5, 63), (16, 16, 8, 64, 64, 64, 6, 63),     # 128 heads: sixteen tiles and more
    (32, 32, 8, 64, 64, 64, 13, 63), (32, 32, 8, 64, 64, 64, 14, 63),   # 256 heads: 32 tiles and more
    (16, 32, 8, 256, 64, 64, 3, 9),                                     # eight wavefronts do not fit at head dim 256
    (40, 8, 8, 64, 32, 32, 9, 1),                                       # more heads than compute units: one workgroup each
    (5, 32, 8, 256, 64, 64, 33, 0), (5, 32, 8, 256, 64, 64, 38, 0),     # head dim 256: three tiles per wavefront and more
    (24, 32, 8, 128, 64, 64, 9, 63), (24, 32, 8, 128, 64, 64, 13, 63),  # 192 heads, two workgroups each: 15 tiles and more
    (24, 32, 8, 64, 64, 64, 12, 63), (24, 8, 8, 32, 64, 64, 14, 63),    # heads of 64 and 32: 16 tiles and more
    (130, 8, 8, 32, 64, 64, 8, 1),                                      # balanced, more streams than one launch schedules
])
def test_schedules(B, Hq, Hkv, D, W, C, chunks, fill):
    run_case(B, Hq, Hkv, D, W, C, chunks, torch.bfloat16, seed=chunks, fill=fill, q_scale=4.0)


# Rows so that a head's tiles (ceil(rows / 32) + 1) are dealt to `parts` workgroups of four wavefronts.
PARTS = [2, 3, 8, 9, 16, 17, 20, 24, 25, 33, 34, 36, 40, 41, 48, 49, 52, 56, 57, 63, 64]


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("parts", PARTS)
def test_numbers_of_partial_results(D, parts):
    """Scores around zero and all of them far below it (2^-200 against zero)."""
    for shift in (None, -140.0):
        run_case(1, 8, 2, D, 32, 32, 4 * parts - 4, torch.bfloat16, seed=parts, frac=(1.0, 1.0), q_scale=4.0, shift=shift)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("parts", PARTS)
def test_every_partial_result_counts(D, parts):
    """One key carries a head's output: it lies in the first workgroup's tiles for one head, in the next one's for another."""
    from neuralattentionsearch_amd import ops
    say("decode: one key per head", D, parts)
    g = torch.Generator().manual_seed(parts + D)
    H, n_rows = 8, 32 * (4 * parts - 2)
    k, v = (torch.randn(1, H, n_rows, D, generator=g).bfloat16() for _ in range(2))
    q = torch.randn(1, H, 1, D, generator=g).bfloat16()
    valid = torch.ones(1, H, n_rows, dtype=torch.bool)
    for first in range(0, parts, H):
        peaked = k.clone()
        rows = [32 * (4 * ((first + h) % parts) + h % 4) % n_rows + (5 * h) % 32 for h in range(H)]
        for h, r in enumerate(rows):  # a score about 30 nats above the others
            peaked[0, h, r] = (q[0, h, 0].float() * (30.0 * math.sqrt(D) / q[0, h, 0].float().pow(2).sum())).bfloat16()
        want = orc.decode_attention(q, peaked, v, valid, n_rows).float()
        got = ops.decode_attention(q.cuda(), peaked.cuda(), v.cuda(), valid.cuda(), n_rows).cpu().float()
        # the row's own bf16 value, rounded once more (2^-8 of up to 4), and what the other keys weigh (below 1e-8)
        assert (got - want).abs().max().item() <= 4 * 2.0 ** -8, (first, (got - want).abs().amax(-1).flatten().tolist())
