"""The decode schedules (several workgroups per head, one of eight or of four wavefronts per head, the balanced one) on both
sides of the lines between them, with unequal heads and invalid rows that hold NaN, against the oracle at the tolerance of
tests/test_gpu_decode.py."""
import pytest
import torch

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
    (130, 8, 8, 32, 64, 64, 8, 1),                                      # balanced, more streams than one launch schedules
])
def test_schedules(B, Hq, Hkv, D, W, C, chunks, fill):
    run_case(B, Hq, Hkv, D, W, C, chunks, torch.bfloat16, seed=chunks, fill=fill)
