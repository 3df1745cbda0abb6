"""GPU: moving a cache into larger buffers in one launch, against torch ops."""
import pytest
import torch

from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,have,rows,D,dtype,keep,pos", [(1, 1, 1, 2, 8, torch.bfloat16, None, False), (2, 3, 70, 200, 128, torch.bfloat16, None, True),
                                                            (1, 8, 333, 1024, 64, torch.float32, 300, True), (3, 2, 64, 64, 256, torch.float32, 0, False),
                                                            (1, 2, 5, 4100, 16, torch.bfloat16, 5, True)])
def test_cache_widen(B, H, have, rows, D, dtype, keep, pos):
    from neuralattentionsearch_amd import ops
    say("widen", B, H, have, rows, D, dtype, keep)
    k, v = (torch.randn(B, H, have, D, device="cuda").to(dtype) for _ in range(2))
    valid = (torch.rand(B, H, have, device="cuda") < 0.5).to(torch.uint8)
    p = torch.randint(0, 99, (B, H, have), device="cuda", dtype=torch.int32) if pos else None
    got = ops.cache_widen(k, v, valid, p, rows, keep)
    n = have if keep is None else keep
    for old, new, fill in zip((k, v, valid, p), got, (0, 0, 0, -1)):
        if old is None:
            assert new is None
            continue
        want = torch.full((B, H, rows, *old.shape[3:]), fill, dtype=old.dtype, device="cuda")
        want[:, :, :n] = old[:, :, :n]
        assert torch.equal(new, want)
    assert ops.cache_widen(k[..., :D // 2], v[..., :D // 2], valid, p, rows) is None  # (not contiguous)
