"""The fp32 matrix kernel at the edges of its tiles (32 query rows, 32 keys, 64-tile windows of its iterator) and of its launch
rule, on a first prefill and on segments over a filled cache, against the oracle.

Tolerance 1e-5 on outputs of order one: 1 / sqrt(visible keys) rounding errors of 6e-8 each in sums of at most a few thousand
fp32 products stay well below it (about 5e-7 measured)."""
import math

import numpy as np
import pytest
import torch

from oracle import nats_oracle as orc
from tests.gpu_util import draw_roles, say, to_dev
from tests.test_gpu_prefill import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,Hq,Hkv,L,C,W", [
    (1, 2, 1, 1, 64, 64), (1, 2, 2, 31, 8, 8), (2, 3, 1, 32, 16, 16), (1, 4, 2, 33, 1, 4), (1, 2, 1, 64, 64, 128), (1, 2, 1, 97, 6, 12),
    (1, 1, 1, 2049, 64, 128),   # the second window of tile summaries
    (4, 33, 11, 300, 32, 64),   # more than four workgroups per compute unit: four wavefronts each
    (1, 8, 8, 1030, 64, 128),   # one block of a head more than the compute units take at once: the two lightest share one
    (1, 16, 4, 1000, 16, 32),   # two workgroups per compute unit, all in pairs
    (2, 9, 3, 1111, 64, 64),    # between two and three and a half workgroups per compute unit
])
def test_tile_edges(B, Hq, Hkv, L, C, W, D):
    run_case(B, Hq, Hkv, L, D, C, W, torch.float32, seed=L)


@pytest.mark.parametrize("C,W,lens", [(64, 128, (300, 65, 1, 40, 700)), (8, 16, (100, 33, 5, 64)), (32, 64, (20, 31, 200))])
def test_segments_over_a_filled_cache(C, W, lens):
    from neuralattentionsearch_amd import ops
    from neuralattentionsearch_amd.cache import NAtSChunkLayerCache
    say("f32 segments", C, W, lens)
    B, Hq, Hkv, D = 2, 6, 2, 64
    g = torch.Generator().manual_seed(C)
    cache = NAtSChunkLayerCache(B, Hkv, W, chunk_size=C, device="cuda")
    st = orc.ChunkCacheOracle(B=B, H=Hkv, W=W, C=C)
    for si, n in enumerate(lens):
        q, k, v = (torch.randn(B, h, n, D, generator=g) for h in (Hq, Hkv, Hkv))
        total = cache.chunk_fill_size + n
        first = cache.get_seq_length() == 0
        roles = draw_roles(si, B, Hkv, max(1, math.ceil(total / C)), p=(0.3, 0.3, 0.4), first_global=first)
        if total < C:
            roles[:] = 0
        elif total % C:
            roles[:, :, -1] = 0
        kk, vv = cache.update(k.cuda(), v.cuda(), orc.one_hot_roles(roles).cuda())
        ko, vo = st.update(k, v, roles)
        if first:
            got = ops.prefill_attention(q.cuda(), kk, vv, to_dev(roles), C, W)
        elif n > 1:
            got = cache.segment_attention(q.cuda())
        else:
            got = ops.decode_attention(q.cuda(), kk, vv, cache.valid_tokens, kk.shape[2])
        want = orc.masked_attention(q, ko, vo, st.generate_mask(n)) if n > 1 else \
            orc.decode_attention(q, ko, vo, torch.from_numpy(st.valid), st.n_ctx_data + 1)
        assert np.abs(got.cpu().numpy() - want.numpy()).max() <= 1e-5, (si, n)
        cache.post_update(n)
        st.post_update(n)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,C,W,first,n", [
    (96, 12, 64, 128, 0, 130), (96, 12, 5, 10, 0, 161), (96, 12, 64, 128, 200, 97), (128, 4, 8, 16, 67, 98),  # four wavefronts: 3.75, 4.5, 3, 4 per compute unit
    (6, 3, 64, 128, 0, 2400), (6, 3, 64, 128, 0, 2049),   # long lists, 1.76 and 1.52: eight
])
def test_wavefronts_of_a_workgroup(Hq, Hkv, C, W, first, n, D):
    """Both forms of the kernel, from empty and over cached rows, with tiles that are masked row by row."""
    from neuralattentionsearch_amd import ops
    from neuralattentionsearch_amd.cache import NAtSChunkLayerCache
    say("f32 wavefronts", Hq, Hkv, C, W, first, n, D)
    B = 2
    if not first:
        run_case(B, Hq, Hkv, n, D, C, W, torch.float32, seed=n)
        return
    g = torch.Generator().manual_seed(n)
    cache = NAtSChunkLayerCache(B, Hkv, W, chunk_size=C, device="cuda")
    st = orc.ChunkCacheOracle(B=B, H=Hkv, W=W, C=C)
    for si, m in enumerate((first, n)):
        q, k, v = (torch.randn(B, h, m, D, generator=g) for h in (Hq, Hkv, Hkv))
        roles = draw_roles(si, B, Hkv, math.ceil((cache.chunk_fill_size + m) / C), p=(0.3, 0.3, 0.4), first_global=si == 0)
        if (cache.chunk_fill_size + m) % C:
            roles[:, :, -1] = 0
        cache.update(k.cuda(), v.cuda(), orc.one_hot_roles(roles).cuda())
        ko, vo = st.update(k, v, roles)
        if si:
            want = orc.masked_attention(q, ko, vo, st.generate_mask(m))
            assert np.abs(cache.segment_attention(q.cuda()).cpu().numpy() - want.numpy()).max() <= 1e-5
        cache.post_update(m)
        st.post_update(m)


@pytest.mark.parametrize("scale", [0.0, -0.3])
def test_scales_that_are_not_positive(scale):
    from neuralattentionsearch_amd import ops
    say("f32 scale", scale)
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, 2, 200, 64, generator=g) for _ in range(3))
    roles = draw_roles(3, 1, 2, 4)
    mask = torch.as_tensor(orc.prefill_mask(roles, 200, 64, 64))
    s = (q.double() @ k.double().transpose(-1, -2) * scale).masked_fill(~mask, -math.inf)
    got = ops.prefill_attention(q.cuda(), k.cuda(), v.cuda(), to_dev(roles), 64, 64, scale).cpu()
    assert (got - (s.softmax(-1) @ v.double())).abs().max().item() <= 1e-5
