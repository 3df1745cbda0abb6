"""Attention modules of the NAtS inference path on top of the HIP kernels.

Same class names, constructor arguments and method names as the reference's modules
(src/nats/models/transformer/attention/base_attention.py:11-283, nats_attention.py:14-195,
nats_chunk_attention.py:19-157); inference only (the training branch and its Triton backward kernels are
outside this build).  Differences a caller can see:

* keys / values are never repeated to H_q heads: the kernels read the kv heads directly (``repeat_kv_values``
  returns its arguments);
* no [B, H, L, N] mask is built: ``multi_head_attention`` calls the prefill kernel for a multi-token segment
  (over an empty cache, or over the rows earlier segments left) and the decode kernel for one token;
  ``cache.generate_mask`` stays available for inspection.
"""
from __future__ import annotations

import math

import torch
from torch import nn

from . import cache as cache_module
from . import ops
from .cache import ChunkMergeType, NAtSCache, NAtSChunkLayerCache, NAtSLayerCache


def rotate_half(x: torch.Tensor) -> torch.Tensor:
    x1, x2 = x[..., : x.shape[-1] // 2], x[..., x.shape[-1] // 2:]
    return torch.cat((-x2, x1), dim=-1)


def apply_rotary_pos_emb(q, k, cos, sin, unsqueeze_dim: int = 1):
    """q * cos + rotate_half(q) * sin, the HF Llama convention the reference imports
    (base_attention.py:8, 147-151); cos / sin are [B, L, D]."""
    cos = cos.unsqueeze(unsqueeze_dim)
    sin = sin.unsqueeze(unsqueeze_dim)
    return (q * cos) + (rotate_half(q) * sin), (k * cos) + (rotate_half(k) * sin)


_ROTATE_HALF, _APPLY_ROTARY = rotate_half, apply_rotary_pos_emb  # (as this module defines them)


def _plain_linear(m: nn.Module) -> bool:
    """An nn.Linear without bias that nobody has wrapped, hooked or re-parametrised: its call is one matrix product."""
    d = m.__dict__
    return (type(m) is nn.Linear and not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"])
            and "forward" not in d and d["_parameters"].get("bias") is None and type(d["_parameters"].get("weight")) is nn.Parameter)


def _plain_execution(x: torch.Tensor, weights) -> bool:
    """Whether a call may be replaced by kernels on raw addresses: nothing records, transforms or traces the torch ops that
    would run in their place (autograd, forward-mode, vmap, autocast, dispatch and function modes, global module hooks)."""
    return (type(x) is torch.Tensor and not torch._C._functorch.is_functorch_wrapped_tensor(x)
            and not (torch.is_grad_enabled() and (x.requires_grad or any(w.requires_grad for w in weights)))
            and torch.autograd.forward_ad._current_level < 0 and not torch.is_autocast_enabled("cuda")
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0
            and not torch.compiler.is_compiling() and not nn.modules.module._has_any_global_hook())


def _segment_roles_pay(chunks: int, streams: int, chunk_size: int, dim: int, dtype: torch.dtype) -> bool:
    """Whether pooling and projecting `chunks` chunks (of all sequences) in the role kernel takes no longer on the GPU than the
    torch ops and the library's product.  Up to 32 chunks the kernel pools every chunk once per stream, with more every workgroup
    reads the whole weight for one chunk's dot products; the ops copy and pad the hidden states.

    GPU us, kernel / ops, bf16, dim 4096: 5 chunks of 64, 8 streams 15 / 33; 33 of 8, 8 streams 18 / 27, 16 streams 30 / 27, 32 streams
    54 / 28; 128 of 64, 32 streams 70 / 78; 512 of 8, 32 streams 99 / 51; 1024 of 8, 8 streams 56 / 71; 1024 of 64, 32 streams 246 / 436; fp32 34 / 29
    (33 of 8, 32 streams), 255 / 821.  Over 1770 sizes (4 to 64 streams, chunks of 8 to 128, 3 to 4096 of them, dims 1024 to 4096) the kernel
    is 5 % slower in two that this takes, and 15 % faster in 44 that it leaves."""
    if chunks <= 32:
        return chunks * streams * (16 + chunk_size) * dim <= 150_000_000
    if dtype == torch.bfloat16:
        kernel, most = streams * max(320, 160 + 1.05 * chunks), 13_500_000
    else:
        kernel, most = streams * max(110, 80 + 0.45 * chunks), 6_400_000
    return (kernel - (chunks - 20) * chunk_size) * dim <= most


class AttentionLayer(nn.Module):
    """Projections and head bookkeeping (base_attention.py:13-137)."""

    def __init__(self, dim: int = 4096, n_heads: int = 32, n_kv_heads: int | None = None, layer_id: int = 0,
                 dropout: float = 0.0, use_flash: bool = True, on_ddp: bool = False):
        super().__init__()
        self.n_kv_heads = n_heads if n_kv_heads is None else n_kv_heads
        self.layer_id = layer_id
        self.n_local_heads = n_heads
        self.n_local_kv_heads = self.n_kv_heads
        self.n_rep = self.n_local_heads // self.n_local_kv_heads
        self.head_dim = dim // n_heads
        self.wq = nn.Linear(dim, n_heads * self.head_dim, bias=False)
        self.wk = nn.Linear(dim, self.n_kv_heads * self.head_dim, bias=False)
        self.wv = nn.Linear(dim, self.n_kv_heads * self.head_dim, bias=False)
        self.wo = nn.Linear(n_heads * self.head_dim, dim, bias=False)
        self.use_flash = use_flash
        self._use_flash = use_flash
        self.dropout = dropout

    def add_rotary_emb(self, xq, xk, pos_emb):
        if pos_emb is not None:
            cos, sin = pos_emb
            # (one kernel with the rounding points of the torch ops, where nothing watches or replaces those)
            if (rotate_half is _ROTATE_HALF and apply_rotary_pos_emb is _APPLY_ROTARY
                    and all(type(t) is torch.Tensor for t in (xk, cos, sin)) and _plain_execution(xq, (xk, cos, sin))
                    and xq.dim() == xk.dim() == 4 and cos.shape == sin.shape == (xq.shape[0], *xq.shape[2:])
                    and (xk.shape[0], *xk.shape[2:]) == cos.shape and xq.shape[3] <= 256 and ops.rope_qk_ok(xq, xk, cos, sin)):
                return ops.rope_qk(xq, xk, cos, sin)
            xq, xk = apply_rotary_pos_emb(xq, xk, cos, sin)
        return xq, xk

    def repeat_kv_values(self, keys, values):
        return keys, values

    def _one_token_step(self, x: torch.Tensor, pos_emb, start_pos: int, cache):
        """The whole forward of one token over a filled cache in a few launches, or None when `forward` has to take its
        general way."""
        return None

    def forward(self, x: torch.Tensor, pos_emb, mask, start_pos: int = 0, cache: NAtSCache | None = None, **kwargs):
        """[B, L, dim] -> [B, L, dim] (base_attention.py:259-283)."""
        if self.training:
            raise NotImplementedError("only the inference path is built; call module.eval()")
        bsz, seqlen, _ = x.shape
        if seqlen == 1 and (step := self._one_token_step(x, pos_emb, start_pos, cache)) is not None:
            return step
        xq, xk, xv, mha_kwargs = self.prepare_x_values(x, bsz=bsz, seqlen=seqlen, pos_emb=pos_emb, start_pos=start_pos,
                                                       cache=cache)
        keys, values = self.prepare_kv(xq, xk, xv, start_pos, cache=cache, kwargs=mha_kwargs)
        keys, values = self.repeat_kv_values(keys, values)
        output = self.multi_head_attention(xq, keys, values, mask=mask, cache=cache, kwargs=mha_kwargs)
        output = output.transpose(1, 2).reshape(bsz, seqlen, -1)
        return self.wo(output)


class BaseNAtSAttentionLayer(AttentionLayer):
    """Role logits and the cache hand-over (nats_attention.py:14-134)."""

    def __init__(self, dim: int = 4096, n_heads: int = 32, n_kv_heads: int | None = None, layer_id: int = 0,
                 dropout: float = 0.0, use_flash: bool = True, on_ddp: bool = False, n_msks: int | None = None,
                 sparse_regularized_value: float = 0.0, local_seq_max_length: int = 4, n_options: int = 3,
                 global_token_enhanced_value: float = 0.1):
        super().__init__(dim, n_heads, n_kv_heads, layer_id, dropout, use_flash, on_ddp)
        if n_msks is None:
            n_msks = n_kv_heads or n_heads
        if n_options != 3:
            raise ValueError("the kernels implement the three roles global / local / sliding window")
        if n_msks != self.n_kv_heads:
            raise NotImplementedError("one role stream per kv head is supported (n_msks == n_kv_heads)")
        self.proj_layer = nn.Linear(dim, n_msks * n_options, bias=False)
        self.n_msks = n_msks
        self.n_options = n_options
        self.n_rep_msk = n_heads // n_msks
        self.sm_scale = 1 / math.sqrt(self.head_dim)
        self.sparse_regularized_value = sparse_regularized_value
        self.local_seq_max_length = local_seq_max_length
        self.global_token_enhanced_value = global_token_enhanced_value
        one_hot_values = torch.zeros(n_options)
        one_hot_values[0] = 1.0
        self.one_hot_values = one_hot_values
        self.executor = None
        self._cache_is_till_updating = None

    def prepare_x_values(self, x, bsz: int, seqlen: int, pos_emb, start_pos: int = 0, cache: NAtSCache | None = None):
        xq, xk, xv = self.wq(x), self.wk(x), self.wv(x)
        xq = xq.view(bsz, seqlen, self.n_local_heads, self.head_dim).transpose(1, 2)
        xk = xk.view(bsz, seqlen, self.n_local_kv_heads, self.head_dim).transpose(1, 2)
        xv = xv.view(bsz, seqlen, self.n_local_kv_heads, self.head_dim).transpose(1, 2)
        token_states_info = self._sample_for_token_info_values_inference(x, start_pos=start_pos, cache=cache)
        xq, xk = self.add_rotary_emb(xq, xk, pos_emb)
        return xq, xk, xv, {"token_states_info": token_states_info}

    def role_logits(self, x_pooled: torch.Tensor) -> torch.Tensor:
        """[B, S, dim] -> [B, S, H_kv, 3]"""
        return self.proj_layer(x_pooled).unflatten(-1, (self.n_msks, self.n_options))

    def _sample_for_token_info_values_inference(self, x, start_pos, cache: NAtSCache | None = None,
                                                sink_token_end: int = 1, force_last_global: bool = False):
        """nats_attention.py:96-109 on the roles kernel: bias on option 0, first maximum, sink slot global."""
        logit = self.role_logits(x)
        _, one_hot = ops.roles_from_logits(logit, self.global_token_enhanced_value,
                                           force_first_global=start_pos < sink_token_end,
                                           force_last_global=force_last_global)
        return one_hot

    def prepare_kv(self, xq, xk, xv, start_pos: int = 0, cache: NAtSCache | None = None, kwargs: dict | None = None):
        if self._cache_is_till_updating is not None:  # nats_attention.py:122-123
            self._cache_is_till_updating.result()
            self._cache_is_till_updating = None
        return cache.update(key_states=xk, value_states=xv, layer_idx=self.layer_id, cache_kwargs=kwargs)

    def _post_update(self, cache: NAtSCache, x_len: int):
        """Eviction after the attention (nats_attention.py:189-195).  With an executor the job is handed to its
        thread together with the caller's stream: torch's current stream is a per-thread setting, and the eviction
        kernels must follow the attention kernel on the stream that ran it."""
        if self.executor is None:
            cache.post_update(layer_idx=self.layer_id, x_len=x_len)
            return
        stream = torch.cuda.current_stream()

        def job():
            with torch.cuda.stream(stream):
                cache.post_update(layer_idx=self.layer_id, x_len=x_len)

        self._cache_is_till_updating = self.executor.submit(job)

    def multi_head_attention(self, xq, keys, values, mask=None, cache: NAtSCache | None = None,
                             is_first_module: bool = True, kwargs: dict | None = None):
        """Inference branch of nats_attention.py:136-195 / nats_chunk_attention.py:97-157 on the kernels: the mask
        the reference takes from cache.generate_mask is evaluated inside them, from the cache's own window."""
        assert "token_states_info" in kwargs, "Token States Infor is required for multi head attention!"
        x_len = xq.shape[-2]
        layer = cache.cache_model[self.layer_id]
        if x_len == 1 and layer.get_seq_length() > 0:
            row_end, tail_start = layer.decode_hint()
            output = ops.decode_attention(xq, keys, values, layer.valid_tokens, keys.shape[2], self.sm_scale,
                                          row_end=row_end, tail_start=tail_start)
        elif layer.get_seq_length() == 0:
            roles = ops.roles_from_one_hot(kwargs["token_states_info"])
            output = ops.prefill_attention(xq, keys, values, roles, layer.chunk_size, layer.sliding_window_size,
                                           self.sm_scale)
        else:
            output = layer.segment_attention(xq, self.sm_scale)
        self._post_update(cache, x_len)
        return output

    def _step_as_defined(self, cache, layer) -> bool:
        """Whether everything `_one_token_step` stands in for is what this package (and torch) defines: nothing of it replaced
        in a subclass, on a class, on an object or in a module."""
        cls, kind = type(self), type(layer)
        return (cls.prepare_x_values is _PREPARE_X and cls.add_rotary_emb is _ADD_ROTARY and cls.prepare_kv is _PREPARE_KV
                and cls.repeat_kv_values is _REPEAT_KV and cls.multi_head_attention is _ATTENTION and cls.role_logits is _ROLE_LOGITS
                and cls._sample_for_token_info_values_inference in _SAMPLES
                and BaseNAtSAttentionLayer._sample_for_token_info_values_inference is _SAMPLE
                and apply_rotary_pos_emb is _APPLY_ROTARY and rotate_half is _ROTATE_HALF
                and ops.roles_from_logits is _ROLES_FROM_LOGITS and ops.roles_from_one_hot is _ROLES_FROM_ONE_HOT
                and NAtSCache.update is _CACHE_UPDATE and NAtSCache.merge_new_x_values_in_chunk is _MERGE
                and NAtSCache.update_nats_cached_x_in_chunk is _IN_CHUNK
                and NAtSCache.update_nats_cached_x_across_chunk is _ACROSS_CHUNK
                and kind.update in _LAYER_UPDATES and kind.valid_tokens in _VALID_TOKENS
                and nn.Linear.forward is _LINEAR_FORWARD and nn.functional.linear is _LINEAR and nn.Module.__call__ is _CALL
                and self.__dict__.keys().isdisjoint(_STEP_METHODS) and cache.__dict__.keys().isdisjoint(_CACHE_METHODS)
                and "update" not in layer.__dict__)

    def _one_token_step(self, x, pos_emb, start_pos, cache):
        """One token per sequence over a filled cache: projections, chunk statistic and roles in one launch, the rotary
        embedding with the cache append in a second, then the decode kernel and the output projection.  (The torch ops of
        the general way are about thirty launches, and a token waits for each of them.)  The results are the same ops with
        the same rounding points; only the order of the fp32 sums inside the products differs."""
        layer_id = self.layer_id
        if type(cache) is not NAtSCache or pos_emb is None or len(cache.cache_model) <= layer_id:
            return None
        layer = cache.cache_model[layer_id]
        chunked = type(layer) is NAtSChunkLayerCache
        if not (chunked or type(layer) is NAtSLayerCache) or not self._step_as_defined(cache, layer):
            return None
        C = cache.chunk_size
        is_chunk_module = isinstance(self, BaseNAtSChunkAttentionLayer)
        if is_chunk_module:
            if self.chunk_size != C or (C > 1 and self.chunk_merge_method is not ChunkMergeType.MEAN):
                return None
        elif C != 1:
            return None
        mods = self._modules
        linears = (mods.get("wq"), mods.get("wk"), mods.get("wv"), mods.get("wo"), mods.get("proj_layer"))
        if not all(map(_plain_linear, linears)):
            return None
        wq, wk, wv, wo, wr = (m._parameters["weight"] for m in linears)
        cos, sin = pos_emb
        B, _, dim = x.shape
        Hq, Hkv, D = self.n_local_heads, self.n_local_kv_heads, self.head_dim
        if (not _plain_execution(x, (wq, wk, wv, wo, wr)) or type(cos) is not torch.Tensor or type(sin) is not torch.Tensor
                or not ops.matvec_takes(x, wo, Hq * D) or not ops.matvec_takes(x, wr, dim) or wr.shape[0] != 3 * Hkv
                or wq.shape[0] != Hq * D or wk.shape[0] != Hkv * D or wv.shape[0] != Hkv * D or cos.shape != (B, 1, D) or sin.shape != cos.shape or cos.dtype != x.dtype or sin.dtype != x.dtype
                or not cos.is_cuda or not sin.is_cuda or cos.stride(-1) != 1 or sin.stride(-1) != 1 or D > 256 or D % 2):
            return None
        if self._cache_is_till_updating is not None:  # nats_attention.py:122-123
            self._cache_is_till_updating.result()
            self._cache_is_till_updating = None
        if layer.bsz != B or layer.get_seq_length() <= 0 or not layer.takes_rotated_rows(x.dtype, D):
            return None
        pre_fill = cache.get_nats_chunk_fill_size(layer_id)
        carry_in = None
        if pre_fill:
            carry_in = cache.get_nats_cached_x_in_chunk(layer_id)
            if (carry_in is None or carry_in.shape != x.shape or carry_in.dtype != x.dtype or carry_in.device != x.device
                    or not carry_in.is_contiguous() or carry_in.data_ptr() % 16):
                return None
        roles = None
        if pre_fill + 1 >= C:
            if not chunked:
                roles = layer.role_destination(1)
            if roles is None:
                roles = torch.empty(B, Hkv, 1, dtype=torch.uint8, device=x.device)
        projected = ops.try_step_project(x, (wq, wk, wv), C, carry_in, roles is None, wr, roles, self.global_token_enhanced_value,
                                         start_pos < C)
        if projected is None:
            return None
        qkv, carry = projected
        if is_chunk_module:
            cache._update_cache_x(carry, layer_id)
        if layer_id == 0:
            cache.cache_model[-1].settle()  # (as `NAtSCache.update` does)
        q, k, v = qkv.view(B, 1, Hq + 2 * Hkv, D).transpose(1, 2).split_with_sizes((Hq, Hkv, Hkv), 1)
        output = layer.step_attention(q, k, v, cos, sin, None, roles, self.sm_scale)
        self._post_update(cache, 1)
        return ops.matvec(output.view(B, 1, Hq * D), wo)


_STEP_METHODS = frozenset(("prepare_x_values", "add_rotary_emb", "prepare_kv", "repeat_kv_values", "multi_head_attention",
                           "role_logits", "_sample_for_token_info_values_inference"))
_CACHE_METHODS = frozenset(("update", "merge_new_x_values_in_chunk", "update_nats_cached_x_in_chunk", "update_nats_cached_x_across_chunk"))


class BaseNAtSChunkAttentionLayer(BaseNAtSAttentionLayer):
    """Chunk-granular roles (nats_chunk_attention.py:19-157)."""

    def __init__(self, dim: int = 4096, n_heads: int = 32, n_kv_heads: int | None = None, layer_id: int = 0,
                 dropout: float = 0.0, use_flash: bool = True, on_ddp: bool = False, n_msks: int | None = None,
                 sparse_regularized_value: float = 0.0, local_seq_max_length: int = 4, n_options: int = 3,
                 chunk_size: int = 8, chunk_merge_method: str = "mean", compress_on_q: bool = False):
        super().__init__(dim, n_heads, n_kv_heads, layer_id, dropout, use_flash, on_ddp, n_msks,
                         sparse_regularized_value, local_seq_max_length, n_options)
        if chunk_merge_method == "mean":
            self.chunk_merge_method = ChunkMergeType.MEAN
        elif chunk_merge_method == "max":
            self.chunk_merge_method = ChunkMergeType.MAX
        else:
            raise ValueError(f"Unknown chunk merge method: {chunk_merge_method}")
        self.chunk_size = chunk_size
        self.compress_on_q = compress_on_q

    def get_pad_size(self, x_len):
        return (-x_len) % self.chunk_size

    def _sample_for_token_info_values_inference(self, x, start_pos, cache: NAtSCache | None = None):
        """nats_chunk_attention.py:64-95: while the open chunk is not complete the hidden states are only
        accumulated and a global placeholder role is handed on; otherwise one role per chunk touched, from the
        pooled hidden states, with the open last chunk forced global."""
        x_len = x.shape[1]
        pre_fill = cache.get_nats_chunk_fill_size(self.layer_id)
        if pre_fill + x_len < self.chunk_size:
            cache.update_nats_cached_x_in_chunk(x, self.layer_id, self.chunk_merge_method)
            return self.one_hot_values.to(x).reshape(1, 1, 1, -1).expand(x.shape[0], self.n_kv_heads, 1, -1)
        if (roles := self._segment_roles(x, pre_fill, start_pos, cache)) is not None:
            return roles
        x_pooled, pad_size = cache.update_nats_cached_x_across_chunk(x, pre_fill, self.layer_id, self.chunk_merge_method)
        return super()._sample_for_token_info_values_inference(x_pooled, start_pos, sink_token_end=self.chunk_size,
                                                               force_last_global=pad_size != 0)

    def _segment_roles(self, x, pre_fill: int, start_pos: int, cache):
        """The pooling, the role projection and the roles of a segment that completes a chunk, in one launch where the torch
        ops and the library product they stand in for are up to eleven (a turn of 301 tokens at dim 4096 waits for all of
        them).  None where something of it is replaced, watched or not what the kernel computes: a mean over a chunk size
        that is a power of two (dividing by it is exact, so the statistics are those of the torch ops; the fp32 sums of the
        projection run in another order) from 8 on, in sizes at which the kernel is no slower (`_segment_roles_pay`), rows of whole 16
        bytes."""
        C, H = self.chunk_size, self.n_msks
        proj = self._modules.get("proj_layer")
        if (type(cache) is not NAtSCache or cache.chunk_size != C or C < 8 or C & (C - 1)
                or self.chunk_merge_method is not ChunkMergeType.MEAN or x.dim() != 3 or proj is None or not _plain_linear(proj)):
            return None
        w = proj._parameters["weight"]
        B, _, dim = x.shape
        if (not _plain_execution(x, (w,)) or not x.is_cuda or x.device != w.device or x.dtype != w.dtype
                or x.dtype not in (torch.bfloat16, torch.float32) or x.stride(-1) != 1 or not w.is_contiguous() or w.shape != (3 * H, dim)
                or H > 256 or (dim + 3 * H) * 4 > 160 * 1024 or not 0 < B <= 65535 or not self._segment_as_defined(cache)
                or not _segment_roles_pay(B * -(-(pre_fill + x.shape[1]) // C), H, C, dim, x.dtype)
                or (dim * x.element_size() | x.stride(0) * x.element_size() | x.stride(1) * x.element_size() | x.data_ptr() | w.data_ptr()) % 16):
            return None
        carry = None
        if pre_fill:
            carry = cache.get_nats_cached_x_in_chunk(self.layer_id)
            if carry is None or carry.shape != (B, 1, dim) or carry.dtype != x.dtype or carry.device != x.device:
                return None
        step = ops.role_step(x, w, C, 0, pre_fill=pre_fill, carry_in=carry, global_bias=self.global_token_enhanced_value,
                             force_first_global=start_pos < C)
        cache._update_cache_x(step["carry"], self.layer_id)
        return step["token_states_info"]

    def _segment_as_defined(self, cache) -> bool:
        """Whether everything `_segment_roles` stands in for is what this package (and torch) defines."""
        return (type(self).role_logits is _ROLE_LOGITS and super()._sample_for_token_info_values_inference.__func__ is _SAMPLE
                and ops.roles_from_logits is _ROLES_FROM_LOGITS and cache_module.pool_chunks is _POOL_CHUNKS
                and NAtSCache.merge_new_x_values_in_chunk is _MERGE and NAtSCache.update_nats_cached_x_across_chunk is _ACROSS_CHUNK
                and NAtSCache._update_cache_x is _UPDATE_X and NAtSCache.get_nats_cached_x_in_chunk is _CACHED_X
                and NAtSCache.get_nats_chunk_fill_size is _FILL_SIZE
                and nn.Linear.forward is _LINEAR_FORWARD and nn.functional.linear is _LINEAR and nn.Module.__call__ is _CALL
                and "role_logits" not in self.__dict__ and cache.__dict__.keys().isdisjoint(_SEGMENT_CACHE_METHODS))



class GPTNAtSAttentionLayer(BaseNAtSAttentionLayer):
    """Per-token roles (chunk_size == 1), nats_attention.py:198-199."""


class LlamaNAtSAttentionLayer(BaseNAtSAttentionLayer):
    """Per-token roles (chunk_size == 1), nats_attention.py:202-203."""


class GPTNAtSChunkAttentionLayer(BaseNAtSChunkAttentionLayer):
    pass


class LlamaNAtSChunkAttentionLayer(BaseNAtSChunkAttentionLayer):
    pass


# What `_one_token_step` stands in for, as it is when this module is loaded.
_PREPARE_X = BaseNAtSAttentionLayer.prepare_x_values
_ADD_ROTARY = AttentionLayer.add_rotary_emb
_PREPARE_KV = BaseNAtSAttentionLayer.prepare_kv
_REPEAT_KV = AttentionLayer.repeat_kv_values
_ATTENTION = BaseNAtSAttentionLayer.multi_head_attention
_ROLE_LOGITS = BaseNAtSAttentionLayer.role_logits
_SAMPLE = BaseNAtSAttentionLayer._sample_for_token_info_values_inference
_SAMPLES = (BaseNAtSChunkAttentionLayer._sample_for_token_info_values_inference, _SAMPLE)
_ROLES_FROM_LOGITS, _ROLES_FROM_ONE_HOT = ops.roles_from_logits, ops.roles_from_one_hot
_CACHE_UPDATE, _MERGE = NAtSCache.update, NAtSCache.merge_new_x_values_in_chunk
_IN_CHUNK, _ACROSS_CHUNK = NAtSCache.update_nats_cached_x_in_chunk, NAtSCache.update_nats_cached_x_across_chunk
_LAYER_UPDATES = (NAtSChunkLayerCache.update, NAtSLayerCache.update)
_VALID_TOKENS = (NAtSChunkLayerCache.valid_tokens, NAtSLayerCache.valid_tokens)
_LINEAR_FORWARD, _LINEAR, _CALL = nn.Linear.forward, nn.functional.linear, nn.Module.__call__
_POOL_CHUNKS = cache_module.pool_chunks
_UPDATE_X, _CACHED_X, _FILL_SIZE = NAtSCache._update_cache_x, NAtSCache.get_nats_cached_x_in_chunk, NAtSCache.get_nats_chunk_fill_size
_SEGMENT_CACHE_METHODS = _CACHE_METHODS | {"_update_cache_x", "get_nats_cached_x_in_chunk", "get_nats_chunk_fill_size"}
