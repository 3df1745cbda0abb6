"""What a program that uses this package has it do: the cases that performance work is measured on.

Six kinds of work, each through the public entry points a program calls:

* prefill       role logits -> roles -> role-masked attention of a prompt (`ops.roles_from_logits`,
                `ops.prefill_attention`): what every attention layer does once per prompt
* decode        one query token per sequence over the ragged, evicted cache (`ops.decode_attention`): what every layer
                does once per generated token
* evict         one layer's cache takes a stream in, all at once or piece by piece, and drops what the roles say
                (`cache.NAtSChunkLayerCache.update` / `post_update`)
* segments      a prompt cut into segments over one cache: update, attention over the evicted cache, eviction
* conversation  the attention module a model is patched with (`attention.LlamaNAtSChunkAttentionLayer`, or
                `LlamaNAtSAttentionLayer` for a role per token): a prompt, then user turns and one-token steps between them
* serve         a whole random-weight Llama-architecture model (`llama.NAtSLlamaForCausalLM`): a prompt, then one-token
                steps with eviction live in every layer

Every case is a dict of plain values; `listed()` gives the fixed ones, `draw(rng)` one more from the same ranges.
"""
import math

import torch

from neuralattentionsearch_amd import ops
from neuralattentionsearch_amd.attention import LlamaNAtSAttentionLayer, LlamaNAtSChunkAttentionLayer
from neuralattentionsearch_amd.cache import NAtSCache, NAtSChunkLayerCache
from neuralattentionsearch_amd.llama import NAtSLlamaConfig, NAtSLlamaForCausalLM, rotary_tables

DEVICE = "cuda"
GLOBAL_BIAS = 0.1  # what the attention modules add to the global logit

# Role logits are N(0, 1) plus a constant per role (global, local, sliding window).  With GLOBAL_BIAS the argmax then
# lands on the shares beside them: a trained model's sparse mix, a denser one, and what random weights give.
MIXES = {
    "sparse": ((-2.17317727, -1.38648285, 0.0), (0.05, 0.15, 0.80)),
    "denser": ((-1.67833392, -1.31208150, 0.0), (0.10, 0.15, 0.75)),
    "even": ((0.0, 0.0, 0.0), (0.37, 0.315, 0.315)),
}


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # a long document at the Llama-3-8B head shape: the package's headline workload
        dict(name="prefill-32k", kind="prefill", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, L=32768, C=64, W=256, mix="sparse"),
        # a batch of ordinary prompts of odd length at chunk 32, the chunk size of the Llama adapter
        dict(name="prefill-batch", kind="prefill", dtype="bf16", B=4, Hq=32, Hkv=8, D=128, L=3001, C=32, W=256, mix="denser"),
        # a role per token
        dict(name="prefill-token-roles", kind="prefill", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, L=8192, C=1, W=256, mix="sparse"),
        # a short question, where latency and launches are what a user waits for
        dict(name="prefill-short", kind="prefill", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, L=173, C=64, W=256, mix="sparse"),
        # single precision: the configuration that is also checked on a CPU
        dict(name="prefill-f32", kind="prefill", dtype="f32", B=1, Hq=8, Hkv=8, D=64, L=2048, C=64, W=128, mix="even"),
        # a serving batch over long contexts of which each head has kept 10-30 %
        dict(name="decode-batch", kind="decode", dtype="bf16", B=32, Hq=32, Hkv=8, D=128, context=65536, C=64, W=256),
        # one user's token over an ordinary context
        dict(name="decode-one", kind="decode", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, context=16384, C=64, W=256),
        # the eviction that follows the prefill of a batch of long prompts
        dict(name="evict-bulk", kind="evict", dtype="bf16", B=16, Hkv=8, D=128, L=65536, piece=65536, C=64, W=512, mix="denser"),
        # the same cache filled chunk by chunk
        dict(name="evict-stream", kind="evict", dtype="bf16", B=16, Hkv=8, D=128, L=8192, piece=64, C=64, W=512, mix="denser"),
        # a prompt taken in segments, so that its activations stay small
        dict(name="segments", kind="segments", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, L=16384, piece=4096, C=64, W=256, mix="sparse"),
        # one layer of a chat: a prompt, then turns of the user and generated tokens in between
        dict(name="conversation", kind="conversation", dtype="bf16", B=1, dim=4096, Hq=32, Hkv=8, C=64, W=256, prompt=2048,
             turns=2, turn=301, steps=18, mix="sparse"),
        # a model answers a prompt: the Llama-3-8B shape with eight of its layers, which are all alike
        dict(name="serve", kind="serve", dtype="bf16", B=1, layers=8, dim=4096, ffn=14336, vocab=128256, Hq=32, Hkv=8, C=64, W=256,
             prompt=1024, steps=16),
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _chunk_window(rng):
    c = rng.choice([64, 64, 64, 32, 32, 16, 8, 1, 128])
    w = rng.choice([16, 128, 256, 256, 512])
    return c, max(c, w // c * c)


def draw(rng):
    kind = rng.choice(["prefill"] * 5 + ["decode"] * 3 + ["evict"] * 2 + ["segments"] * 2 + ["conversation", "serve"])
    mix = rng.choice(["sparse", "sparse", "denser", "even"])
    hq, hkv = rng.choice([(32, 8), (32, 8), (32, 8), (8, 8), (16, 4), (32, 32), (24, 8)])
    d = rng.choice([128, 128, 128, 64, 64, 32, 256])
    c, w = _chunk_window(rng)
    if kind == "prefill":
        if rng.random() < 0.2:
            hq, hkv = rng.choice([(8, 8), (8, 4), (16, 4)])
            return dict(kind=kind, dtype="f32", B=rng.choice([1, 1, 2]), Hq=hq, Hkv=hkv, D=rng.choice([64, 64, 128]), L=_log_int(rng, 40, 3000),
                        C=c, W=w, mix=mix)
        most = 2 ** 27 // (hq * d)  # elements of q of the largest listed prompt
        length = _log_int(rng, 40, min(32768, most))
        return dict(kind=kind, dtype="bf16", B=_log_int(rng, 1, max(1, min(8, most // length))), Hq=hq, Hkv=hkv, D=d, L=length, C=c, W=w, mix=mix)
    if kind == "decode":
        f32 = rng.random() < 0.15
        context = _log_int(rng, 256, 16384 if f32 else 131072)
        most = 32 * 8 * 65536 * 128 // (hkv * d * context)  # cached elements of the largest listed batch
        return dict(kind=kind, dtype="f32" if f32 else "bf16", B=_log_int(rng, 1, max(1, min(8 if f32 else 64, most))), Hq=hq, Hkv=hkv, D=d,
                    context=context, C=64, W=256)
    if kind == "evict":
        c = max(c, 8)
        w = max(c, w // c * c)
        length = _log_int(rng, 200, 65536)
        pieces = 1 if rng.random() < 0.5 else rng.choice([8, 32, 100])
        return dict(kind=kind, dtype="bf16", B=_log_int(rng, 1, max(1, min(16, 16 * 8 * 65536 * 128 // (hkv * d * length)))), Hkv=hkv, D=d,
                    L=length, piece=max(c, -(-length // pieces)), C=c, W=w, mix=mix)
    if kind == "segments":
        length = _log_int(rng, 500, min(16384, 2 ** 26 // (hq * d)))
        return dict(kind=kind, dtype="bf16", B=1 if length > 4096 else rng.choice([1, 2]), Hq=hq, Hkv=hkv, D=d, L=length,
                    piece=max(c, -(-length // rng.choice([2, 3, 5]))), C=c, W=w, mix=mix)
    if kind == "conversation":
        c = rng.choice([64, 32, 8, 1])
        dim, hq, hkv = rng.choice([(4096, 32, 8), (2048, 32, 8), (1024, 8, 8), (512, 8, 8)])
        return dict(kind=kind, dtype="bf16", B=rng.choice([1, 1, 2, 4]), dim=dim, Hq=hq, Hkv=hkv, C=c, W=w if w % c == 0 and w >= 16 else 256,
                    prompt=_log_int(rng, 100, 2048), turns=rng.choice([1, 2, 3]), turn=_log_int(rng, 2, 400), steps=rng.choice([5, 9, 17]), mix=mix)
    dim, hq, hkv, ffn, vocab = rng.choice([(4096, 32, 8, 14336, 128256), (2048, 32, 8, 8192, 128256), (1024, 16, 4, 2816, 32000)])
    return dict(kind=kind, dtype="bf16", B=rng.choice([1, 1, 2, 4]), layers=rng.choice([4, 6, 8]), dim=dim, ffn=ffn, vocab=vocab, Hq=hq, Hkv=hkv,
                C=rng.choice([64, 64, 32, 1]), W=256, prompt=_log_int(rng, 60, 1024), steps=rng.choice([8, 12, 16]))


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.bfloat16


def _randn(g, *shape, dtype, scale=1.0):
    t = torch.randn(*shape, generator=g, device=DEVICE, dtype=dtype)
    return t.mul_(scale) if scale != 1.0 else t


def _logits(g, B, S, H, mix):
    return _randn(g, B, S, H, 3, dtype=torch.float32) + torch.tensor(MIXES[mix][0], device=DEVICE)


def _pieces(case):
    """[(first token, end)] of the segments a stream is cut into."""
    return [(i, min(i + case["piece"], case["L"])) for i in range(0, case["L"], case["piece"])]


def _chunks_touched(C, begin, end):
    """Chunks that tokens [begin, end) of a stream complete or touch, or 0 while the open chunk stays open."""
    fill = begin % C
    return 0 if fill + end - begin < C else -(-(fill + end - begin) // C)


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    return dict(case=case, **{"prefill": _prepare_prefill, "decode": _prepare_decode, "evict": _prepare_stream, "segments": _prepare_stream,
                              "conversation": _prepare_conversation, "serve": _prepare_serve}[case["kind"]](case, g, int(seed)))


def _prepare_prefill(c, g, seed):
    dt, s = _dtype(c), 1.0 if c["dtype"] == "f32" else 1.0 / math.sqrt(c["D"])
    return dict(q=_randn(g, c["B"], c["Hq"], c["L"], c["D"], dtype=dt, scale=s), k=_randn(g, c["B"], c["Hkv"], c["L"], c["D"], dtype=dt, scale=s),
                v=_randn(g, c["B"], c["Hkv"], c["L"], c["D"], dtype=dt, scale=s),
                logits=_logits(g, c["B"], -(-c["L"] // c["C"]), c["Hkv"], c["mix"]))


def _decode_rows(c):
    """Rows of the cache: ring, the longest head's own rows, the open chunk and the new token."""
    base = c["W"] + int(round(0.30 * c["context"] / c["C"])) * c["C"]
    return base, base + 17 + 1


def _prepare_decode(c, g, seed):
    B, H, C, W, dt = c["B"], c["Hkv"], c["C"], c["W"], _dtype(c)
    share = torch.rand(B, H, generator=g, device=DEVICE) * 0.2 + 0.1  # every head has kept 10-30 % of the context
    own = (share * c["context"] / C).round().long() * C
    base, n_rows = _decode_rows(c)
    alloc = -(-n_rows // C) * C
    rows = torch.arange(alloc, device=DEVICE)
    valid = (rows >= W) & (rows < W + own.unsqueeze(-1))
    valid[:, :, :W] = (torch.rand(B, H, W // C, generator=g, device=DEVICE) < 0.8).repeat_interleave(C, dim=-1)
    valid[:, :, base:n_rows] = True
    return dict(q=_randn(g, B, c["Hq"], 1, c["D"], dtype=dt), k=_randn(g, B, H, alloc, c["D"], dtype=dt), v=_randn(g, B, H, alloc, c["D"], dtype=dt),
                valid=valid, n_rows=n_rows, row_end=W + own, tail_start=base)


def _greedy_head(logits, done, end, mix):
    """Heads differ in how much they keep.  The first head of a stream keeps more than any other, and the same number of
    chunks whatever the seed, so that the longest head, which the cache's size follows, is as long for every seed.
    logits [n, 3] of the chunks a piece touches, of which it completes number `done` ... `end - 1` of the stream."""
    pg, pl, _ = MIXES[mix][1]
    most = [min(s, math.ceil(pg * s + 5 * math.sqrt(pg * s) + 5 * pl / pg)) for s in (done, end)]
    logits[:, 1] = logits[:, 2] - 1.0  # (its other chunks slide)
    own, other = logits[:end - done, 0], logits[:end - done, 2]
    margin = own - other
    if done == 0 and end:
        margin[0] = math.inf  # (a stream's first chunk is global)
    own.copy_(other - 1.0)
    pick = margin.topk(min(end - done, most[1] - most[0])).indices
    own[pick] = other[pick] + 1.0


def _prepare_stream(c, g, seed):
    """A stream's keys and values (and queries), the role logits of each of its pieces, and the layer's cache."""
    B, H, D, L, C, dt = c["B"], c["Hkv"], c["D"], c["L"], c["C"], _dtype(c)
    s = 1.0 / math.sqrt(D) if c["kind"] == "segments" else 1.0
    q = _randn(g, B, c["Hq"], L, D, dtype=dt, scale=s) if c["kind"] == "segments" else None
    k, v = (_randn(g, B, H, L, D, dtype=dt, scale=s) for _ in range(2))
    parts = []
    for lo, hi in _pieces(c):
        n = _chunks_touched(C, lo, hi)
        logits = _logits(g, B, n, H, c["mix"]) if n else None
        if n:
            _greedy_head(logits[0, :, 0], lo // C, hi // C, c["mix"])
        parts.append(dict(q=None if q is None else q[:, :, lo:hi], k=k[:, :, lo:hi], v=v[:, :, lo:hi], logits=logits, first=lo < C, open=hi % C != 0))
    if C == 1:  # (the per-token layer cache is built by the container)
        cache = NAtSCache(c["W"], 1)
    else:
        cache = NAtSChunkLayerCache(B, H, c["W"], chunk_size=C, device=DEVICE)
    return dict(parts=parts, cache=cache)


def _prepare_conversation(c, g, seed):
    torch.manual_seed(seed)
    dim, dt = c["dim"], _dtype(c)
    kw = dict(dim=dim, n_heads=c["Hq"], n_kv_heads=c["Hkv"], layer_id=0, local_seq_max_length=c["W"])
    with torch.device(DEVICE):
        module = LlamaNAtSAttentionLayer(**kw) if c["C"] == 1 else LlamaNAtSChunkAttentionLayer(chunk_size=c["C"], **kw)
    module = module.to(dt).eval().requires_grad_(False)
    # Hidden states are N(0, 1) with one channel that is always on, as trained models have; through it the role projection
    # carries the constants of the role mix, and the mean over a chunk of its other inputs is scaled back to N(0, 1).
    w = _randn(g, c["Hkv"] * 3, dim, dtype=torch.float32, scale=math.sqrt(c["C"] / dim))
    w[:, 0] = torch.tensor(MIXES[c["mix"]][0], device=DEVICE).repeat(c["Hkv"]) / 4.0
    module.proj_layer.weight.copy_(w.to(dt))
    lengths = [c["prompt"]] + ([1] * c["steps"] + [c["turn"]]) * c["turns"] + [1] * c["steps"]
    calls, at = [], 0
    for n in lengths:
        x = _randn(g, c["B"], n, dim, dtype=dt)
        x[..., 0] = 4.0
        pos = torch.arange(at, at + n, device=DEVICE)[None].expand(c["B"], -1)
        calls.append((x, rotary_tables(pos, dim // c["Hq"], 500000.0, dt), at))
        at += n
    return dict(module=module, calls=calls, cache=NAtSCache(c["W"], c["C"]))


def _prepare_serve(c, g, seed):
    cfg = NAtSLlamaConfig(vocab_size=c["vocab"], hidden_size=c["dim"], intermediate_size=c["ffn"], num_hidden_layers=c["layers"],
                          num_attention_heads=c["Hq"], num_key_value_heads=c["Hkv"], chunk_size=c["C"], local_seq_max_length=c["W"], fused_role_step=True)
    # a residual stream of order one, matrices that keep it so, and branches scaled for a depth of 32, as models are trained from
    std = 1.0 / math.sqrt(c["dim"])
    model = NAtSLlamaForCausalLM.random_init(cfg, device=DEVICE, dtype=_dtype(c), seed=seed, std=std)
    with torch.no_grad():
        model.embed_tokens.weight.mul_(1.0 / std)
        for layer in model.layers:
            layer.self_attn.o_proj.weight.mul_(0.125)
            layer.mlp.down_proj.weight.mul_(0.125 * math.sqrt(c["dim"] / c["ffn"]))
    ids = torch.randint(0, c["vocab"], (c["B"], c["prompt"] + c["steps"]), generator=g, device=DEVICE)
    return dict(model=model, prompt=ids[:, :c["prompt"]].contiguous(), tokens=[ids[:, c["prompt"] + i:c["prompt"] + i + 1].contiguous() for i in range(c["steps"])],
                cache=model.new_cache())


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def run(state):
    return {"prefill": _run_prefill, "decode": _run_decode, "evict": _run_evict, "segments": _run_segments,
            "conversation": _run_conversation, "serve": _run_serve}[state["case"]["kind"]](state)


def _run_prefill(s):
    c = s["case"]
    roles, _ = ops.roles_from_logits(s["logits"], GLOBAL_BIAS, True, c["L"] % c["C"] != 0, with_one_hot=False)
    return ops.prefill_attention(s["q"], s["k"], s["v"], roles, c["C"], c["W"])


def _run_decode(s):
    return ops.decode_attention(s["q"], s["k"], s["v"], s["valid"], s["n_rows"], row_end=s["row_end"], tail_start=s["tail_start"])


def _layer(s):
    """The layer cache of a stream, empty: the object itself, or the one a container builds at the first update."""
    s["cache"].reset_cache()
    if isinstance(s["cache"], NAtSCache):
        return None, lambda k, v, **kw: s["cache"].update(k, v, 0, kw), lambda n: s["cache"].post_update(0, n)
    return s["cache"], s["cache"].update, s["cache"].post_update


def _roles_of(part):
    if part["logits"] is None:  # the open chunk stays open: nobody needs a role yet
        return None, None
    return ops.roles_from_logits(part["logits"], GLOBAL_BIAS, part["first"], part["open"])


def _contents(layer):
    return dict(k=layer.cache_k, v=layer.cache_v, valid=layer.valid_tokens, size_global=layer.size_global_kv, size_local=layer.size_local_kv,
                rows=layer.n_ctx_data)


def _run_evict(s):
    layer, update, post_update = _layer(s)
    for part in s["parts"]:
        roles, one_hot = _roles_of(part)
        update(part["k"], part["v"], token_states_info=one_hot, roles=roles)
        post_update(part["k"].shape[2])
    return _contents(layer if layer is not None else s["cache"].cache_model[0])


def _run_segments(s):
    c = s["case"]
    layer, update, post_update = _layer(s)
    outs = []
    for i, part in enumerate(s["parts"]):
        roles, one_hot = _roles_of(part)
        keys, values = update(part["k"], part["v"], token_states_info=one_hot, roles=roles)
        layer = layer if layer is not None else s["cache"].cache_model[0]
        if i == 0:
            outs.append(ops.prefill_attention(part["q"], keys, values, roles, c["C"], c["W"]))
        else:
            outs.append(layer.segment_attention(part["q"]))
        post_update(part["k"].shape[2])
    return dict(outs=outs, **_contents(layer))


def _run_conversation(s):
    cache = s["cache"]
    cache.reset_cache()
    with torch.no_grad():
        outs = [s["module"](x, pos_emb, None, start_pos=at, cache=cache) for x, pos_emb, at in s["calls"]]
    return dict(prompt=outs[0], turns=[o for o in outs[1:] if o.shape[1] > 1], steps=torch.cat([o for o in outs[1:] if o.shape[1] == 1], dim=1))


def _run_serve(s):
    cache = s["cache"]
    cache.reset_cache()
    at = s["prompt"].shape[1]
    logits = [s["model"](s["prompt"], 0, cache)]
    for i, token in enumerate(s["tokens"]):
        logits.append(s["model"](token, at + i, cache))
    return torch.stack(logits, dim=1)


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------
def _pairs(L, C, W, mix):
    """(query, key) pairs a stream's roles leave visible, on average: every chunk sees itself up to the diagonal, a sliding
    chunk is seen by the next W / C, a local one up to and including the next global one, a global one by all that follow."""
    pg, pl, ps = MIXES[mix][1]
    S = -(-L // C)
    later = pg * (S - 1) / 2 + ps * min(W // C, S / 2) + pl * min(1 / pg, S / 2)
    return min(L * (L + 1) / 2, S * (C * (C + 1) / 2 + later * C * C))


def _kept_rows(L, C, W, mix):
    """Rows of one head that an eviction keeps: the window's sliding chunks, the global ones and the newest local ones."""
    pg, pl, ps = MIXES[mix][1]
    return min(L, ps * W + pg * L + pl / pg * C)


def work(case):
    c, es = case, 4 if case["dtype"] == "f32" else 2
    if c["kind"] == "prefill":
        io = (2 * c["Hq"] + 2 * c["Hkv"]) * c["B"] * c["L"] * c["D"] * es
        return dict(bytes=io + 12 * c["B"] * c["Hkv"] * -(-c["L"] // c["C"]), flops=4 * c["D"] * c["Hq"] * c["B"] * _pairs(c["L"], c["C"], c["W"], c["mix"]))
    if c["kind"] == "decode":
        rows = c["B"] * c["Hkv"] * (0.2 * c["context"] + 0.8 * c["W"] + 18)
        return dict(bytes=rows * (2 * c["D"] * es + 1) + 2 * c["B"] * c["Hq"] * c["D"] * es, flops=4 * c["D"] * (c["Hq"] // c["Hkv"]) * rows)
    if c["kind"] == "evict":
        kept = _kept_rows(c["L"], c["C"], c["W"], c["mix"])
        read = kept if c["piece"] >= c["L"] else c["L"]  # in one piece the rows that are dropped need not be read
        return dict(bytes=(read + kept) * c["B"] * c["Hkv"] * c["D"] * es * 2, flops=0)
    if c["kind"] == "segments":
        io = (2 * c["Hq"] + 2 * c["Hkv"]) * c["B"] * c["L"] * c["D"] * es
        kept = 2 * _kept_rows(c["L"], c["C"], c["W"], c["mix"]) * c["B"] * c["Hkv"] * c["D"] * es
        return dict(bytes=io + kept, flops=4 * c["D"] * c["Hq"] * c["B"] * _pairs(c["L"], c["C"], c["W"], c["mix"]))
    d = c["dim"] // c["Hq"]
    attn = c["dim"] * (c["Hq"] + 2 * c["Hkv"]) * d + c["Hq"] * d * c["dim"] + c["dim"] * 3 * c["Hkv"]
    if c["kind"] == "conversation":
        n = c["prompt"] + c["turns"] * (c["turn"] + c["steps"]) + c["steps"]
        calls = 1 + c["turns"] * (c["steps"] + 1) + c["steps"]
        ones = (c["turns"] + 1) * c["steps"]
        cached = _kept_rows(n, c["C"], c["W"], c["mix"]) * c["B"] * c["Hkv"] * d * es * 2
        return dict(bytes=calls * attn * es + 2 * n * c["B"] * c["dim"] * es + ones * cached,
                    flops=2 * attn * n * c["B"] + 4 * d * c["Hq"] * c["B"] * _pairs(n, c["C"], c["W"], c["mix"]))
    n = c["prompt"] + c["steps"]
    layer = attn + 3 * c["dim"] * c["ffn"]
    cached = _kept_rows(c["prompt"], c["C"], c["W"], "even") * c["B"] * c["Hkv"] * d * es * 2
    return dict(bytes=(c["steps"] + 1) * (c["layers"] * layer + c["dim"] * c["vocab"]) * es + c["steps"] * c["layers"] * cached,
                flops=2 * c["B"] * (n * c["layers"] * layer + (c["steps"] + 1) * c["dim"] * c["vocab"])
                + 4 * d * c["Hq"] * c["B"] * c["layers"] * _pairs(n, c["C"], c["W"], "even"))


def tolerance(case):
    """About four times how far a pass is from one whose attention is computed in fp32 (bf16 cases) or fp64 (fp32 cases):
    2e-3 ... 3e-3 (largest 0.05) for bf16 attention and its layer, 5e-3 (0.023) for the logits of eight layers, 4.5e-7 (4.5e-6) for
    fp32 attention."""
    if case["kind"] == "evict":
        return "exact"
    if case["dtype"] == "f32":
        return dict(rel=2e-6, max=2e-5)
    if case["kind"] == "serve":
        return dict(rel=2e-2, max=0.1)
    return dict(rel=1e-2, max=0.2)
