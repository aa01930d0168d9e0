"""The work that a user of this package gives the GPU, as cases that can be timed and compared.

A model of the Llama kind whose every matrix is a factor pair is asked for one token (``kind`` "token", through the decode
engine that ``step.make_persistent_decoder`` picks: the resident step for one sequence, else ``graphs.GraphedDecoder``) or
takes in a prompt ("prompt", the model's own forward); below the model, the operators that other runtimes call one by one:
the prompt attention on rank coefficients ("attend", ``FlashSVDRoPEAttention``), decode attention over a dense cache
("kv_attention", ``flash_attn_with_kvcache``), and the dual-split MLP on the ``x @ W`` operand layouts ("mlp").

A case names sizes only: ``hidden`` / ``heads`` / ``kv_heads`` / ``head_dim`` / ``inter`` / ``vocab`` / ``layers`` of the
model, its factor ranks, ``batch`` sequences, ``context`` tokens already cached, ``tokens`` new ones, ``dtype``, ``cache``
("dense" post-rotation keys and values, or "rank" coefficients) and ``int4`` factors.  Weights are N(0, 0.02), as the
models of the tests and of ``bench.py``.
"""
from __future__ import annotations

import math

import torch

from flashsvd_amd import llama, quant
from flashsvd_amd.graphs import GraphedDecoder
from flashsvd_amd.kernels.dual_split import flashsvd_mlp_dual_split_triton_v2
from flashsvd_amd.kernels.rope_attn import FlashSVDRoPEAttention, QKVFactors
from flashsvd_amd.runtime import decode_registry
from flashsvd_amd.runtime.cache import FlashSVDLegacySparseKVCache, FlashSVDV15DenseKVCache
from flashsvd_amd.step import PersistentDecoder, make_persistent_decoder

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
STD = 0.02

# model shapes: the one-block configuration of the tests, and the 7B shape with as many kv heads as query heads or a
# quarter of them
SMALL = dict(hidden=512, heads=8, kv_heads=8, head_dim=64, inter=1376, vocab=32000)
WIDE = dict(hidden=4096, heads=32, kv_heads=32, head_dim=128, inter=11008, vocab=32000)
GROUPED = dict(WIDE, kv_heads=8)
MIDDLE = dict(hidden=2048, heads=16, kv_heads=16, head_dim=128, inter=5504, vocab=32000)


def listed():
    token = dict(kind="token", tokens=1, int4=False, dtype="bf16", cache="dense")
    prompt = dict(kind="prompt", int4=False, dtype="bf16", cache="dense", context=0)
    return [
        # one token of a small model: the smallest step, all launches and gaps
        dict(token, name="token_small", **SMALL, layers=1, attn_rank=128, mlp_rank=256, batch=1, context=136),
        # interactive generation with the 7B shape at half the parameters, one sequence: the headline configuration
        dict(token, name="token_7b", **WIDE, layers=32, attn_rank=1024, mlp_rank=1536, batch=1, context=528),
        # the same with int4 factors under float16 activations
        dict(token, name="token_int4", **WIDE, layers=8, attn_rank=1024, mlp_rank=1536, batch=1, context=777)
        | dict(int4=True, dtype="fp16"),
        # sixteen sequences decoded together over the dense cache
        dict(token, name="token_batch", **WIDE, layers=4, attn_rank=1024, mlp_rank=1536, batch=16, context=1000),
        # sixteen long sequences over the rank-space cache at 0.8 of the parameters: the stress configuration
        dict(token, name="token_rank_long", **WIDE, layers=2, attn_rank=1664, mlp_rank=2432, batch=16, context=4090) | dict(cache="rank"),
        # the headline configuration's prompt
        dict(prompt, name="prompt_7b", **WIDE, layers=32, attn_rank=1024, mlp_rank=1536, batch=1, tokens=512),
        # the stress configuration's prompts into the rank-space cache: the largest call
        dict(prompt, name="prompt_long", **WIDE, layers=8, attn_rank=1664, mlp_rank=2432, batch=8, tokens=2048) | dict(cache="rank"),
        # a checkpoint as the parameter-ratio rule leaves it (ratio 0.5: MLP rank 1492, no multiple of 8), an odd prompt
        dict(prompt, name="prompt_ratio", **WIDE, layers=2, attn_rank=1024, mlp_rank=1492, batch=1, tokens=333),
        # the next turn of two conversations: a chunk behind cached tokens, grouped-query heads, float16
        dict(prompt, name="prompt_chunk", **GROUPED, layers=4, attn_rank=1024, mlp_rank=1536, batch=2, tokens=77)
        | dict(dtype="fp16", context=1411),
        # full-sequence attention from rank coefficients with padded rows, as an evaluation batch calls it
        dict(kind="attend", name="attend_padded", heads=32, kv_heads=32, head_dim=128, attn_rank=1024, batch=4, tokens=1024, dtype="bf16"),
        # attend-with-append over a grouped-query cache, as a serving runtime calls it
        dict(kind="kv_attention", name="kv_attention_grouped", heads=32, kv_heads=8, head_dim=128, batch=16, context=4001, dtype="bf16"),
        # the MLP of eight decoded rows on the reference's operand layouts
        dict(kind="mlp", name="mlp_rows", hidden=4096, inter=11008, mlp_rank=1536, batch=8, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["token", "token", "token", "prompt", "prompt", "prompt", "attend", "kv_attention", "mlp"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "attend":
        heads = rng.choice([8, 16, 32])
        tokens = _log(rng, 17, 2048)
        return dict(kind=kind, heads=heads, kv_heads=rng.choice([heads, heads // 4]), head_dim=128, attn_rank=8 * rng.randint(12, 208),
                    batch=max(1, min(8, _log(rng, 256, 8192) // tokens)), tokens=tokens, dtype=dtype)
    if kind == "kv_attention":
        batch = _log(rng, 1, 64)
        return dict(kind=kind, heads=32, kv_heads=rng.choice([32, 8]), head_dim=rng.choice([64, 128, 128]), batch=batch,
                    context=_log(rng, 20, min(8192, 65536 // batch)), dtype=dtype)
    ratio = rng.uniform(0.35, 0.8)      # of the parameters: ranks as the compression leaves them, or rounded to whole tiles
    shape = rng.choice([WIDE, WIDE, GROUPED, MIDDLE])
    attn = llama.lowrank_rank(shape["hidden"], shape["hidden"], ratio)
    mlp = llama.lowrank_rank(shape["inter"], shape["hidden"], ratio)
    tile = rng.choice([1, 64, 64, 128])
    attn, mlp = (max(tile, r // tile * tile) for r in (attn, mlp))
    if kind == "mlp":
        return dict(kind=kind, hidden=shape["hidden"], inter=shape["inter"], mlp_rank=mlp, batch=_log(rng, 1, 64), dtype=dtype)
    cache = rng.choice(["dense", "dense", "rank"])
    if cache == "rank":
        attn = attn // 8 * 8            # the rank-space cache takes ranks of whole 16-byte pieces
    case = dict(kind=kind, **shape, layers=rng.randint(1, 3), attn_rank=attn, mlp_rank=mlp, int4=False, dtype=dtype, cache=cache)
    if kind == "token":
        batch = rng.choice([1, 1, _log(rng, 2, 64)])
        int4 = cache == "dense" and batch <= 16 and rng.random() < 0.3
        if int4:
            case.update(attn_rank=max(256, attn // 256 * 256), mlp_rank=max(256, mlp // 256 * 256), inter=shape["inter"] // 256 * 256)
        return dict(case, int4=int4, batch=batch, tokens=1, context=_log(rng, 16, min(4096, 65536 // batch)))
    batch = rng.choice([1, 1, 2, 4])
    tokens = _log(rng, 17, (3000 if attn % 8 == 0 else 600) // batch)
    return dict(case, batch=batch, tokens=tokens, context=rng.choice([0, 0, _log(rng, 16, 1024)]))


# ---- what a program has in hand before the call ----------------------------------------------------------------------
def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return gen


def _normal(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(dtype)


def _int4_factors(model, gen, dtype):
    """Every factor as a group-wise int4 module, its packed buffers filled as if read from a checkpoint."""
    for name in quant.factor_linear_names(model):
        lin = quant.get_submodule(model, name)
        mod = quant.PackedQuantLinear(in_features=lin.in_features, out_features=lin.out_features, bits=4, group_size=128, bias=False,
                                      compute_dtype=dtype).to("cuda")
        mod.qweight.random_(0, 256, generator=gen)
        # sixteen levels around 7.5 with a spread of 4.6 levels: a scale near 0.02 / 4.6 keeps the weights' deviation
        mod.scales.copy_(STD / 4.6 * (0.9 + 0.2 * torch.rand(mod.scales.shape, generator=gen, device="cuda")))
        mod.zeros.random_(7, 9, generator=gen)
        quant.set_submodule(model, name, mod)
    for layer in model.model.layers:
        layer.self_attn._reset_runtime_state()


def _model(case, seed, gen):
    dtype = DTYPES[case["dtype"]]
    model = llama.build_model(hidden_size=case["hidden"], num_heads=case["heads"], num_kv_heads=case["kv_heads"],
                              head_dim=case["head_dim"], intermediate_size=case["inter"], num_layers=case["layers"],
                              vocab_size=case["vocab"], attn_rank=case["attn_rank"], mlp_rank=case["mlp_rank"],
                              max_position_embeddings=8192)
    model = llama.materialize(model, "cuda", dtype, seed=seed, std=STD)
    if case["int4"]:
        _int4_factors(model, gen, dtype)
    return model


def _cache(case, model, gen):
    """The cache of the case's sequences, its first ``context`` rows filled, and the storage of all layers as two tensors."""
    dtype = DTYPES[case["dtype"]]
    length = case["context"] + case["tokens"] + 8
    if case["cache"] == "rank":
        cache = FlashSVDLegacySparseKVCache(model.config, max_batch_size=case["batch"], max_cache_len=length, device="cuda", dtype=dtype)
        row = (case["attn_rank"],)
    else:
        cache = FlashSVDV15DenseKVCache(model.config, max_batch_size=case["batch"], max_cache_len=length, device="cuda", dtype=dtype)
        row = (case["kv_heads"], case["head_dim"])
    keys = torch.zeros(case["layers"], case["batch"], length, *row, dtype=dtype, device="cuda")
    values = torch.zeros_like(keys)
    # coefficients of a normalised hidden state; keys and values are one factor further on
    std = STD * math.sqrt(case["hidden"])
    if case["cache"] != "rank":
        std *= STD * math.sqrt(case["attn_rank"])
    for i in range(case["layers"]):
        if case["context"]:
            keys[i, :, : case["context"]] = _normal(gen, case["batch"], case["context"], *row, std=std, dtype=dtype)
            values[i, :, : case["context"]] = _normal(gen, case["batch"], case["context"], *row, std=std, dtype=dtype)
        cache.key_cache[i], cache.value_cache[i] = keys[i], values[i]
    cache._seen_tokens = case["context"]
    return cache, keys, values


@torch.no_grad()
def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    dtype = DTYPES[case["dtype"]]
    if kind in ("token", "prompt"):
        model = _model(case, seed, gen)
        cache, keys, values = _cache(case, model, gen)
        first, last = case["context"], case["context"] + case["tokens"]
        state = dict(kind=kind, model=model, cache=cache, keys=keys[:, :, first:last], values=values[:, :, first:last])
        ids = torch.randint(0, case["vocab"], (case["batch"], case["tokens"]), generator=gen, device="cuda")
        if kind == "prompt":
            return dict(state, ids=ids, positions=torch.arange(first, last))
        engine = make_persistent_decoder(model, cache, case["batch"])
        if engine is None:
            engine = GraphedDecoder(model, cache, case["batch"])
            engine.set_state(ids, first)
            engine.capture()
            return dict(state, engine=engine, ids=ids, position=first)
        return dict(state, engine=engine, ids=int(ids), position=first)
    batch = case["batch"]
    if kind == "mlp":
        r, d, n = case["mlp_rank"], case["inter"], case["hidden"]
        std = STD * math.sqrt(n)
        return dict(kind=kind, up=_normal(gen, batch, 1, r, std=std, dtype=dtype), gate=_normal(gen, batch, 1, r, std=std, dtype=dtype),
                    weights=[_normal(gen, *s, std=STD, dtype=dtype) for s in ((r, d), (r, d), (d, r), (r, n))])
    H, Hk, Dh = case["heads"], case["kv_heads"], case["head_dim"]
    if kind == "attend":
        M, r = case["tokens"], case["attn_rank"]
        attention = FlashSVDRoPEAttention(H, Dh, llama.LlamaRotaryEmbedding(Dh, 8192, device="cuda"))
        std = STD * math.sqrt(H * Dh)
        p = [_normal(gen, batch, 1, M, r, std=std, dtype=dtype).expand(batch, h, M, r) for h in (H, Hk, Hk)]
        v = [_normal(gen, h, r, Dh, std=STD, dtype=dtype) for h in (H, Hk, Hk)]
        lengths = torch.randint(max(1, M // 2), M + 1, (batch, 1), generator=gen, device="cuda")
        positions = torch.arange(M, device="cuda").unsqueeze(0)
        mask = (positions < lengths).to(torch.int64)
        return dict(kind=kind, attention=attention, factors=QKVFactors(*p, *v), mask=mask, positions=positions)
    S = case["context"] + 8
    cos, sin = (t[0, 0, :, : Dh // 2].contiguous()
                for t in llama.LlamaRotaryEmbedding(Dh, 8192, device="cuda")(torch.empty(1, dtype=dtype, device="cuda"), seq_len=S))
    keys = _normal(gen, batch, S, Hk, Dh, dtype=dtype)
    values = _normal(gen, batch, S, Hk, Dh, dtype=dtype)
    # sequences of a batch differ in length, the longest one fills the context
    lens = torch.randint(max(1, case["context"] * 3 // 4), case["context"] + 1, (batch,), generator=gen, device="cuda", dtype=torch.int32)
    lens[0] = case["context"]
    return dict(kind=kind, q=_normal(gen, batch, 1, H, Dh, dtype=dtype), k=_normal(gen, batch, 1, Hk, Dh, dtype=dtype),
                v=_normal(gen, batch, 1, Hk, Dh, dtype=dtype), keys=keys, values=values, lens=lens, cos=cos, sin=sin)


# ---- one pass -----------------------------------------------------------------------------------------------------------
@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "token":
        engine = state["engine"]
        engine.set_state(state["ids"], state["position"])
        if isinstance(engine, PersistentDecoder):
            engine.step_token()
        else:
            engine.step()
        return dict(logits=engine.logits, keys=state["keys"], values=state["values"])
    if kind == "prompt":
        out = state["model"](state["ids"], past_key_values=state["cache"], cache_position=state["positions"], logits_to_keep=1)
        return dict(logits=out.logits, hidden=out.hidden_states, keys=state["keys"], values=state["values"])
    if kind == "attend":
        return state["attention"](state["factors"], state["mask"], state["positions"])
    if kind == "mlp":
        return flashsvd_mlp_dual_split_triton_v2(state["up"], state["gate"], *state["weights"])
    fn = decode_registry.get_flash_attn_with_kvcache()
    out = decode_registry.call_flash_attn_with_kvcache(
        fn, state["q"], state["keys"], state["values"], k_bmhd=state["k"], v_bmhd=state["v"], cache_seqlens=state["lens"],
        rotary_cos=state["cos"], rotary_sin=state["sin"], causal=True)
    return dict(out=out, keys=state["keys"], values=state["values"])


# ---- what one pass cannot do without ----------------------------------------------------------------------------------------
def work(case):
    kind, B = case["kind"], case["batch"]
    if kind == "mlp":
        r, d, n = case["mlp_rank"], case["inter"], case["hidden"]
        factors = r * (3 * d + n)
        return dict(bytes=2 * (factors + B * (2 * r + n)), flops=2 * B * factors)
    H, Hk, Dh = case["heads"], case["kv_heads"], case["head_dim"]
    if kind == "kv_attention":
        keys = B * (case["context"] * 7 // 8 + 1)
        return dict(bytes=2 * (2 * keys * Hk * Dh + 2 * B * (H + Hk) * Dh), flops=4 * keys * H * Dh)
    r, M = case["attn_rank"], case["tokens"]
    if kind == "attend":
        rows = B * M
        return dict(bytes=2 * (3 * rows * r + (H + 2 * Hk) * Dh * r + rows * H * Dh),
                    flops=2 * rows * (H + 2 * Hk) * Dh * r + 4 * B * H * Dh * M * (M + 1) // 2)
    d, D, rm, L, C = case["hidden"], case["inter"], case["mlp_rank"], case["layers"], case["context"]
    rows = B * M
    factors = r * (3 * d + (H + 2 * Hk) * Dh + H * Dh + d) + 3 * rm * (d + D)       # per layer
    per_factor = 0.5 + 4 / 128 if case["int4"] else 2.0
    head = case["vocab"] * d
    kept = 2 * r if case["cache"] == "rank" else 2 * Hk * Dh                            # cached values of one token
    pairs = B * (M * C + M * (M + 1) // 2)                                              # query-key pairs under the causal mask
    nbytes = L * (factors * per_factor + 2 * kept * B * (C + M)) + 2 * (head + B * case["vocab"] + 2 * rows * d)
    flops = L * (2 * rows * factors + 4 * pairs * H * Dh) + 2 * B * head
    if case["cache"] == "rank" and C:
        flops += L * 2 * B * C * Hk * Dh * r                                            # keys of the context from their coefficients
        if kind == "prompt":
            flops += L * 2 * B * C * Hk * Dh * r                                        # and its values
        else:
            flops += L * (2 * B * C * H * r - 2 * B * C * H * Dh)                       # weights times value coefficients
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """Four times what a case differs from itself when every sum runs in another order (hidden, rank and intermediate axes
    of all factors permuted; cached keys permuted; int4: the two decode engines against each other).

    A model rounds to 16 bits after every operator and each layer hands its flipped roundings on, so the difference grows
    with the square root of the depth.  Measured in bf16: rel 0.004 to 0.010 at one layer, 0.012 at two to four, 0.024 at
    eight, 0.046 at thirty-two, the largest element 0.05 at two, 0.14 at eight, 0.25 at thirty-two; in fp16 an eighth of
    that.  The single operators round once or twice: prompt attention rel 1.9e-4 (largest element 0.011), decode attention
    3e-5 (0.005), the MLP 6.5e-4 (0.008)."""
    if case["kind"] in ("token", "prompt"):
        depth = math.sqrt(case["layers"])
        if case["dtype"] == "fp16":
            return {"rel": 0.004 * depth, "max": 0.02 * depth}
        return {"rel": 0.032 * depth, "max": min(0.95, 0.18 * depth)}
    rel, most = {"attend": (8e-4, 0.04), "kv_attention": (2e-4, 0.02), "mlp": (2.6e-3, 0.03)}[case["kind"]]
    return {"rel": rel, "max": most}
