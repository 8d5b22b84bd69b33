"""The work that this framework is measured on: what one serving step asks of it, through its public entry points.

Twelve listed cases and, from `draw`, more of the same ranges.  A kind of case is one piece of a step:

step      a decode step of a whole dense model through `Engine.forward_logits` (metadata, captured graph, logits)
decode    paged attention of a decode batch through `HipAttnBackend.forward` (store K / V, attend)
prefill   the same entry point with a portion of new tokens per request, with or without cached tokens before it
sample    the token draw of a batch with temperature, top-k and top-p
latent    latent attention of a hybrid decoder: prompt portions, decoded tokens
experts   a routed feed-forward: router, bucketing, both segmented products with the gate between them
window    sliding-window attention whose heads' scores are mixed before the softmax
delta     the gated delta-rule recurrence, fp32 state per request
maps      the difference of two softmax maps, with a window and kept first tokens or over all keys

Sizes are those of the presets in model.py (Qwen3-0.6B / 14B / 32B head counts), of the reference's offline benchmark (256 sequences of
100 - 1024 tokens, chunks of up to 16384) and of the hybrid decoders' benchmarks under tools/.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch
import torch.nn.functional as F

DEV = "cuda:0"
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one user, one token: the smallest model of the benchmark, the reference's default page size
        {"name": "step 0.6B x1", "kind": "step", "model": "qwen3-0.6b", "batch": 1, "lo": 533, "hi": 533, "page": 1},
        # the headline decode batch: 256 sequences at the benchmark's context lengths, Qwen3-14B heads
        {"name": "decode 14B x256", "kind": "decode", "heads": 40, "kv_heads": 8, "batch": 256, "lo": 100, "hi": 2000, "page": 256, "dtype": "bf16"},
        # one full chunk of the benchmark's prompts (100 - 1024 tokens each, 16384 in all), nothing cached
        {"name": "prefill 14B chunk", "kind": "prefill", "heads": 40, "kv_heads": 8, "batch": 29, "new_lo": 100, "new_hi": 1024, "old": 0,
         "page": 256, "dtype": "bf16"},
        # a chunk of one long document, the chunks before it in the cache, Qwen3-32B heads
        {"name": "prefill 32B long", "kind": "prefill", "heads": 64, "kv_heads": 8, "batch": 1, "new_lo": 8192, "new_hi": 8192, "old": 16384,
         "page": 256, "dtype": "bf16"},
        # the draw of a busy server's step: every row with top-k and top-p, the Qwen3 vocabulary
        {"name": "sample x64", "kind": "sample", "batch": 64, "vocab": 151936, "top_k": True, "top_p": True},
        # latent attention at the hybrid benchmark's size m: a prompt portion, then a decode batch
        {"name": "latent prompt", "kind": "latent", "batch": 4, "new_lo": 1500, "new_hi": 2548, "old": 0, "heads": 16, "rank": 512, "rot": 64, "sink": False},
        {"name": "latent decode x32", "kind": "latent", "batch": 32, "new_lo": 1, "new_hi": 1, "old": 4096, "heads": 16, "rank": 512, "rot": 64, "sink": False},
        # the routed feed-forward of size m of the group-limited sigmoid router: a prompt portion, then a decode batch
        {"name": "experts prompt", "kind": "experts", "tokens": 8192, "width": 2048, "experts": 64, "top": 6, "groups": 8, "keep": 4, "ff": 512},
        {"name": "experts decode x32", "kind": "experts", "tokens": 32, "width": 2048, "experts": 64, "top": 6, "groups": 8, "keep": 4, "ff": 512},
        # mixed-head attention at size m, a portion of prompts of uneven length
        {"name": "window prompt", "kind": "window", "batch": 4, "new_lo": 1500, "new_hi": 2548, "old": 0, "heads": 16, "kv_heads": 4, "window": 2048},
        # the delta rule at size m with a decay per key channel, the same portion
        {"name": "delta prompt", "kind": "delta", "batch": 4, "new_lo": 1500, "new_hi": 2548, "old": 0, "heads": 16, "per_channel": True},
        # two softmax maps of half the head size over the values of a whole head, all earlier keys, the same portion
        {"name": "maps prompt", "kind": "maps", "batch": 4, "new_lo": 1500, "new_hi": 2548, "old": 0, "heads": 16, "kv_heads": 4, "window": 0, "keep": 0,
         "gate": False},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng: random.Random):
    kind = rng.choice(["step", "decode", "prefill", "prefill", "sample", "latent", "latent", "experts", "experts", "window", "delta", "maps"])
    if kind == "step":
        lo = _log(rng, 16, 2000)
        return {"kind": kind, "model": "qwen3-0.6b", "batch": _log(rng, 1, 8), "lo": lo, "hi": min(2000, lo + _log(rng, 1, 1000)),
                "page": rng.choice([1, 16, 256])}
    heads, kv = rng.choice([(16, 8), (40, 8), (64, 8), (10, 2), (16, 2), (5, 1)])  # whole models and shards of them
    if kind == "decode":
        lo = _log(rng, 10, 2000)
        return {"kind": kind, "heads": heads, "kv_heads": kv, "batch": _log(rng, 1, 256), "lo": lo, "hi": min(2000, lo + _log(rng, 1, 1900)),
                "page": rng.choice([1, 16, 256]), "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "prefill":
        batch = _log(rng, 1, 32)
        lo = _log(rng, 2, 8000 // batch)
        return {"kind": kind, "heads": heads, "kv_heads": kv, "batch": batch, "new_lo": lo, "new_hi": min(12000 // batch, lo + _log(rng, 1, 1000)),
                "old": rng.choice([0, _log(rng, 1, 8000 // batch)]), "page": rng.choice([1, 16, 256]), "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "sample":
        flags = rng.choice([(True, True), (True, False), (False, True), (False, False)])
        return {"kind": kind, "batch": _log(rng, 1, 256), "vocab": rng.choice([151936, 128256, _log(rng, 32000, 152000)]), "top_k": flags[0], "top_p": flags[1]}
    if kind == "experts":
        experts, groups, keep = rng.choice([(64, 8, 4), (32, 4, 2), (16, 4, 2), (16, 1, 1)])
        return {"kind": kind, "tokens": _log(rng, 1, 8000), "width": rng.choice([1024, 2048]), "experts": experts, "top": rng.randint(1, 6),
                "groups": groups, "keep": keep, "ff": rng.choice([512, 768, 1024])}
    # the sequence mixers: a decode batch, or portions of prompts, fresh or continued
    if rng.random() < 0.3:
        size = {"batch": _log(rng, 1, 64), "new_lo": 1, "new_hi": 1, "old": _log(rng, 16, 4096)}
    else:
        batch = _log(rng, 1, 8)
        lo = _log(rng, 2, 6000 // batch)
        size = {"batch": batch, "new_lo": lo, "new_hi": min(8000 // batch, lo + _log(rng, 1, 1000)), "old": rng.choice([0, 0, _log(rng, 1, 2000)])}
    if kind == "latent":
        rank, rot = rng.choice([(512, 64), (256, 64)])
        return {"kind": kind, **size, "heads": rng.choice([8, 16]), "rank": rank, "rot": rot, "sink": rng.random() < 0.5}
    if kind == "window":
        return {"kind": kind, **size, "heads": 16, "kv_heads": 4, "window": rng.choice([512, 1024, 2048])} if rng.random() < 0.6 else \
            {"kind": kind, **size, "heads": 8, "kv_heads": 2, "window": rng.choice([512, 1024])}
    if kind == "delta":
        return {"kind": kind, **size, "heads": rng.choice([8, 16]), "per_channel": rng.random() < 0.5}
    window = rng.choice([0, 0, 1024, 2048])
    return {"kind": kind, **size, "heads": rng.choice([8, 16]), "kv_heads": rng.choice([2, 4]), "window": window, "keep": 64 if window else 0,
            "gate": rng.random() < 0.5}


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed: int, salt: int = 0) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + salt)


def _rnd(g: torch.Generator, *shape, dtype=BF16, std: float = 1.0, mean: float = 0.0) -> torch.Tensor:
    return (torch.randn(shape, generator=g, device=DEV, dtype=F32) * std + mean).to(dtype)


def _lengths(case: dict):
    """(new tokens, cached tokens) per request: spread evenly from lo to hi in an order that stays the same for a case."""
    n = case["batch"]
    if case["kind"] in ("step", "decode"):
        lens = [case["lo"] + round((case["hi"] - case["lo"]) * i / max(1, n - 1)) for i in range(n)]
        random.Random(n).shuffle(lens)
        return [1] * n, [k - 1 for k in lens]
    new = [case["new_lo"] + round((case["new_hi"] - case["new_lo"]) * i / max(1, n - 1)) for i in range(n)]
    random.Random(n).shuffle(new)
    return new, [case["old"]] * n


def _pages(seed: int, lens, page: int):
    """(token slots per request, pages in all): every request's pages drawn from a shuffled free list, as on a server that has run for a while."""
    need = [-(-k // page) for k in lens]
    order = np.random.default_rng(seed).permutation(sum(need)).astype(np.int64)
    slots, at = [], 0
    for k, n in zip(lens, need):
        s = (order[at: at + n, None] * page + np.arange(page)[None, :]).reshape(-1)[:k]
        slots.append(torch.from_numpy(s).to(DEV))
        at += n
    return slots, sum(need)


def _requests(new, old):
    from mini_sglang_amd.core import Req

    return [Req(input_ids=torch.zeros(k + n, dtype=torch.int32), table_idx=i, cached_len=k, output_len=8, uid=i) for i, (n, k) in enumerate(zip(new, old))]


def _table(slots, rows: int) -> torch.Tensor:
    width = -(-max(s.numel() for s in slots) // 32) * 32
    table = torch.zeros((rows, width), dtype=torch.int32, device=DEV)
    for i, s in enumerate(slots):
        table[i, : s.numel()] = s.to(torch.int32)
    return table


def _batch(reqs, phase: str, slots, new, old):
    from mini_sglang_amd.core import Batch

    batch = Batch(reqs=reqs, phase=phase)
    batch.positions = torch.cat([torch.arange(k, k + n, dtype=torch.int32, device=DEV) for n, k in zip(new, old)])
    batch.out_loc = torch.cat([s[k: k + n] for s, n, k in zip(slots, new, old)]).to(torch.int32)
    return batch


def _hybrid(case: dict, seed: int, config):
    """Context, cache and metadata of one step of a hybrid decoder, as its engine builds them."""
    from mini_sglang_amd.attention import MixAttnBackend
    from mini_sglang_amd.core import Context
    from mini_sglang_amd.kvcache import create_kvcache_pool

    new, old = _lengths(case)
    slots, pages = _pages(seed, [a + b for a, b in zip(new, old)], 16)
    ctx = Context(16)
    ctx.page_table = _table(slots, len(new) + 1)
    ctx.kv_cache = create_kvcache_pool(config, pages + 1, 16, BF16, torch.device(DEV), state_rows=len(new) + 1)
    ctx.attn_backend = MixAttnBackend(config, ctx)
    batch = _batch(_requests(new, old), "prefill", slots, new, old)
    ctx.attn_backend.prepare_metadata(batch)
    return {"ctx": ctx, "batch": batch, "slots": slots, "new": new, "old": old, "T": sum(new)}


def _pairs(case: dict) -> int:
    """Visible (query token, key) pairs of a case."""
    new, old = _lengths(case)
    window, keep = case.get("window", 0), case.get("keep", 0)
    total = 0
    for n, k in zip(new, old):
        seen = np.arange(k + 1, k + n + 1, dtype=np.int64)
        total += int((np.minimum(seen, window) + np.minimum(np.maximum(seen - window, 0), keep)).sum() if window else seen.sum())
    return total


def _keys(case: dict) -> int:
    """Key rows that a case has to read: a window hides the oldest ones."""
    new, old = _lengths(case)
    window, keep = case.get("window", 0), case.get("keep", 0)
    return sum(min(n + k, n - 1 + window + keep) if window else n + k for n, k in zip(new, old))


def _new_rows(x: torch.Tensor, s: dict):
    """Rows of [T, ...] per request."""
    return torch.split(x, s["new"])


# ------------------------------------------------------------------------------------------------ a decode step of a whole dense model
def _step_weights(m, seed: int):
    g = _gen(seed)
    H, D, I = m.hidden_size, m.head_dim, m.intermediate_size
    w = {"model.embed_tokens.weight": _rnd(g, m.vocab_size, H, std=0.2), "model.norm.weight": _rnd(g, H, std=0.05, mean=0.5)}
    for i in range(m.num_layers):
        p = f"model.layers.{i}."
        for n in ("input_layernorm", "post_attention_layernorm"):
            w[p + n + ".weight"] = _rnd(g, H, std=0.1, mean=1.0)
        for n, rows, cols in (("self_attn.q_proj", m.num_qo_heads * D, H), ("self_attn.k_proj", m.num_kv_heads * D, H), ("self_attn.v_proj", m.num_kv_heads * D, H),
                              ("self_attn.o_proj", H, m.num_qo_heads * D), ("mlp.gate_proj", I, H), ("mlp.up_proj", I, H), ("mlp.down_proj", H, I)):
            # what a layer adds to the stream is kept small beside it, as in a trained model
            w[p + n + ".weight"] = _rnd(g, rows, cols, std=0.02 if rows != H else 0.02 * (2 * m.num_layers) ** -0.5)
        for n in ("q_norm", "k_norm"):
            w[p + f"self_attn.{n}.weight"] = _rnd(g, D, std=0.1, mean=1.0)
    return w


def _step_cached(m, total: int, seed: int, layer: int):
    """What the cache holds of the earlier tokens of all requests: unit-sized keys, values as small as this model's."""
    g = _gen(seed, 1 + layer)
    return _rnd(g, total, m.num_kv_heads, m.head_dim), _rnd(g, total, m.num_kv_heads, m.head_dim, std=0.6)


def _step_ids(m, case: dict, seed: int):
    return torch.randint(0, m.vocab_size, (case["batch"],), generator=_gen(seed, 777), device=DEV, dtype=torch.int32)


def _prepare_step(case: dict, seed: int):
    from mini_sglang_amd.engine import Engine, EngineConfig
    from mini_sglang_amd.model import PRESETS

    m, B, page = PRESETS[case["model"]], case["batch"], case["page"]
    new, old = _lengths(case)
    slots, pages = _pages(seed, [k + 1 for k in old], page)
    eng = Engine(EngineConfig(model=m, max_running_req=B, cuda_graph_bs=[B], page_size=page, num_page_override=max(pages, -(-max(old) // page) + 1),
                              max_seq_len_override=max(old) + 1), torch.device(DEV))
    eng.model.load_hf_state(_step_weights(m, seed))
    table = _table(slots, B + 1)
    eng.page_table[:B, : table.shape[1]] = table[:B, : eng.page_table.shape[1]]
    where = torch.cat([s[:k] for s, k in zip(slots, old)])
    for i in range(m.num_layers):
        k, v = _step_cached(m, sum(old), seed, i)
        eng.kv_cache.k_tokens(i)[where], eng.kv_cache.v_tokens(i)[where] = k, v
    ids = _step_ids(m, case, seed)
    return {"eng": eng, "reqs": _requests(new, old), "slots": slots, "new": new, "old": old, "ids": ids, "batch": _batch(_requests(new, old), "decode", slots, new, old)}


def _run_step(case: dict, s: dict):
    from mini_sglang_amd.core import Batch

    eng = s["eng"]
    for r, k in zip(s["reqs"], s["old"]):  # the same token of the same requests again
        r.cached_len = k
    batch = Batch(reqs=s["reqs"], phase="decode")
    eng.graph_runner.pad_batch(batch)
    batch.input_ids, batch.positions, batch.out_loc = s["ids"], s["batch"].positions, s["batch"].out_loc
    eng.attn_backend.prepare_metadata(batch)
    return eng.forward_logits(batch)


def _exact_step(case: dict, seed: int):
    from mini_sglang_amd.model import PRESETS  # sizes only

    m = PRESETS[case["model"]]
    w = _step_weights(m, seed)
    _, old = _lengths(case)
    B, D, Hq, Hk = case["batch"], m.head_dim, m.num_qo_heads, m.num_kv_heads

    def norm(x, weight):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + m.rms_norm_eps) * weight.to(F64)

    pos = torch.tensor(old, dtype=F64, device=DEV)
    ang = pos[:, None] * (m.rope_base ** (-2.0 * torch.arange(D // 2, dtype=F64, device=DEV) / D))[None, :]

    def rot(x):
        a, b = x[..., : D // 2], x[..., D // 2:]
        c, sn = ang.cos()[:, None, :], ang.sin()[:, None, :]
        return torch.cat([a * c - b * sn, b * c + a * sn], dim=-1)

    x = w["model.embed_tokens.weight"][_step_ids(m, case, seed).long()].to(F64)
    for i in range(m.num_layers):
        p = f"model.layers.{i}."

        def lin(h, n):
            return h @ w[p + n + ".weight"].to(F64).T

        h = norm(x, w[p + "input_layernorm.weight"])
        q = rot(norm(lin(h, "self_attn.q_proj").view(B, Hq, D), w[p + "self_attn.q_norm.weight"]))
        k = rot(norm(lin(h, "self_attn.k_proj").view(B, Hk, D), w[p + "self_attn.k_norm.weight"]))
        v = lin(h, "self_attn.v_proj").view(B, Hk, D)
        kc, vc = _step_cached(m, sum(old), seed, i)
        out, at = [], 0
        for b, n in enumerate(old):
            kk, vv = torch.cat([kc[at: at + n].to(F64), k[b: b + 1]]), torch.cat([vc[at: at + n].to(F64), v[b: b + 1]])
            at += n
            sc = torch.matmul(q[b].view(Hk, Hq // Hk, D), kk.permute(1, 2, 0).contiguous()) * D ** -0.5
            out.append(torch.matmul(torch.softmax(sc, dim=-1), vv.permute(1, 0, 2).contiguous()).reshape(Hq * D))
        x = x + lin(torch.stack(out), "self_attn.o_proj")
        h = norm(x, w[p + "post_attention_layernorm.weight"])
        x = x + lin(F.silu(lin(h, "mlp.gate_proj")) * lin(h, "mlp.up_proj"), "mlp.down_proj")
    return norm(x, w["model.norm.weight"]) @ w["model.embed_tokens.weight"].to(F64).T


def _work_step(case: dict):
    from mini_sglang_amd.model import PRESETS

    m = PRESETS[case["model"]]
    _, old = _lengths(case)
    layer = m.hidden_size * ((2 * m.num_qo_heads + 2 * m.num_kv_heads) * m.head_dim + 3 * m.intermediate_size)
    params = m.num_layers * layer + m.vocab_size * m.hidden_size
    row = m.num_layers * m.num_kv_heads * m.head_dim * 2
    return {"bytes": 2 * params + 2 * row * (sum(old) + 2 * len(old)) + 2 * len(old) * m.vocab_size,
            "flops": 2 * len(old) * params + 4 * m.num_layers * m.num_qo_heads * m.head_dim * (sum(old) + len(old))}


# ------------------------------------------------------------------------------------------------ paged attention: decode, prefill
def _paged_inputs(case: dict, seed: int):
    """q, k, v of the new tokens and what the pool holds of the earlier ones, row after row."""
    new, old = _lengths(case)
    g, dt = _gen(seed), torch.float16 if case["dtype"] == "fp16" else BF16
    T, Hq, Hk = sum(new), case["heads"], case["kv_heads"]
    return (_rnd(g, T, Hq, 128, dtype=dt), _rnd(g, T, Hk, 128, dtype=dt), _rnd(g, T, Hk, 128, dtype=dt), _rnd(g, sum(old), Hk, 128, dtype=dt),
            _rnd(g, sum(old), Hk, 128, dtype=dt))


def _prepare_paged(case: dict, seed: int):
    from mini_sglang_amd.attention import HipAttnBackend
    from mini_sglang_amd.core import Context
    from mini_sglang_amd.kvcache import create_kvcache_pool
    from mini_sglang_amd.model import ModelConfig

    q, k, v, kc, vc = _paged_inputs(case, seed)
    new, old = _lengths(case)
    slots, pages = _pages(seed, [a + b for a, b in zip(new, old)], case["page"])
    m = ModelConfig(num_layers=1, num_qo_heads=case["heads"], num_kv_heads=case["kv_heads"], head_dim=128, hidden_size=128 * case["heads"], vocab_size=1024,
                    intermediate_size=1024)
    ctx = Context(case["page"])
    ctx.page_table = _table(slots, len(new) + 1)
    ctx.kv_cache = create_kvcache_pool(m, pages + 1, case["page"], q.dtype, torch.device(DEV))
    where = torch.cat([s[:n] for s, n in zip(slots, old)])
    ctx.kv_cache.k_tokens(0)[where], ctx.kv_cache.v_tokens(0)[where] = kc, vc
    backend = HipAttnBackend(m, ctx)
    batch = _batch(_requests(new, old), case["kind"], slots, new, old)
    backend.prepare_metadata(batch)
    return {"backend": backend, "batch": batch, "q": q, "k": k.view(k.shape[0], -1), "v": v.view(v.shape[0], -1)}


def _run_paged(case: dict, s: dict):
    return s["backend"].forward(s["q"], s["k"], s["v"], 0, s["batch"])


def _exact_paged(case: dict, seed: int):
    q, k, v, kc, vc = _paged_inputs(case, seed)
    new, old = _lengths(case)
    Hq, Hk, out, a, b = case["heads"], case["kv_heads"], [], 0, 0
    for n, c in zip(new, old):
        kk, vv = torch.cat([kc[b: b + c], k[a: a + n]]).to(F64), torch.cat([vc[b: b + c], v[a: a + n]]).to(F64)
        o = torch.empty((n, Hq, 128), dtype=F64, device=DEV)
        hidden = torch.arange(c + n, device=DEV)[None, :] > torch.arange(c, c + n, device=DEV)[:, None]
        for h in range(Hq):
            j = h // (Hq // Hk)
            sc = (q[a: a + n, h].to(F64) @ kk[:, j].T) * 128 ** -0.5
            o[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), dim=-1) @ vv[:, j]
        out.append(o)
        a, b = a + n, b + c
    return torch.cat(out)


def _work_paged(case: dict):
    new, old = _lengths(case)
    T, Hq, Hk = sum(new), case["heads"], case["kv_heads"]
    return {"bytes": 2 * 128 * (2 * T * Hq + 2 * Hk * (2 * T + sum(old))) + 4 * (T + sum(old)), "flops": 4 * Hq * 128 * _pairs(case)}


# ------------------------------------------------------------------------------------------------ the token draw
def _prepare_sample(case: dict, seed: int):
    from mini_sglang_amd import flashinfer_compat as fi

    g, B, V = _gen(seed), case["batch"], case["vocab"]
    torch.manual_seed(seed)  # the draws' key, as an engine sets it once for all its ranks
    # logits as a trained model's: most of the mass on some tens of tokens
    logits = _rnd(g, B, V, std=2.5)
    u = torch.rand((3, B), generator=g, device=DEV)
    top_k = (10 + 90 * u[1]).to(torch.int32) if case["top_k"] else None
    top_p = 0.7 + 0.28 * u[2] if case["top_p"] else None
    return {"draw": type(fi.sampling)(), "logits": logits, "temperature": 0.4 + 0.6 * u[0], "top_k": top_k, "top_p": top_p}


def _run_sample(case: dict, s: dict):
    d = s["draw"]
    probs = d.softmax(s["logits"], s["temperature"])
    if s["top_k"] is None and s["top_p"] is None:
        return d.sampling_from_probs(probs)
    if s["top_p"] is None:
        return d.top_k_sampling_from_probs(probs, s["top_k"])
    if s["top_k"] is None:
        return d.top_p_sampling_from_probs(probs, s["top_p"])
    return d.top_k_top_p_sampling_from_probs(probs, s["top_k"], s["top_p"])


def _work_sample(case: dict):
    n = case["batch"] * case["vocab"]
    return {"bytes": 2 * n + 16 * case["batch"], "flops": 4 * n}


# ------------------------------------------------------------------------------------------------ latent attention
def _latent_config(case: dict):
    from mini_sglang_amd.hybrid import HybridConfig

    mixer = {"heads": case["heads"], "dim": 128, "rot_dim": case["rot"], "vdim": 128, "kv_rank": case["rank"], "scale": (128 + case["rot"]) ** -0.5,
             "rot": {"base": 1e6, "dims": case["rot"], "scaling": {"factor": 8.0, "fast": 32.0, "original": 4096, "slow": 1.0}}}
    return HybridConfig.from_json({"architecture": "Nidorax", "layers": [{"type": "latent_attention", "mixer": mixer}], "norm": {"eps": 1e-6}, "postln_alpha": 2.0,
                                   "vocab": 1024, "width": 1024})


def _latent_inputs(case: dict, seed: int):
    new, old = _lengths(case)
    g, n = _gen(seed), case["rank"] + case["rot"]
    # queries carried into latent space: scores of about 1.5 before the softmax
    q = _rnd(g, sum(new), case["heads"], n, dtype=F32, std=1.5 / (n ** 0.5 * (128 + case["rot"]) ** -0.5))
    return q, _rnd(g, sum(new) + sum(old), n), _rnd(g, case["heads"], dtype=F32) if case["sink"] else None


def _prepare_latent(case: dict, seed: int):
    s = _hybrid(case, seed, _latent_config(case))
    s["q"], rows, s["sink"] = _latent_inputs(case, seed)
    s["ctx"].kv_cache.latent_rows(0)[torch.cat(s["slots"])] = rows
    return s


def _run_latent(case: dict, s: dict):
    from mini_sglang_amd import mixops

    md, ctx, H = s["batch"].attn_metadata, s["ctx"], case["heads"]
    out = torch.empty((s["T"], H, case["rank"]), dtype=F32, device=DEV)
    splits = mixops.latent_attn_splits(md.batch, s["T"], H, md.max_seqlen_k) if md.max_seqlen_q <= 16 else 1
    mixops.latent_attn(out, s["q"], ctx.kv_cache.latent_rows(0), ctx.page_table, md.req_rows, md.seq_lens, md.cu_seqlens_q, md.batch, case["rank"],
                       (128 + case["rot"]) ** -0.5, splits=splits, sink=s["sink"])
    return out


def _exact_latent(case: dict, seed: int):
    q, rows, sink = _latent_inputs(case, seed)
    new, old = _lengths(case)
    out, a, b = [], 0, 0
    for n, c in zip(new, old):
        kk = rows[b: b + c + n].to(F64)
        hidden = torch.arange(c + n, device=DEV)[None, :] > torch.arange(c, c + n, device=DEV)[:, None]
        o = torch.empty((n, case["heads"], case["rank"]), dtype=F64, device=DEV)
        for h in range(case["heads"]):
            sc = (q[a: a + n, h].to(F64) @ kk.T) * (128 + case["rot"]) ** -0.5
            sc = sc.masked_fill(hidden, -math.inf)
            if sink is not None:
                sc = torch.cat([sc, sink[h].to(F64).expand(n, 1)], dim=1)
            o[:, h] = torch.softmax(sc, dim=-1)[:, : c + n] @ kk[:, : case["rank"]]
        out.append(o)
        a, b = a + n, b + c + n
    return torch.cat(out)


def _work_latent(case: dict):
    new, _ = _lengths(case)
    H, R, r = case["heads"], case["rank"], case["rot"]
    return {"bytes": 2 * _keys(case) * (R + r) + 4 * sum(new) * H * (2 * R + r), "flops": 2 * _pairs(case) * H * (2 * R + r)}


# ------------------------------------------------------------------------------------------------ routed feed-forward
def _experts_inputs(case: dict, seed: int):
    g, W, E, ff = _gen(seed), case["width"], case["experts"], case["ff"]
    return {"h": _rnd(g, case["tokens"], W), "router": _rnd(g, E, W, std=W ** -0.5), "bias": _rnd(g, E, std=0.01), "up": _rnd(g, E, 2 * ff, W, std=W ** -0.5),
            "down": _rnd(g, E, W, ff, std=ff ** -0.5)}


def _run_experts(case: dict, s: dict):
    """A long portion or a decode batch of gated experts: choice, buckets, gate and up rows in one product, gate, down product."""
    from mini_sglang_amd import mixops

    T, W, E, top, ff = case["tokens"], case["width"], case["experts"], case["top"], case["ff"]
    ids, wts = mixops.route(s["h"], s["router"], s["bias"], top, case["groups"], case["keep"], sigmoid=True, group_best=2, scale=2.0)
    seg, perm = mixops.moe_sort(ids, E)
    gu = torch.empty((T * top, 2 * ff), dtype=BF16, device=DEV)
    mixops.gemm_nt(gu, s["h"], s["up"], T * top, 2 * ff, W, lda=W, ldb=W, ldc=2 * ff, groups=E, b_gs=2 * ff * W, seg=seg, a_rows=perm, a_div=top)
    act = mixops.silu_mul(gu)
    y = torch.empty((T, top, W), dtype=BF16, device=DEV)
    mixops.gemm_nt(y, act, s["down"], T * top, W, ff, lda=ff, ldb=ff, ldc=W, groups=E, b_gs=W * ff, seg=seg, c_rows=perm)
    return {"y": y, "ids": ids, "weights": wts}


def _exact_experts(case: dict, seed: int):
    s = _experts_inputs(case, seed)
    T, E, top, ff = case["tokens"], case["experts"], case["top"], case["ff"]
    h = s["h"].to(F64)
    score = torch.sigmoid(h @ s["router"].to(F64).T)
    pick = score + s["bias"].to(F64)
    per = pick.view(T, case["groups"], E // case["groups"])
    best = per.topk(min(2, per.shape[2]), dim=2).values.sum(dim=2).topk(case["keep"], dim=1).indices
    open_ = torch.zeros((T, case["groups"]), dtype=torch.bool, device=DEV).scatter_(1, best, True).repeat_interleave(E // case["groups"], dim=1)
    ids = pick.masked_fill(~open_, -math.inf).topk(top, dim=1).indices
    chosen = score.gather(1, ids)
    y = torch.empty((T, top, case["width"]), dtype=F64, device=DEV)
    for e in range(E):
        t, k = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            gu = h[t] @ s["up"][e].to(F64).T
            y[t, k] = (F.silu(gu[:, :ff]) * gu[:, ff:]) @ s["down"][e].to(F64).T
    return {"y": y, "ids": None, "weights": 2.0 * chosen / chosen.sum(dim=1, keepdim=True)}


def _work_experts(case: dict):
    T, W, E, top, ff = case["tokens"], case["width"], case["experts"], case["top"], case["ff"]
    used = E * (1.0 - (1.0 - top / E) ** T)  # experts that a batch is expected to touch
    return {"bytes": 2 * used * 3 * ff * W + 2 * T * W * (1 + top) + 2 * E * W + 8 * T * top, "flops": 2 * T * top * 3 * ff * W + 2 * T * E * W}


# ------------------------------------------------------------------------------------------------ mixed-head window attention
def _window_config(case: dict):
    from mini_sglang_amd.hybrid import bedarax_config

    mixer = {"heads": case["heads"], "kv_heads": case["kv_heads"], "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": case["window"]}, "v_mix": True}
    return bedarax_config({"architecture": "Bedarax", "layers": [{"type": "attention", "mixer": mixer}], "norm": {"eps": 1e-6}, "vocab": 1024, "width": 1024})


def _window_inputs(case: dict, seed: int):
    new, old = _lengths(case)
    g, H, G, n = _gen(seed), case["heads"], case["kv_heads"], sum(new) + sum(old)
    talk = torch.eye(H, dtype=F32, device=DEV) + _rnd(g, H, H, dtype=F32, std=0.2)
    return _rnd(g, sum(new), H * 128 + H), _rnd(g, n, G * 128), _rnd(g, n, G * 128), talk


def _prepare_window(case: dict, seed: int):
    s = _hybrid(case, seed, _window_config(case))
    s["src"], k, v, s["talk"] = _window_inputs(case, seed)
    kc, vc = s["ctx"].kv_cache.kv_rows(0)
    where = torch.cat(s["slots"])
    kc[where], vc[where] = k, v
    return s


def _run_window(case: dict, s: dict):
    from mini_sglang_amd import mixops

    md, ctx, H, G, T = s["batch"].attn_metadata, s["ctx"], case["heads"], case["kv_heads"], s["T"]
    kc, vc = ctx.kv_cache.kv_rows(0)
    out = torch.empty((T, H * 128), dtype=BF16, device=DEV)
    mixops.window_attn(out, s["src"], H * 128, kc, vc, ctx.page_table, md.req_rows, md.seq_lens, md.cu_seqlens_q, md.batch, H, G, 128, 128, case["window"],
                       128 ** -0.5, s["talk"], splits=mixops.window_attn_splits(md.batch, T, case["window"], md.max_seqlen_k))
    return out


def _hidden(n: int, c: int, window: int, keep: int = 0):
    i, j = torch.arange(c, c + n, device=DEV)[:, None], torch.arange(c + n, device=DEV)[None, :]
    return (j > i) | ((i - j >= window) & (j >= keep)) if window else j > i


def _exact_window(case: dict, seed: int):
    src, k, v, talk = _window_inputs(case, seed)
    new, old = _lengths(case)
    H, G, out, a, b = case["heads"], case["kv_heads"], [], 0, 0
    for n, c in zip(new, old):
        kk, vv = (x[b: b + c + n].to(F64).view(c + n, G, 128).permute(1, 0, 2).repeat_interleave(H // G, dim=0) for x in (k, v))
        parts = []
        for t in range(0, n, 512):  # some query rows at a time: all heads' scores are held at once
            e = min(t + 512, n)
            q = src[a + t: a + e, : H * 128].to(F64).view(e - t, H, 128).permute(1, 0, 2)
            raw = torch.stack([q[h] @ kk[h].T for h in range(H)]) * 128 ** -0.5
            sc = (talk.to(F64) @ raw.view(H, -1)).view_as(raw).masked_fill(_hidden(n, c, case["window"])[t: e], -math.inf)
            p = torch.softmax(sc, dim=-1)
            parts.append(torch.stack([p[h] @ vv[h] for h in range(H)], dim=1) * torch.sigmoid(src[a + t: a + e, H * 128:].to(F64))[:, :, None])
        out.append(torch.cat(parts).reshape(n, H * 128))
        a, b = a + n, b + c + n
    return torch.cat(out)


def _work_window(case: dict):
    new, _ = _lengths(case)
    H, G = case["heads"], case["kv_heads"]
    return {"bytes": 2 * (_keys(case) * 2 * G * 128 + sum(new) * (2 * H * 128 + H)), "flops": 2 * _pairs(case) * H * (256 + H)}


# ------------------------------------------------------------------------------------------------ gated delta rule
def _delta_config(case: dict):
    from mini_sglang_amd.hybrid import bedarax_config

    kind = "channel_delta" if case["per_channel"] else "delta"
    mixer = {"heads": case["heads"], "kv_heads": case["heads"], "dim": 128, "vdim": 128, "conv": 4}
    return bedarax_config({"architecture": "Bedarax", "layers": [{"type": kind, "mixer": mixer}], "norm": {"eps": 1e-6}, "vocab": 1024, "width": 1024},
                          shapes={"l0.mix.a1": (128, 1024), "l0.mix.g1": (128, 1024)})


def _delta_inputs(case: dict, seed: int):
    new, old = _lengths(case)
    g, H, T = _gen(seed), case["heads"], sum(new)
    q, k = (F.normalize(F.silu(_rnd(g, T, H, 128, dtype=F32)), dim=-1) for _ in range(2))
    v = F.silu(_rnd(g, T, H * 128, dtype=F32))
    n = H * 128 if case["per_channel"] else H
    state = _rnd(g, len(new) + 1, H, 128, 128, dtype=F32, std=0.1 if case["old"] else 0.0)
    return {"qkv": torch.cat([(q * 128 ** -0.5).reshape(T, -1), k.reshape(T, -1), v], dim=1), "b": _rnd(g, T, H), "a": _rnd(g, T, n), "state": state,
            "rate": -torch.exp(_rnd(g, H, dtype=F32, std=0.5)), "dt": _rnd(g, n, dtype=F32, std=0.5)}


def _prepare_delta(case: dict, seed: int):
    s = _hybrid(case, seed, _delta_config(case))
    s.update(_delta_inputs(case, seed))
    s["ctx"].kv_cache.state(0).copy_(s["state"])
    return s


def _run_delta(case: dict, s: dict):
    from mini_sglang_amd import mixops

    md, kv, H, T = s["batch"].attn_metadata, s["ctx"].kv_cache, case["heads"], s["T"]
    out = torch.empty((T, H * 128), dtype=F32, device=DEV)
    mixops.delta_rule(out, s["qkv"], kv.state(0), s["b"], s["a"], case["per_channel"], s["rate"], s["dt"], md.cu_seqlens_q, md.seq_lens, md.req_rows, md.batch, H,
                      chunks=md.delta_chunks)
    return out, kv.state(0)[: md.batch]


def _exact_delta(case: dict, seed: int):
    s = _delta_inputs(case, seed)
    new, old = _lengths(case)
    H, B, N = case["heads"], len(new), max(new)
    pad = torch.nn.utils.rnn.pad_sequence

    def rows(x):  # [T, ...] -> [N, B, ...], short requests padded at the end
        return pad([r.to(F64) for r in torch.split(x, new)])

    qkv = rows(s["qkv"])
    q, k, v = (x.reshape(N, B, H, 128) for x in torch.split(qkv, H * 128, dim=2))
    beta = torch.sigmoid(rows(s["b"]))
    n = 128 if case["per_channel"] else 1
    a = rows(s["a"]) + s["dt"].to(F64)
    decay = torch.exp(s["rate"].to(F64)[:, None] * F.softplus(a).reshape(N, B, H, n))
    S = s["state"][:B].to(F64) * (1.0 if case["old"] else 0.0)
    out = torch.empty((N, B, H, 128), dtype=F64, device=DEV)
    live = torch.tensor(new, device=DEV)
    for t in range(N):
        Sd = S * decay[t][..., None]
        u = beta[t][..., None] * (v[t] - (Sd * k[t][..., None]).sum(dim=2))
        Sn = Sd + k[t][..., None] * u[..., None, :]
        out[t] = (Sn * q[t][..., None]).sum(dim=2)
        S = torch.where((t < live)[:, None, None, None], Sn, S)
    return torch.cat([out[:m, b] for b, m in enumerate(new)]).reshape(sum(new), H * 128), S


def _work_delta(case: dict):
    new, _ = _lengths(case)
    H, T = case["heads"], sum(new)
    n = H * 128 if case["per_channel"] else H
    return {"bytes": T * (4 * H * 128 * 4 + 2 * (H + n)) + 2 * 4 * len(new) * H * 128 * 128, "flops": 7 * T * H * 128 * 128}


# ------------------------------------------------------------------------------------------------ difference of two softmax maps
def _maps_config(case: dict):
    from mini_sglang_amd.hybrid import nagezen_config

    mixer = {"heads": case["heads"], "kv_heads": case["kv_heads"], "dim": 64, "vdim": 128, "scale": 64 ** -0.5, "diff": 0.4, "rot": {"base": 1e5, "dims": 64},
             "mask": {"size": case["window"], "keep_first": case["keep"]}}
    return nagezen_config({"architecture": "Nagezen", "layers": [{"type": "attention", "mixer": mixer}], "norm": {"eps": 1e-5}, "vocab": 1024, "width": 1024,
                           "streams": 2})


def _maps_inputs(case: dict, seed: int):
    new, old = _lengths(case)
    g, H, G, n, T = _gen(seed), case["heads"], case["kv_heads"], sum(new) + sum(old), sum(new)
    return (_rnd(g, T, H * 128, dtype=F32), _rnd(g, n, G * 128), _rnd(g, n, G * 128), torch.full((1,), 0.4, dtype=F32, device=DEV),
            _rnd(g, T, H * 128) if case["gate"] else None)


def _prepare_maps(case: dict, seed: int):
    s = _hybrid(case, seed, _maps_config(case))
    s["q"], k, v, s["lam"], s["gate"] = _maps_inputs(case, seed)
    kc, vc = s["ctx"].kv_cache.kv_rows(0)
    where = torch.cat(s["slots"])
    kc[where], vc[where] = k, v
    return s


def _run_maps(case: dict, s: dict):
    from mini_sglang_amd import mixops

    md, ctx, H, G, T = s["batch"].attn_metadata, s["ctx"], case["heads"], case["kv_heads"], s["T"]
    kc, vc = ctx.kv_cache.kv_rows(0)
    out = torch.empty((T, H * 128), dtype=BF16, device=DEV)
    splits = mixops.sink_attn_splits(md.batch, T, H, G, case["window"], md.max_seqlen_k, case["keep"]) if md.max_seqlen_q <= 16 else 1
    mixops.diff_attn(out, s["q"], kc, vc, ctx.page_table, md.req_rows, md.seq_lens, md.cu_seqlens_q, md.batch, H, G, 64, 128, 64 ** -0.5, case["window"],
                     case["keep"], s["lam"], 0.6, 1e-5, gate=s["gate"], splits=splits)
    return out


def _exact_maps(case: dict, seed: int):
    q, k, v, lam, gate = _maps_inputs(case, seed)
    new, old = _lengths(case)
    H, G, out, a, b = case["heads"], case["kv_heads"], [], 0, 0
    for n, c in zip(new, old):
        hidden = _hidden(n, c, case["window"], case["keep"])
        o = torch.empty((n, H, 128), dtype=F64, device=DEV)
        for h in range(H):
            j = h // (H // G)
            both = []
            for m in range(2):
                qm = q[a: a + n, (2 * h + m) * 64: (2 * h + m + 1) * 64].to(F64)
                km = k[b: b + c + n, (2 * j + m) * 64: (2 * j + m + 1) * 64].to(F64)
                p = torch.softmax(((qm @ km.T) * 64 ** -0.5).masked_fill(hidden, -math.inf), dim=-1)
                both.append(p @ v[b: b + c + n, j * 128: (j + 1) * 128].to(F64))
            d = both[0] - lam.to(F64) * both[1]
            o[:, h] = d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * 0.6
        o = o.reshape(n, H * 128)
        out.append(o if gate is None else o * torch.sigmoid(gate[a: a + n].to(F64)))
        a, b = a + n, b + c + n
    return torch.cat(out)


def _work_maps(case: dict):
    new, _ = _lengths(case)
    H, G = case["heads"], case["kv_heads"]
    return {"bytes": 2 * _keys(case) * 2 * G * 128 + sum(new) * H * 128 * (4 + 2 + (2 if case["gate"] else 0)), "flops": _pairs(case) * H * (4 * 64 + 4 * 128)}


# ------------------------------------------------------------------------------------------------ what is called from outside
# per kind: prepare(case, seed), run(case, state), exact(case, seed) or None, work(case), tolerance
_KINDS = {
    "step": (_prepare_step, _run_step, _exact_step, _work_step, {"rel": 0.03, "max": 0.3}),
    "decode": (_prepare_paged, _run_paged, _exact_paged, _work_paged, {"rel": 0.01, "max": 0.1}),
    "prefill": (_prepare_paged, _run_paged, _exact_paged, _work_paged, {"rel": 0.01, "max": 0.1}),
    "sample": (_prepare_sample, _run_sample, None, _work_sample, "exact"),
    "latent": (_prepare_latent, _run_latent, _exact_latent, _work_latent, {"rel": 0.01, "max": 0.1}),
    "experts": (lambda case, seed: _experts_inputs(case, seed), _run_experts, _exact_experts, _work_experts, {"rel": 0.01, "max": 0.3, "differ": 1e-4}),
    "window": (_prepare_window, _run_window, _exact_window, _work_window, {"rel": 0.01, "max": 0.1}),
    "delta": (_prepare_delta, _run_delta, _exact_delta, _work_delta, {"rel": 1e-5, "max": 2e-4}),
    "maps": (_prepare_maps, _run_maps, _exact_maps, _work_maps, {"rel": 0.012, "max": 0.2}),
}


def prepare(case: dict, seed: int):
    return {"case": case, "state": _KINDS[case["kind"]][0](case, seed)}


def run(state: dict):
    case = state["case"]
    return _KINDS[case["kind"]][1](case, state["state"])


def exact(case: dict, seed: int):
    f = _KINDS[case["kind"]][2]
    return None if f is None else f(case, seed)


def work(case: dict):
    return _KINDS[case["kind"]][3](case)


def tolerance(case: dict):
    if case.get("dtype") == "fp16":  # three more bits than bf16 in inputs, probabilities and results
        return {"rel": 0.0012, "max": 0.012}
    return _KINDS[case["kind"]][4]
