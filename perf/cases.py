"""The workloads this backend is timed on, through the entry points a serving engine calls.

Three kinds of case:

  attend  one layer's attention step as kvserve's `Attention.attend` drives it: `write_kv` of the
          step's new K/V rows, then `forward` over the paged cache. Batches of decoding
          sequences (one or a few query tokens each), prompt chunks, or both in one step, over
          16-bit or E4M3 caches, with or without a prefix shared by every table.
  rope    `rope_and_cache`: the fused QKV projection of a step split, rotated and written to the
          cache, the queries handed back.
  decode  a decoder's whole decode step, replayed from its HIP graph: step metadata, layers over
          the paged cache, logits.

Sizes are those of the two Llama shapes the engine is configured for (1B: 32 query heads over 8
kv heads of 64; 8B: 32 over 8 of 128) and of the benchmark's workloads. Lengths follow from the
case alone, values and physical block orders from the seed.
"""

from __future__ import annotations

import math
import random

import torch

from kvserve_amd import HipAttention, build_metadata
from kvserve_amd.engine import LLAMA_3_1_8B, LLAMA_3_2_1B, ModelRunner, build_model
from kvserve_amd.engine.model import rope_tables

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
E4M3_SCALES = {"k_scale": 1.0, "v_scale": 0.5}  # per-tensor scales of an E4M3 cache
MODELS = {"1b": LLAMA_3_2_1B, "8b": LLAMA_3_1_8B}


def _attend(name: str | None = None, **kw) -> dict:
    """An attend case: `decodes` sequences of `q` query tokens over lo .. hi cached tokens, then
    `chunks` sequences computing chunk_lo .. chunk_hi prompt tokens over ctx_lo .. ctx_hi cached
    ones; `shared` leading tokens of every decoding sequence lie in the same physical blocks."""
    c = {
        "kind": "attend", "dtype": "bf16", "cache": "16bit", "heads": 32, "kv_heads": 8, "head_dim": 128, "block": 16,
        "decodes": 0, "q": 1, "lo": 0, "hi": 0, "shared": 0,
        "chunks": 0, "chunk_lo": 0, "chunk_hi": 0, "ctx_lo": 0, "ctx_hi": 0, "lens": 0,
    }  # fmt: skip
    c.update(kw)
    return {"name": name, **c} if name else c


def listed() -> list[dict]:
    return [
        # a small model answering a few short chats: the smallest step, bound by launches and latency
        _attend("decode_1b_b8", head_dim=64, decodes=8, lo=63, hi=511),
        # ordinary chat decoding of the 8B shape, fp16
        _attend("decode_8b_b16_fp16", dtype="fp16", decodes=16, lo=200, hi=2200),
        # a busy server's decode step, long contexts (the benchmark's headline shape)
        _attend("decode_8b_b64", decodes=64, lo=1023, hi=8191),
        # the same over an E4M3 cache
        _attend("decode_8b_b64_e4m3", cache="e4m3", decodes=64, lo=1023, hi=8191),
        # long documents behind one 12k-token system prompt, its blocks shared by prefix caching
        _attend("decode_8b_b16_prefix", decodes=16, lo=15999, hi=31999, shared=12000),
        # speculative decoding: five draft tokens verified per sequence
        _attend("verify_8b_b32_q5", decodes=32, q=5, lo=2048, hi=4096),
        # a continuous-batching step: decodes of many sequences and four prompt chunks in one batch
        # (the largest step)
        _attend("mixed_8b", decodes=512, lo=255, hi=4095, chunks=4, chunk_lo=384, chunk_hi=384, ctx_hi=4096),
        # whole prompts computed in one step (time to first token), ragged lengths
        _attend("prefill_8b_prompts", chunks=4, chunk_lo=300, chunk_hi=2500),
        # chunks of long prompts over what is already cached, E4M3 cache
        _attend("prefill_8b_chunk_e4m3", cache="e4m3", chunks=2, chunk_lo=900, chunk_hi=1024, ctx_lo=4000, ctx_hi=10000),
        # a 2048-token step's projection rotated and written to the cache
        {"name": "rope_8b_2048", "kind": "rope", "model": "8b", "dtype": "bf16", "cache": "16bit", "tokens": 2048},
        # token generation of the 1B model, eight users, the whole model
        {"name": "decode_model_1b_b8", "kind": "decode", "model": "1b", "layers": 16, "dtype": "bf16", "batch": 8,
         "lo": 200, "hi": 900, "lens": 0},
        # token generation at the 8B layer shape, thirty-two users, two layers and the head
        {"name": "decode_layers_8b_b32", "kind": "decode", "model": "8b", "layers": 2, "dtype": "bf16", "batch": 32,
         "lo": 200, "hi": 900, "lens": 0},
    ]  # fmt: skip


def _log(rng: random.Random, lo: int, hi: int) -> int:
    """A whole number in lo .. hi, spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))) - 0.5)))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode", "decode", "decode", "verify", "mixed", "prefill", "prefill", "prefix", "rope", "model"])
    if kind == "rope":
        return {"kind": "rope", "model": rng.choice(["1b", "8b"]), "dtype": rng.choice(["bf16", "bf16", "fp16"]),
                "cache": rng.choice(["16bit", "e4m3"]), "tokens": _log(rng, 1, 4096)}  # fmt: skip
    if kind == "model":
        model = rng.choice(["1b", "8b"])
        layers = rng.randint(2, 16) if model == "1b" else rng.randint(1, 4)
        lo = _log(rng, 16, 900)
        return {"kind": "decode", "model": model, "layers": layers, "dtype": rng.choice(["bf16", "bf16", "fp16"]),
                "batch": _log(rng, 1, 64), "lo": lo, "hi": lo + _log(rng, 1, 900), "lens": rng.randrange(1 << 20)}  # fmt: skip
    c = {"dtype": rng.choice(["bf16", "bf16", "fp16"]), "cache": rng.choice(["16bit", "16bit", "e4m3"]),
         "head_dim": rng.choice([64, 128, 128]), "block": rng.choice([16, 16, 32]), "lens": rng.randrange(1 << 20)}  # fmt: skip
    if kind != "prefix":
        c["heads"], c["kv_heads"] = rng.choice([(32, 8), (32, 8), (32, 8), (32, 4), (16, 16)])
    most = 8_000_000 // c.get("kv_heads", 8)  # cached tokens of a batch at most
    if kind in ("decode", "verify"):
        n = _log(rng, 1, 256)
        hi = min(_log(rng, 64, 16384), most // n)
        c.update(decodes=n, q=1 if kind == "decode" else rng.randint(2, 8), lo=rng.randint(1, hi), hi=hi)
    elif kind == "mixed":
        n = _log(rng, 4, 300)
        hi = min(_log(rng, 64, 8192), most // n)
        c.update(decodes=n, lo=rng.randint(1, hi), hi=hi, chunks=rng.randint(1, 4), ctx_hi=_log(rng, 1, 8192))
        c["chunk_hi"] = _log(rng, 17, 1024)
        c["chunk_lo"] = rng.randint(17, c["chunk_hi"])
    elif kind == "prefill":
        c.update(chunks=_log(rng, 1, 8), ctx_hi=rng.choice([0, _log(rng, 1, 12000)]))
        c["chunk_hi"] = _log(rng, 20, 2500)
        pairs = 15_000_000 // c["chunks"]  # (query, key) pairs of a sequence at most
        c["chunk_hi"] = max(20, min(c["chunk_hi"], pairs // (c["ctx_hi"] + c["chunk_hi"])))
        c["chunk_lo"] = rng.randint(20, c["chunk_hi"])
    else:
        n = _log(rng, 2, 24)
        c.update(shared=rng.randint(4096, 16000))
        lo = c["shared"] + _log(rng, 1, 4000)
        c.update(decodes=n, lo=lo, hi=lo + _log(rng, 1, 12000))
    return _attend(**c)


# -- attention steps -------------------------------------------------------------------------------


def _lengths(case: dict) -> tuple[list[int], list[int]]:
    """(query lengths, cached lengths) of an attend case, decoding sequences first."""
    rng = random.Random(case["lens"])
    q, ctx = [], []
    for _ in range(case["decodes"]):
        q.append(case["q"])
        ctx.append(rng.randint(case["lo"], case["hi"]))
    for _ in range(case["chunks"]):
        q.append(rng.randint(case["chunk_lo"], case["chunk_hi"]))
        ctx.append(rng.randint(case["ctx_lo"], case["ctx_hi"]))
    return q, ctx


def _tables(case: dict, q: list[int], ctx: list[int], seed: int) -> tuple[list[list[int]], int]:
    """A physical block table per sequence from a shuffled pool, and the pool's size."""
    bs = case["block"]
    shared = case["shared"] // bs
    need = [-(-(c + n) // bs) - (shared if i < case["decodes"] else 0) for i, (n, c) in enumerate(zip(q, ctx))]
    blocks = shared + sum(need)
    blocks += blocks // 10 + 8
    ids = list(range(blocks))
    random.Random(seed).shuffle(ids)
    prefix, at, tables = ids[:shared], shared, []
    for i, n in enumerate(need):
        tables.append((prefix if i < case["decodes"] else []) + ids[at : at + n])
        at += n
    return tables, blocks


def _normal(gen: torch.Generator, shape: tuple[int, ...], dtype: torch.dtype) -> torch.Tensor:
    """N(0, 1) values, drawn in fp32 slices and stored as `dtype`."""
    out = torch.empty(shape, dtype=dtype, device=DEVICE)
    rows = max(1, (1 << 27) // max(1, out[0].numel()))
    for r in range(0, shape[0], rows):
        part = out[r : r + rows]
        part.copy_(torch.randn(part.shape, generator=gen, device=DEVICE, dtype=torch.float32))
    return out


def _e4m3(x: torch.Tensor, scale: float) -> torch.Tensor:
    return (x.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn)


def _caches(gen: torch.Generator, case: dict, shape: tuple[int, ...]) -> tuple[torch.Tensor, torch.Tensor, dict]:
    """K and V caches of N(0, 1) values (in E4M3 with their scales), and the scale arguments."""
    dt = DTYPES[case["dtype"]]
    k, v = _normal(gen, shape, dt), _normal(gen, shape, dt)
    if case["cache"] == "16bit":
        return k, v, {}
    out = []
    for x, s in ((k, E4M3_SCALES["k_scale"]), (v, E4M3_SCALES["v_scale"])):
        y = torch.empty(shape, dtype=torch.float8_e4m3fn, device=DEVICE)
        rows = max(1, (1 << 27) // x[0].numel())
        for r in range(0, shape[0], rows):
            y[r : r + rows] = _e4m3(x[r : r + rows], s)
        out.append(y)
    return out[0], out[1], dict(E4M3_SCALES)


def _prepare_attend(case: dict, seed: int) -> dict:
    q, ctx = _lengths(case)
    tables, blocks = _tables(case, q, ctx, seed)
    bs, H, Hkv, D = case["block"], case["heads"], case["kv_heads"], case["head_dim"]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    T = sum(q)
    k_cache, v_cache, scales = _caches(gen, case, (blocks, bs, Hkv, D))
    # q, k, v as a layer hands them over: k and v are views of its fused projection's rows
    qkv = _normal(gen, (T, (H + 2 * Hkv) * D), dt)
    k_new = qkv[:, H * D : (H + Hkv) * D].unflatten(1, (Hkv, D))
    v_new = qkv[:, (H + Hkv) * D :].unflatten(1, (Hkv, D))
    slots = [t[p // bs] * bs + p % bs for t, n, c in zip(tables, q, ctx) for p in range(c, c + n)]
    meta = build_metadata(DEVICE, tables, slots, [n + c for n, c in zip(q, ctx)], q)
    return {"case": case, "q": qkv[:, : H * D].unflatten(1, (H, D)).contiguous(), "k": k_new.contiguous(), "v": v_new,
            "k_cache": k_cache, "v_cache": v_cache, "meta": meta, "scale": D**-0.5, "scales": scales}  # fmt: skip


def _run_attend(s: dict):
    HipAttention.write_kv(s["k_cache"], s["v_cache"], s["k"], s["v"], s["meta"].slot_mapping, **s["scales"])
    out = HipAttention.forward(s["q"], s["k_cache"], s["v_cache"], s["meta"], s["scale"], **s["scales"])
    return {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


def _write(cache: torch.Tensor, rows: torch.Tensor, slots: torch.Tensor, scale: float | None) -> torch.Tensor:
    """The cache after `rows` were stored at `slots` (the cache's own storage, updated)."""
    if scale is None:
        cache.view(-1, *cache.shape[2:])[slots] = rows
    else:
        cache.view(torch.uint8).view(-1, *cache.shape[2:])[slots] = _e4m3(rows, scale).view(torch.uint8)
    return cache


def _attention64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, ctx: int, scale: float) -> torch.Tensor:
    """Causal attention in 64 bits of one sequence: q [n, H, D] at positions ctx .., k, v [S, Hkv, D]."""
    n, H, D = q.shape
    S, Hkv = k.shape[:2]
    G = H // Hkv
    hidden = torch.arange(S, device=q.device)[None, :] > ctx + torch.arange(n, device=q.device)[:, None]
    out = torch.empty((n, H, D), dtype=torch.float64, device=q.device)
    for h in range(Hkv):
        kh, vh = k[:, h].double().contiguous(), v[:, h].double().contiguous()
        kt = kh.t().contiguous()
        for g in range(h * G, (h + 1) * G):
            s = (q[:, g].double().contiguous() @ kt) * scale
            out[:, g] = torch.softmax(s.masked_fill(hidden, -math.inf), dim=-1) @ vh
    return out


def _exact_attend(case: dict, seed: int):
    q, ctx = _lengths(case)
    if sum(n * (n + c) for n, c in zip(q, ctx)) * case["heads"] * case["head_dim"] > 2e12:
        return None
    s = _prepare_attend(case, seed)
    ks, vs = s["scales"].get("k_scale"), s["scales"].get("v_scale")
    kc = _write(s["k_cache"], s["k"], s["meta"].slot_mapping, ks)
    vc = _write(s["v_cache"], s["v"], s["meta"].slot_mapping, vs)
    bs, out, t0 = case["block"], [], 0
    for i, (n, c) in enumerate(zip(q, ctx)):
        blocks = s["meta"].block_tables[i, : -(-(n + c) // bs)]
        k, v = ((x.view(torch.uint8)[blocks].view(x.dtype) if x.element_size() == 1 else x[blocks]) for x in (kc, vc))
        k, v = (x.flatten(0, 1)[: n + c].double() * (f or 1.0) for x, f in ((k, ks), (v, vs)))
        out.append(_attention64(s["q"][t0 : t0 + n], k, v, c, s["scale"]))
        t0 += n
    return {"out": torch.cat(out), "k_cache": kc, "v_cache": vc}


def _work_attend(case: dict) -> dict:
    q, ctx = _lengths(case)
    H, Hkv, D = case["heads"], case["kv_heads"], case["head_dim"]
    eb = 1 if case["cache"] == "e4m3" else 2
    T = sum(q)
    again = case["shared"] // case["block"] * case["block"] * max(0, case["decodes"] - 1)  # read once for all
    rows = sum(ctx) + T - again
    blocks = sum(-(-(n + c) // case["block"]) for n, c in zip(q, ctx))
    seen = sum(n * c + n * (n + 1) // 2 for n, c in zip(q, ctx))
    return {
        "bytes": 2 * Hkv * D * (eb * rows + (2 + eb) * T) + 2 * T * H * D * 2 + 8 * (blocks + T + 3 * len(q) + 1),
        "flops": 4 * H * D * seen,
    }


# -- RoPE and cache write --------------------------------------------------------------------------


def _prepare_rope(case: dict, seed: int) -> dict:
    cfg, T, bs = MODELS[case["model"]], case["tokens"], 16
    H, Hkv, D = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    blocks = -(-T // bs) * 2 + 8
    k_cache, v_cache, scales = _caches(gen, case, (blocks, bs, Hkv, D))
    # the step computes T consecutive positions of one prompt, from a multiple of its chunk
    start = T * random.Random(seed).randint(0, 3)
    table = list(range(blocks))
    random.Random(seed).shuffle(table)
    slots = torch.tensor([table[p // bs] * bs + p % bs for p in range(T)], dtype=torch.long, device=DEVICE)
    cos, sin = rope_tables(cfg, 4 * T, DEVICE)
    return {"case": case, "qkv": _normal(gen, (T, (H + 2 * Hkv) * D), dt), "cos": cos, "sin": sin, "slots": slots,
            "positions": torch.arange(start, start + T, device=DEVICE), "k_cache": k_cache, "v_cache": v_cache,
            "scales": scales, "heads": H}  # fmt: skip


def _run_rope(s: dict):
    q = HipAttention.rope_and_cache(s["qkv"], s["positions"], s["cos"], s["sin"], s["k_cache"], s["v_cache"],
                                    s["slots"], s["heads"], **s["scales"])  # fmt: skip
    return {"q": q, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


def _rotate64(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """x [T, heads, D] in 64 bits rotated by the tokens' table rows [T, D]."""
    x, half = x.double(), x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos.double()[:, None, :] + turned * sin.double()[:, None, :]


def _exact_rope(case: dict, seed: int):
    s = _prepare_rope(case, seed)
    cfg = MODELS[case["model"]]
    H, Hkv, D = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    cos, sin = s["cos"][s["positions"]], s["sin"][s["positions"]]
    q, k, v = s["qkv"].split([H * D, Hkv * D, Hkv * D], dim=1)
    out = {"q": _rotate64(q.unflatten(1, (H, D)), cos, sin)}
    rows = {"k_cache": _rotate64(k.unflatten(1, (Hkv, D)), cos, sin), "v_cache": v.unflatten(1, (Hkv, D)).double()}
    for name, x in rows.items():
        scale = s["scales"].get(name[0] + "_scale")
        c = s[name].double()
        c.view(-1, Hkv, D)[s["slots"]] = x / scale if scale else x
        out[name] = c
    return out


def _work_rope(case: dict) -> dict:
    cfg, T = MODELS[case["model"]], case["tokens"]
    H, Hkv, D = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    eb = 1 if case["cache"] == "e4m3" else 2
    return {"bytes": T * D * (2 * (H + 2 * Hkv) + 2 * H + 2 * Hkv * eb + 8) + 16 * T, "flops": 3 * T * (H + Hkv) * D}


# -- decode steps of a decoder ---------------------------------------------------------------------


def _prepare_decode(case: dict, seed: int) -> dict:
    cfg, bs = MODELS[case["model"]].with_layers(case["layers"]), 16
    rng = random.Random(case["lens"])
    lens = [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    max_len = max(lens) + 1
    dt = DTYPES[case["dtype"]]
    model = build_model(cfg, DEVICE, dt, max_len, seed=seed)
    blocks = sum(-(-(n + 1) // bs) for n in lens) + 8
    runner = ModelRunner(model, num_blocks=blocks, block_size=bs, max_model_len=max_len, piecewise_graphs=False,
                         max_graph_batch=case["batch"], max_seqs=case["batch"], token_budget=case["batch"])  # fmt: skip
    # the contexts' keys and values, as earlier steps left them
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    for layer in runner.kv_caches:
        for cache in layer:
            cache.copy_(_normal(gen, tuple(cache.shape), dt))
    order = list(range(blocks))
    random.Random(seed).shuffle(order)
    tables, at = [], 0
    for n in lens:
        need = -(-(n + 1) // bs)
        tables.append(order[at : at + need])
        at += need
    ids = [random.Random(seed + 2 + i).randrange(cfg.vocab_size) for i in range(len(lens))]
    return {"case": case, "runner": runner, "keyed": list(enumerate(tables)), "lens": lens, "ids": ids, "cfg": cfg}


def _run_decode(s: dict):
    r = s["runner"]
    hidden = r.decode_runner.replay_device(r.dm, s["keyed"], s["lens"], s["ids"])
    return {"logits": r.model.logits(hidden), "kv": r.kv_caches}


def _norm64(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    return weight.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _exact_decode(case: dict, seed: int):
    s = _prepare_decode(case, seed)
    cfg, w, kv = s["cfg"], s["runner"].model.w, s["runner"].kv_caches
    H, Hkv, D, bs = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, 16
    pos = torch.tensor(s["lens"], device=DEVICE)
    cos, sin = s["runner"].model.cos[pos], s["runner"].model.sin[pos]
    x = w.embed[torch.tensor(s["ids"], device=DEVICE)].double()

    def linear(a: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
        parts = weight.split(16384)
        return torch.cat([a @ p.double().t().contiguous() for p in parts], dim=-1)

    for i, lw in enumerate(w.layers):
        q, k, v = linear(_norm64(x, lw.attn_norm, cfg.rms_norm_eps), lw.wqkv).split([H * D, Hkv * D, Hkv * D], dim=1)
        q = _rotate64(q.unflatten(1, (H, D)), cos, sin)
        k, v = _rotate64(k.unflatten(1, (Hkv, D)), cos, sin), v.unflatten(1, (Hkv, D))
        rows = []
        for b, (_, table) in enumerate(s["keyed"]):
            t, n = torch.tensor(table, device=DEVICE), s["lens"][b]
            old = [kv[i, j][t].flatten(0, 1)[:n].double() for j in (0, 1)]
            kb, vb = torch.cat((old[0], k[b : b + 1])), torch.cat((old[1], v[b : b + 1]))
            rows.append(_attention64(q[b : b + 1], kb, vb, n, D**-0.5))
        x = x + linear(torch.cat(rows).flatten(1), lw.wo)
        gate, up = linear(_norm64(x, lw.mlp_norm, cfg.rms_norm_eps), lw.w_gate_up).chunk(2, dim=-1)
        x = x + linear(torch.nn.functional.silu(gate) * up, lw.w_down)
    return {"logits": linear(_norm64(x, w.final_norm, cfg.rms_norm_eps), w.lm_head), "kv": None}


def _work_decode(case: dict) -> dict:
    cfg, B = MODELS[case["model"]], case["batch"]
    rng = random.Random(case["lens"])
    keys = sum(rng.randint(case["lo"], case["hi"]) + 1 for _ in range(B))
    H, Hkv, D, hid = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.hidden_size
    layer = hid * (H + 2 * Hkv) * D + H * D * hid + 3 * hid * cfg.intermediate_size
    params = case["layers"] * layer + cfg.vocab_size * hid
    kv = case["layers"] * 2 * Hkv * D * 2 * (keys + B)
    return {"bytes": 2 * params + kv + 4 * B * cfg.vocab_size,
            "flops": 2 * B * params + case["layers"] * 4 * H * D * keys}  # fmt: skip


# -- the cases' common face ------------------------------------------------------------------------


_KINDS = {
    "attend": (_prepare_attend, _run_attend, _exact_attend, _work_attend),
    "rope": (_prepare_rope, _run_rope, _exact_rope, _work_rope),
    "decode": (_prepare_decode, _run_decode, _exact_decode, _work_decode),
}


def prepare(case: dict, seed: int) -> dict:
    return _KINDS[case["kind"]][0](case, seed)


def run(state: dict):
    return _KINDS[state["case"]["kind"]][1](state)


def exact(case: dict, seed: int):
    return _KINDS[case["kind"]][2](case, seed)


def work(case: dict) -> dict:
    return _KINDS[case["kind"]][3](case)


def tolerance(case: dict):
    """Measured against `exact` (relative 2-norm), about four times what is seen: one attention
    step 2.3e-3 in bf16 and 2.6e-4 in fp16; a decode step's logits 0.012 after 2 layers and
    0.031 after 16 in bf16, an eighth of that in fp16. RoPE and the cache writes are bit for bit
    those of the separate PyTorch operations."""
    if case["kind"] == "rope":
        return "exact"
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "decode":
        return {"rel": (0.025 if bf16 else 0.003) * math.sqrt(case["layers"])}
    return {"rel": 1e-2 if bf16 else 1.2e-3}
