"""The calls a serving program makes, as timed cases.

Six kinds, each through an entry point of ``pagelora_amd`` that a program
calls: one layer of paged decode attention, one layer of paged prefill
attention, a layer's no-merge LoRA delta on all seven modules, a projection at
decode batch sizes, one captured decode step of a Qwen3-shaped decoder, and
the prefill of a prompt segment.  ``listed`` names twelve of them, ``draw``
takes others of the same ranges.
"""

from __future__ import annotations

import math
import random

import torch

from pagelora_amd.attention_backend import PagedDecodeAttention
from pagelora_amd.decode_graph import BatchDecodeGraphRunner
from pagelora_amd.decoder import DecoderConfig, DecoderWeights, prefill, prefill_backend
from pagelora_amd.kv_pool import PagedKVPool, Request
from pagelora_amd.linear import ShuffledWeight, linear_shuffled
from pagelora_amd.lora import lora_delta_groups_

PAGE = 16
HEAD_DIM = 128
# (q heads, kv heads): Qwen3-8B (GQA 4), Llama-2-7B (MHA),
# DeepSeek-R1-Distill-Qwen-7B (GQA 7)
HEADS = {"gqa4": (32, 8), "mha": (32, 32), "gqa7": (28, 4)}
# Qwen3-8B widths: hidden 4096, intermediate 12288, 32 q / 8 kv heads; a head of
# 32000 tokens, which four layers outweigh as the model's 36 do its own head
HIDDEN, INTER, VOCAB = 4096, 12288, 32000
Q_DIM, KV_DIM = 32 * HEAD_DIM, 8 * HEAD_DIM
ROPE_THETA, EPS = 1_000_000.0, 1e-6
RANK, ALPHA = 16, 32.0
# packed groups of a layer: (input width, ((module, output width), ...))
GROUPS = ((HIDDEN, (("q", Q_DIM), ("k", KV_DIM), ("v", KV_DIM))), (Q_DIM, (("o", HIDDEN),)),
          (HIDDEN, (("gate", INTER), ("up", INTER))), (INTER, (("down", HIDDEN),)))


def listed():
    return [
        # one request's decode, the least a step can be: latency and launches
        {"name": "decode_attn_1x2048_bf16", "kind": "decode_attn", "heads": "gqa4", "rows": 1, "min_len": 2048,
         "max_len": 2048, "dtype": "bf16"},
        # a medium batch of ragged chats, odd row count, a GQA ratio that is no power of two
        {"name": "decode_attn_23_ragged_gqa7_bf16", "kind": "decode_attn", "heads": "gqa7", "rows": 23, "min_len": 33,
         "max_len": 4099, "dtype": "bf16"},
        # a full batch of ragged contexts without GQA, the largest decode call
        {"name": "decode_attn_64_ragged_mha_fp16", "kind": "decode_attn", "heads": "mha", "rows": 64, "min_len": 128,
         "max_len": 8192, "dtype": "fp16"},
        # an ordinary prompt from scratch (2119 tokens)
        {"name": "prefill_attn_2119_mha_fp16", "kind": "prefill_attn", "heads": "mha", "requests": 1, "tokens": 2119,
         "prefix": 0, "dtype": "fp16"},
        # the next turn of a long chat: a short segment behind a long cached prefix
        {"name": "prefill_attn_77_behind_32000_bf16", "kind": "prefill_attn", "heads": "gqa4", "requests": 1,
         "tokens": 77, "prefix": 32000, "dtype": "bf16"},
        # the last 8192-token segment of a 32768-token prompt, the largest prefill call
        {"name": "prefill_attn_8192_of_32768_bf16", "kind": "prefill_attn", "heads": "gqa4", "requests": 1,
         "tokens": 8192, "prefix": 24576, "dtype": "bf16"},
        # a decode batch of 64 rows over 4 adapters: a layer's delta on all seven modules
        {"name": "lora_delta_64_bf16", "kind": "lora_delta", "tokens": 64, "adapters": 4, "dtype": "bf16"},
        # the same layer's delta over an ordinary prompt bound to its adapter
        {"name": "lora_delta_2112_bf16", "kind": "lora_delta", "tokens": 2112, "adapters": 1, "dtype": "bf16"},
        # the widest projection (gate/up) at an ordinary serving batch
        {"name": "linear_48_gate_up_bf16", "kind": "linear", "tokens": 48, "in": HIDDEN, "out": 2 * INTER,
         "dtype": "bf16"},
        # a captured decode step, 4 rows behind a shared prompt prefix (four layers + head)
        {"name": "decode_step_4_shared_2048_bf16", "kind": "decode_step", "rows": 4, "layers": 4, "prefix": 2048,
         "min_len": 64, "max_len": 64, "adapters": 1, "dtype": "bf16"},
        # a new user turn behind a cached system prompt (four layers + head)
        {"name": "prefill_77_behind_2048_bf16", "kind": "prefill", "tokens": 77, "prefix": 2048, "layers": 4,
         "adapters": 1, "dtype": "bf16"},
        # an ordinary prompt from scratch (four layers + head)
        {"name": "prefill_2112_bf16", "kind": "prefill", "tokens": 2112, "prefix": 0, "layers": 4, "adapters": 1,
         "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("decode_attn", "prefill_attn", "lora_delta", "linear", "decode_step", "prefill"))
    dtype = rng.choice(("bf16", "fp16"))
    if kind == "decode_attn":
        hi = _log_int(rng, 17, 8192)
        return {"kind": kind, "heads": rng.choice(sorted(HEADS)), "rows": _log_int(rng, 1, 64),
                "min_len": max(1, hi // rng.choice((1, 2, 64))), "max_len": hi, "dtype": dtype}
    if kind == "prefill_attn":
        return {"kind": kind, "heads": rng.choice(sorted(HEADS)), "requests": rng.choice((1, 1, 2, 3)),
                "tokens": _log_int(rng, 2, 2200), "prefix": rng.choice((0, _log_int(rng, 1, 32000))), "dtype": dtype}
    if kind == "lora_delta":
        return {"kind": kind, "tokens": _log_int(rng, 1, 2112), "adapters": rng.choice((1, 2, 4, 7)), "dtype": dtype}
    if kind == "linear":
        return {"kind": kind, "tokens": _log_int(rng, 1, 64), "in": 32 * _log_int(rng, 32, 384),
                "out": _log_int(rng, 1000, 2 * INTER), "dtype": dtype}
    if kind == "decode_step":
        hi = _log_int(rng, 17, 2048)
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "layers": rng.choice((2, 4)),
                "prefix": PAGE * rng.choice((0, 4, 128)), "min_len": max(1, hi // rng.choice((1, 8))), "max_len": hi,
                "adapters": rng.choice((1, 1, 3)), "dtype": dtype}
    return {"kind": kind, "tokens": _log_int(rng, 1, 2112), "prefix": PAGE * rng.choice((0, 9, 128)),
            "layers": rng.choice((2, 4)), "adapters": rng.choice((1, 1, 3)), "dtype": dtype}


# ------------------------------------------------------------------- inputs
def _dtype(case):
    return {"bf16": torch.bfloat16, "fp16": torch.float16}[case["dtype"]]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, dtype, std=1.0):
    t = torch.randn(shape, dtype=dtype, device="cuda", generator=gen)
    return t.mul_(std) if std != 1.0 else t


def _lens(case):
    """Row lengths: a function of the sizes alone, so that every seed does the same work."""
    rng = random.Random(case["rows"] * 1_000_003 + case["max_len"])
    lens = [rng.randint(case["min_len"], case["max_len"]) for _ in range(case["rows"])]
    return lens


def _page_table(lens, seed, shared=0):
    """Random pages for rows of the given lengths, the first ``shared`` pages
    common to all: (pages per row, indptr, indices, last page lengths, pool
    size).  Page 0 stays unused."""
    need = [-(-n // PAGE) for n in lens]
    total = shared + sum(n - shared for n in need)
    ids = list(range(1, total + 1))
    random.Random(seed).shuffle(ids)
    rows, at = [], shared
    for n in need:
        rows.append(ids[:shared] + ids[at:at + n - shared])
        at += n - shared
    indptr = [0]
    for r in rows:
        indptr.append(indptr[-1] + len(r))

    def i32(x):
        return torch.tensor(x, dtype=torch.int32)

    last = [n - PAGE * (k - 1) for n, k in zip(lens, need)]
    return rows, i32(indptr), i32([p for r in rows for p in r]), i32(last), total + 1


def _attention_inputs(case, seed):
    hq, hkv = HEADS[case["heads"]]
    gen, dt = _gen(seed), _dtype(case)
    if case["kind"] == "decode_attn":
        lens, tokens = _lens(case), case["rows"]
    else:
        lens = [case["prefix"] + case["tokens"]] * case["requests"]
        tokens = case["requests"] * case["tokens"]
    rows, indptr, indices, last, pool = _page_table(lens, seed)
    cache = _normal(gen, (pool, 2, PAGE, hkv, HEAD_DIM), dt)
    q = _normal(gen, (tokens, hq, HEAD_DIM), dt)
    return q, cache, lens, rows, indptr, indices, last


def _lora_inputs(case, seed):
    """The groups' inputs and, per module, A, B and the base output the delta
    lands in: column views of a group's packed output, all groups in one
    buffer (returned first)."""
    gen, dt, T, n = _gen(seed), _dtype(case), case["tokens"], case["adapters"]
    widths = [sum(out for _, out in modules) for _, modules in GROUPS]
    base = _normal(gen, (T * sum(widths),), dt)
    groups, at = [], 0
    for (fin, modules), width in zip(GROUPS, widths):
        x = _normal(gen, (T, fin), dt)
        packed = base[at:at + T * width].view(T, width)
        at += T * width
        mods, col = [], 0
        for _, out in modules:
            mods.append((_normal(gen, (n, RANK, fin), dt, fin ** -0.5), _normal(gen, (n, out, RANK), dt, 0.1),
                         packed[:, col:col + out], ALPHA / RANK))
            col += out
        groups.append((x, mods))
    return base, groups, _adapter_ids(case, seed, T)


def _adapter_ids(case, seed, n):
    rng = random.Random(seed)
    return torch.tensor([rng.randrange(case["adapters"]) for _ in range(n)], dtype=torch.int32, device="cuda")


def _config(case):
    return DecoderConfig(num_layers=case["layers"], hidden=HIDDEN, num_qo_heads=32, num_kv_heads=8, head_dim=HEAD_DIM,
                         intermediate=INTER, vocab=VOCAB, rope_theta=ROPE_THETA, rms_eps=EPS, qk_norm=True,
                         lora_rank=RANK, lora_alpha=ALPHA)


def _model_tensors(case, gen):
    """The weights of a decoder and its adapters, as a checkpoint holds them."""
    dt = _dtype(case)

    def norm(n):
        return (1.0 + 0.1 * torch.randn(n, device="cuda", generator=gen)).to(dt)

    embed, head, final = (_normal(gen, (VOCAB, HIDDEN), dt, 0.02), _normal(gen, (VOCAB, HIDDEN), dt, 0.02),
                          norm(HIDDEN))
    layers = []
    adapters = [{} for _ in range(case["adapters"])]
    for li in range(case["layers"]):
        layer = {"input_norm": norm(HIDDEN), "post_norm": norm(HIDDEN), "q_norm": norm(HEAD_DIM),
                 "k_norm": norm(HEAD_DIM)}
        for fin, modules in GROUPS:
            for m, out in modules:
                layer[m] = _normal(gen, (out, fin), dt, 0.02)
                for a in adapters:
                    a[(li, m)] = (_normal(gen, (RANK, fin), dt, fin ** -0.5), _normal(gen, (out, RANK), dt, 0.01))
        layers.append(layer)
    return embed, head, final, layers, adapters


def _model_inputs(case, seed):
    """Weights, KV pool contents, page table and tokens of a decode step or a prefill."""
    gen, dt = _gen(seed), _dtype(case)
    tensors = _model_tensors(case, gen)
    if case["kind"] == "decode_step":
        # lengths with the step's token, which the step itself appends
        lens = [case["prefix"] + n + 1 for n in _lens(case)]
        shared, n_tokens = case["prefix"] // PAGE, case["rows"]
    else:
        lens, shared, n_tokens = [case["prefix"] + case["tokens"]], 0, case["tokens"]
    rows, indptr, indices, last, pool = _page_table(lens, seed, shared)
    cache = _normal(gen, (case["layers"], pool, 2, PAGE, 8, HEAD_DIM), dt)
    cache[:, 0] = 0
    tokens = torch.randint(0, VOCAB, (n_tokens,), device="cuda", generator=gen)
    return tensors, cache, tokens, lens, rows, indptr, indices, last


def _pool(case, cache):
    pool = PagedKVPool(num_layers=case["layers"], capacity_pages=cache.shape[1], page_size=PAGE, num_kv_heads=8,
                       head_dim=HEAD_DIM, dtype=cache.dtype, device=cache.device, max_pages=None)
    pool.cache.copy_(cache)
    return pool


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode_attn", "prefill_attn"):
        q, cache, lens, rows, indptr, indices, last = _attention_inputs(case, seed)
        hq, hkv = HEADS[case["heads"]]
        be = PagedDecodeAttention(device=q.device, workspace_mb=128, num_qo_heads=hq, num_kv_heads=hkv,
                                  head_dim=HEAD_DIM, page_size=PAGE)
        # one plan serves every layer of a step, so it is not part of a layer's call
        if kind == "decode_attn":
            be.plan_decode(paged_kv_indptr=indptr, paged_kv_indices=indices, paged_kv_last_page_len=last)
        else:
            qo = torch.arange(case["requests"] + 1, dtype=torch.int32) * case["tokens"]
            be.plan_prefill(qo_indptr=qo, paged_kv_indptr=indptr, paged_kv_indices=indices,
                            paged_kv_last_page_len=last, causal=True)
        return {"kind": kind, "backend": be, "q": q, "cache": cache}
    if kind == "lora_delta":
        out, groups, ids = _lora_inputs(case, seed)
        return {"kind": kind, "ids": ids, "groups": groups, "out": out, "base": out.clone()}
    if kind == "linear":
        gen, dt = _gen(seed), _dtype(case)
        x = _normal(gen, (case["tokens"], case["in"]), dt)
        return {"kind": kind, "x": x, "w": ShuffledWeight(_normal(gen, (case["out"], case["in"]), dt, 0.02))}
    (embed, head, final, layers, adapters), cache, tokens, lens, rows, indptr, indices, last = _model_inputs(case, seed)
    cfg = _config(case)
    weights = DecoderWeights.from_tensors(cfg, embed=embed, final_norm=final, lm_head=head, layers=layers,
                                          adapters=adapters, device="cuda", dtype=_dtype(case))
    pool = _pool(case, cache)
    if kind == "prefill":
        request = Request(own_pages=rows[0], length=lens[0])
        return {"kind": kind, "weights": weights, "pool": pool, "request": request, "tokens": tokens,
                "adapter": seed % case["adapters"], "backend": prefill_backend(cfg, PAGE, tokens.device)}
    be = PagedDecodeAttention(device=tokens.device, workspace_mb=128, num_qo_heads=32, num_kv_heads=8,
                              head_dim=HEAD_DIM, page_size=PAGE)
    be.plan_decode(paged_kv_indptr=indptr, paged_kv_indices=indices, paged_kv_last_page_len=last)
    runner = BatchDecodeGraphRunner(weights, pool, be)
    with torch.no_grad():
        entry = runner.entry(case["rows"], uniform_adapter=0 if case["adapters"] == 1 else -1)
    if entry is None:
        raise RuntimeError(f"decode step was not captured: {runner.disabled_reason}")
    ctx = entry.ctx
    ctx.positions.copy_(torch.tensor([n - 1 for n in lens]))
    ctx.page_id.copy_(torch.tensor([r[-1] for r in rows]))
    ctx.page_offset.copy_(torch.tensor([(n - 1) % PAGE for n in lens]))
    ctx.adapter_ids.copy_(_adapter_ids(case, seed, case["rows"]))
    pool.cache.copy_(cache)  # the warm-up before the capture wrote the scratch page
    return {"kind": kind, "runner": runner, "entry": entry, "pool": pool, "tokens": tokens}


# ---------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    if kind == "decode_attn":
        return state["backend"].run_decode(state["q"], state["cache"])
    if kind == "prefill_attn":
        return state["backend"].run_prefill(state["q"], state["cache"])
    if kind == "lora_delta":
        # the delta lands in place, so each pass starts from the base outputs
        state["out"].copy_(state["base"])
        lora_delta_groups_(state["groups"], state["ids"])
        return state["out"]
    if kind == "linear":
        return linear_shuffled(state["x"], state["w"])
    if kind == "decode_step":
        ctx = state["entry"].ctx
        ctx.tokens.copy_(state["tokens"])  # the step leaves its picks there
        logits = state["runner"].replay(state["entry"])
        return {"logits": logits, "kv": state["pool"].cache}
    logits = prefill(state["weights"], state["pool"], state["request"], state["tokens"], adapter=state["adapter"],
                     backend=state["backend"])
    return {"logits": logits, "kv": state["pool"].cache}


# --------------------------------------------------------------------- work
def _causal_pairs(tokens, prefix):
    return tokens * prefix + tokens * (tokens + 1) // 2


def _layer_params():
    return sum(fin * out for fin, mods in GROUPS for _, out in mods)


def _lora_params():
    return sum(RANK * (fin + out) for fin, mods in GROUPS for _, out in mods)


def work(case):
    kind = case["kind"]
    if kind == "decode_attn":
        hq, hkv = HEADS[case["heads"]]
        n = sum(_lens(case))
        return {"bytes": 2 * (2 * n * hkv + 2 * case["rows"] * hq) * HEAD_DIM, "flops": 4 * n * hq * HEAD_DIM}
    if kind == "prefill_attn":
        hq, hkv = HEADS[case["heads"]]
        R, T, P = case["requests"], case["tokens"], case["prefix"]
        return {"bytes": 2 * R * (2 * (T + P) * hkv + 2 * T * hq) * HEAD_DIM,
                "flops": 4 * R * _causal_pairs(T, P) * hq * HEAD_DIM}
    if kind == "lora_delta":
        T, n = case["tokens"], min(case["adapters"], case["tokens"])
        # out: the copy of the base output reads and writes it, and so does the delta
        x = sum(fin for fin, _ in GROUPS)
        out = sum(o for _, mods in GROUPS for _, o in mods)
        return {"bytes": 2 * (n * _lora_params() + T * x + 4 * T * out), "flops": 2 * T * _lora_params()}
    if kind == "linear":
        T, fin, out = case["tokens"], case["in"], case["out"]
        return {"bytes": 2 * (fin * out + T * (fin + out)), "flops": 2 * T * fin * out}
    L, n = case["layers"], case["adapters"]
    kv_row = 2 * 8 * HEAD_DIM
    if kind == "decode_step":
        B, P = case["rows"], case["prefix"]
        own = sum(_lens(case)) + B
        weights = L * (_layer_params() + min(n, B) * _lora_params()) + VOCAB * HIDDEN
        return {"bytes": 2 * (weights + L * (P + own) * kv_row + B * (HIDDEN + VOCAB)),
                "flops": 2 * B * (L * (_layer_params() + _lora_params()) + VOCAB * HIDDEN)
                + 4 * L * (own + B * P) * Q_DIM}
    T, P = case["tokens"], case["prefix"]
    return {"bytes": 2 * (L * (_layer_params() + _lora_params()) + VOCAB * HIDDEN + T * HIDDEN
                          + L * (P + T) * kv_row + VOCAB),
            "flops": 2 * T * L * (_layer_params() + _lora_params()) + 2 * VOCAB * HIDDEN
            + 4 * L * _causal_pairs(T, P) * Q_DIM}


def tolerance(case):
    """Against another correct implementation at the same precision: inputs,
    outputs and the LoRA intermediate in the 16-bit type, sums in fp32.  About
    four times the errors measured against ``exact`` (bf16 / fp16: model 1.7e-2
    / 1.5e-3, attention and linear 1.7e-3 / 2.1e-4 to 2.9e-4, delta 1.9e-3)."""
    bf16 = case["dtype"] == "bf16"
    if case["kind"] in ("decode_step", "prefill"):
        # a rounding in one stage travels through the rest of the layer and the head
        return {"rel": 6e-2 if bf16 else 6e-3}
    if case["kind"] in ("decode_attn", "prefill_attn", "linear"):
        # one rounding of the output
        return {"rel": 6.5e-3 if bf16 else 1e-3}
    return {"rel": 8e-3 if bf16 else 1e-3}  # the intermediate's rounding and the output's


# -------------------------------------------------------------------- exact
def _softmax_rows(s):
    s = s - s.amax(dim=-1, keepdim=True)
    s.exp_()
    return s / s.sum(dim=-1, keepdim=True)


def _attend(q, k, v, first):
    """Causal attention of queries [T, Hq, D] at positions first .. over k, v
    [L, Hkv, D], one q head and a bounded block of queries at a time."""
    T, hq, d = q.shape
    L, hkv, _ = k.shape
    out = torch.empty_like(q)
    block = max(1, (1 << 27) // L)
    pos = torch.arange(L, device=q.device)
    for h in range(hq):
        kh, vh = k[:, h // (hq // hkv)].t().contiguous(), v[:, h // (hq // hkv)].contiguous()
        for t0 in range(0, T, block):
            t1 = min(T, t0 + block)
            s = (q[t0:t1, h] @ kh) * d ** -0.5
            seen = pos[None] <= first + torch.arange(t0, t1, device=q.device)[:, None]
            s.masked_fill_(~seen, -math.inf)
            out[t0:t1, h] = _softmax_rows(s) @ vh
    return out


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    half = HEAD_DIM // 2
    inv = ROPE_THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    ang = (pos.double()[:, None] * inv)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], dim=-1)


def _exact_model(case, seed):
    (embed, head, final, layers, adapters), cache, tokens, lens, rows, *_ = _model_inputs(case, seed)
    step = case["kind"] == "decode_step"
    if step:
        ids = _adapter_ids(case, seed, len(tokens)).tolist()
        if case["adapters"] == 1:
            ids = [0] * len(tokens)
        pos = torch.tensor([n - 1 for n in lens], device="cuda")
        row_of = list(range(len(tokens)))
    else:
        ids = [seed % case["adapters"]] * len(tokens)
        pos = torch.arange(lens[0] - len(tokens), lens[0], device="cuda")
        row_of = [0] * len(tokens)
    kv = cache.double()
    ids_t = torch.tensor(ids, device="cuda")
    page = torch.tensor([rows[r][p // PAGE] for r, p in zip(row_of, pos.tolist())], device="cuda")
    slot = pos % PAGE
    hidden = embed[tokens].double()
    for li, w in enumerate(layers):
        def project(x, m):
            y = x @ w[m].double().t()
            for a, ad in enumerate(adapters):
                A, B = ad[(li, m)]
                y += (ids_t == a).double()[:, None] * ((x @ A.double().t()) @ B.double().t()) * (ALPHA / RANK)
            return y

        x = _rms(hidden, w["input_norm"])
        q = _rope(_rms(project(x, "q").view(-1, 32, HEAD_DIM), w["q_norm"]), pos)
        kv[li, page, 0, slot] = _rope(_rms(project(x, "k").view(-1, 8, HEAD_DIM), w["k_norm"]), pos)
        kv[li, page, 1, slot] = project(x, "v").view(-1, 8, HEAD_DIM)
        attn = torch.empty_like(q)
        for r, n in enumerate(lens):
            own = kv[li][torch.tensor(rows[r], device="cuda")]
            k, v = (own[:, j].reshape(-1, 8, HEAD_DIM)[:n] for j in (0, 1))
            sel = slice(r, r + 1) if step else slice(None)
            attn[sel] = _attend(q[sel], k, v, int(pos[sel][0]))
        hidden = hidden + project(attn.reshape(-1, Q_DIM), "o")
        x = _rms(hidden, w["post_norm"])
        hidden = hidden + project(torch.nn.functional.silu(project(x, "gate")) * project(x, "up"), "down")
    if not step:
        hidden = hidden[-1:]
    return {"logits": _rms(hidden, final) @ head.double().t(), "kv": kv}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode_step", "prefill"):
        return _exact_model(case, seed)
    if kind == "lora_delta":
        base, groups, ids = _lora_inputs(case, seed)
        outs = []
        for x, mods in groups:
            ys = []
            for A, B, out, scale in mods:
                y = out.double()
                for a in range(case["adapters"]):
                    delta = (x.double() @ A[a].double().t()) @ B[a].double().t()
                    y += (ids == a).double()[:, None] * delta * scale
                ys.append(y)
            outs.append(torch.cat(ys, dim=1).reshape(-1))
        return torch.cat(outs)
    if kind == "linear":
        gen, dt = _gen(seed), _dtype(case)
        x = _normal(gen, (case["tokens"], case["in"]), dt)
        return x.double() @ _normal(gen, (case["out"], case["in"]), dt, 0.02).double().t()
    q, cache, lens, rows, *_ = _attention_inputs(case, seed)
    outs = []
    T = 1 if kind == "decode_attn" else case["tokens"]
    for r, n in enumerate(lens):
        own = cache[torch.tensor(rows[r], device="cuda")]
        k, v = (own[:, j].reshape(-1, *own.shape[3:])[:n].double() for j in (0, 1))
        outs.append(_attend(q[r * T:(r + 1) * T].double(), k, v, n - T))
    out = torch.cat(outs)
    return out.unsqueeze(2) if kind == "decode_attn" else out
