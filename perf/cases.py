"""The calls this framework is timed on: one attention layer's decode step in
the forms a serving loop uses (one sequence and batches, one length and one
length per sequence, contiguous and paged caches, fixed and proportional
budgets), the causal attention of a prefill, and a model's prefill and decode
step.  Every case goes through the public entry points: the two extension
modules and ``santa_amd.runtime``.

Shapes are the repository's own (32q/8kv and 64q/8kv heads, 28q/4kv for a
group size outside the tuned kernels, head_dim 128, S = 256 or 512 for
santa_flash and one sample per 64 tokens for santa_prop, the
Llama-3.1-8B layer dimensions) or generic.
"""
import math
import random

import torch

D = 128
KINDS = ("flash", "flash_ragged", "flash_paged", "prop", "prop_ragged", "prop_batch", "attention", "prefill", "step")


def listed():
    return [
        # one user's short chat turn: the smallest call, launch and latency bound
        {"name": "flash_one_short", "kind": "flash", "B": 1, "H": 32, "KVH": 8, "L": 1500, "storage": 2048, "S": 256,
         "dtype": "bf16"},
        # a small batch in the middle of its generation: f16 cache larger than the odd valid length
        {"name": "flash_batch_odd_f16", "kind": "flash", "B": 5, "H": 32, "KVH": 8, "L": 9001, "storage": 12288,
         "S": 256, "dtype": "f16"},
        # the headline workload: batch 8 at 32k tokens
        {"name": "flash_batch_32k", "kind": "flash", "B": 8, "H": 32, "KVH": 8, "L": 32768, "storage": 32768,
         "S": 256, "dtype": "bf16"},
        # eight query heads per KV head at long context: the largest uniform call
        {"name": "flash_wide_64k", "kind": "flash", "B": 8, "H": 64, "KVH": 8, "L": 65536, "storage": 65536,
         "S": 512, "dtype": "bf16"},
        # continuous batching: every sequence at its own length, short and long together
        {"name": "flash_ragged", "kind": "flash_ragged", "B": 16, "H": 32, "KVH": 8, "lo": 1000, "hi": 40000,
         "S": 256, "dtype": "bf16", "lens": 16},
        # the same kind of batch over a page pool with 16-token pages
        {"name": "flash_paged", "kind": "flash_paged", "B": 8, "H": 32, "KVH": 8, "lo": 8000, "hi": 48000, "S": 256,
         "dtype": "bf16", "page": 16, "lens": 17},
        # santa_prop on one sequence through the reference's single-sequence call
        {"name": "prop_one_16k", "kind": "prop", "H": 32, "KVH": 8, "L": 16384, "S": 256, "dtype": "bf16"},
        # batched santa_prop, per-sequence lengths and budgets, long contexts: the most cache bytes
        {"name": "prop_ragged_long", "kind": "prop_ragged", "B": 16, "H": 32, "KVH": 8, "lo": 8192, "hi": 131072,
         "dtype": "bf16", "lens": 1690},
        # batched santa_prop at seven query heads per KV head
        {"name": "prop_gqa7_32k", "kind": "prop_batch", "B": 8, "H": 28, "KVH": 4, "L": 32768, "S": 512,
         "dtype": "bf16"},
        # the exact attention of a prefill, a few thousand prompt tokens
        {"name": "prefill_attention", "kind": "attention", "B": 2, "H": 32, "KVH": 8, "P": 4096, "dtype": "bf16"},
        # a prompt through a decoder layer and the head: logits of the last position and the filled caches
        {"name": "model_prefill", "kind": "prefill", "B": 1, "P": 3001, "layers": 1},
        # one teacher-forced decode step of the exact comparator: logits and the caches
        {"name": "model_step_exact", "kind": "step", "B": 4, "P": 4095, "layers": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16"))
    if kind == "flash":
        B = _log_int(rng, 1, 16)
        L = _log_int(rng, 300, min(131072, 524288 // B))
        return {"kind": kind, "B": B, "H": rng.choice((32, 32, 64)), "KVH": 8, "L": L,
                "storage": L + rng.choice((0, rng.randrange(1, 1024))), "S": rng.choice((128, 256, 512)),
                "dtype": dtype}
    if kind in ("flash_ragged", "flash_paged", "prop_ragged"):
        B = _log_int(rng, 2, 32)
        lo = _log_int(rng, 500, 8000)
        c = {"kind": kind, "B": B, "H": rng.choice((32, 32, 64)), "KVH": 8, "lo": lo,
             "hi": max(lo, min(int(lo * rng.uniform(2, 16)), 524288 // B)), "dtype": dtype,
             "lens": rng.randrange(1 << 30)}
        if kind != "prop_ragged":
            c["S"] = rng.choice((128, 256, 512))
        if kind == "flash_paged":
            c["page"] = rng.choice((16, 32, 64, 256))
        return c
    if kind == "prop":
        L = _log_int(rng, 1000, 65536)
        return {"kind": kind, "H": rng.choice((32, 32, 64)), "KVH": 8, "L": L, "S": max(32, L // 64), "dtype": dtype}
    if kind == "prop_batch":
        H, KVH = rng.choice(((28, 4), (40, 8), (32, 32), (16, 8)))
        B = _log_int(rng, 1, 8)
        L = _log_int(rng, 2000, min(32768, 1048576 // (B * KVH)))
        return {"kind": kind, "B": B, "H": H, "KVH": KVH, "L": L, "S": max(32, L // 64), "dtype": dtype}
    if kind == "attention":
        B = rng.choice((1, 1, 2, 4))
        H, KVH = rng.choice(((32, 8), (64, 8), (28, 4)))
        return {"kind": kind, "B": B, "H": H, "KVH": KVH, "P": _log_int(rng, 100, 4096 // B), "dtype": dtype}
    if kind == "prefill":
        B = rng.choice((1, 1, 2, 4))
        return {"kind": kind, "B": B, "P": _log_int(rng, 64, 3000 // B), "layers": 1}
    return {"kind": "step", "B": rng.randint(1, 8), "P": _log_int(rng, 300, 8000), "layers": rng.choice((1, 2))}


# ------------------------------------------------------------------- inputs
def _dtype(case):
    return torch.float16 if case.get("dtype") == "f16" else torch.bfloat16


def _lens(case):
    r = random.Random(case["lens"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["B"])]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _keys(g, n, KVH, dtype):
    """Keys [n, KVH, D] ~ N(0, 1) plus a rank-4 bias per KV head: scores with
    the spread of a trained model's rather than white noise."""
    K = torch.randn(n, KVH, D, generator=g, device="cuda")
    C = torch.randn(KVH, n, 4, generator=g, device="cuda")
    U = torch.randn(KVH, 4, D, generator=g, device="cuda") * 0.5
    K += torch.bmm(C, U).permute(1, 0, 2)
    return K.to(dtype)


def _cache(g, B, L, KVH, dtype):
    K = torch.stack([_keys(g, L, KVH, dtype) for _ in range(B)])
    V = torch.randn(B, L, KVH, D, generator=g, device="cuda", dtype=dtype)
    return K, V


def _shape(case):
    from santa_amd.runtime import LLAMA_3_1_8B as s, LlamaShape

    return LlamaShape(hidden=s.hidden, intermediate=s.intermediate, heads=s.heads, kv_heads=s.kv_heads,
                      layers=case["layers"], vocab=s.vocab)


def prepare(case, seed):
    kind, dtype = case["kind"], _dtype(case)
    g = _gen(seed)
    if kind in ("prefill", "step"):
        from santa_amd.runtime import ExactDecodeBackend, NHDCache, RandomLlama

        shape = _shape(case)
        B, P = case["B"], case["P"]
        st = {"kind": kind, "model": RandomLlama(shape, seed=seed, device="cuda")}
        st["cache"] = NHDCache(shape, B, P + 16, torch.bfloat16, "cuda")
        if kind == "prefill":
            st["tokens"] = torch.randint(0, shape.vocab, (B, P), generator=g, device="cuda")
            return st
        # the prompt's keys and values, with the spread the model's projections give them
        for t in st["cache"].k + st["cache"].v:
            t[:, :P].normal_(0.0, 1.25, generator=g)
        st["backend"] = ExactDecodeBackend()
        st["tokens"] = torch.randint(0, shape.vocab, (B,), generator=g, device="cuda")
        return st
    H, KVH = case["H"], case["KVH"]
    if kind == "attention":
        B, P = case["B"], case["P"]
        return {"kind": kind, **{n: torch.randn(B, P, h, D, generator=g, device="cuda", dtype=dtype)
                                 for n, h in (("q", H), ("k", KVH), ("v", KVH))}}
    if kind == "prop":
        K, V = _cache(g, 1, case["L"], KVH, dtype)
        return {"kind": kind, "q": torch.randn(H, D, generator=g, device="cuda", dtype=dtype), "K": K[0], "V": V[0],
                "S": case["S"], "seed": seed}
    B = case["B"]
    st = {"kind": kind, "q": torch.randn(B, H, D, generator=g, device="cuda", dtype=dtype), "seed": seed}
    if kind in ("flash", "prop_batch"):
        st["K"], st["V"] = _cache(g, B, case.get("storage", case["L"]), KVH, dtype)
        st["lens"] = case["L"]
        st["S"] = case["S"]
        return st
    st["lens"] = lens = _lens(case)
    st["S"] = case.get("S", [max(1, n // 64) for n in lens])
    if kind != "flash_paged":
        st["K"], st["V"] = _cache(g, B, max(lens), KVH, dtype)
        return st
    page = case["page"]
    used = [-(-n // page) for n in lens]
    pages = sum(used) + 7  # a pool never fits its sequences exactly
    K, V = _cache(g, 1, pages * page, KVH, dtype)
    st["K"], st["V"] = K.view(pages, page, KVH, D), V.view(pages, page, KVH, D)
    order = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)
    st["table"] = torch.zeros(B, max(used), dtype=torch.int32, device="cuda")
    at = 0
    for b, n in enumerate(used):
        st["table"][b, :n] = order[at:at + n]
        at += n
    return st


def run(state):
    kind = state["kind"]
    if kind in ("prefill", "step"):
        cache = state["cache"]
        if kind == "step":
            logits = state["model"].decode_step(state["tokens"], cache.storage - 16, cache, state["backend"])
        else:
            logits = state["model"].prefill(state["tokens"], cache)
        return {"logits": logits, "k": cache.k, "v": cache.v}
    if kind == "attention":
        from santa_amd.runtime import causal_attention

        return {"out": causal_attention(state["q"], state["k"], state["v"])}
    q, K, V, S, seed = state["q"], state["K"], state["V"], state["S"], state["seed"]
    if kind.startswith("flash"):
        import santa_flash_batch_cuda as m
    else:
        import santa_prop_batch_cuda as m
    if kind == "prop":
        out, m_star, _ = m.decode_systematic_scalar(q, K, V, S, seed=seed)
    elif kind == "flash_paged":
        out, m_star, _ = m.decode_systematic_paged(q, K, V, state["table"], state["lens"], S, seed=seed)
    else:
        out, m_star, _ = m.decode_systematic_batched(q, K, V, S, seed=seed, valid_len=state["lens"])
    return {"out": out, "m_star": m_star}


# --------------------------------------------------------------------- work
def _model_flops(shape, tokens):
    per = (shape.heads + 2 * shape.kv_heads) * D * shape.hidden + shape.heads * D * shape.hidden
    per += 3 * shape.hidden * shape.intermediate
    return 2.0 * per * shape.layers * tokens, 2.0 * per * shape.layers  # (flops, weight bytes)


def work(case):
    kind = case["kind"]
    if kind in ("prefill", "step"):
        s = _shape(case)
        B, P = case["B"], case["P"]
        tokens = B * P if kind == "prefill" else B
        flops, wbytes = _model_flops(s, tokens)
        head = 2.0 * s.vocab * s.hidden
        kv = 4.0 * B * P * s.kv_heads * D * s.layers
        pairs = B * P * (P + 1) / 2.0 if kind == "prefill" else B * (P + 1.0)
        flops += head * B + 4.0 * pairs * s.heads * D * s.layers
        return {"bytes": wbytes + head + kv + 2.0 * s.hidden * tokens + 4.0 * B * s.vocab, "flops": flops}
    H, KVH = case["H"], case["KVH"]
    if kind == "attention":
        B, P = case["B"], case["P"]
        return {"bytes": 2.0 * B * P * D * (2 * H + 2 * KVH), "flops": 4.0 * D * H * B * P * (P + 1) / 2.0}
    B = case.get("B", 1)
    lens = _lens(case) if "lens" in case else [case["L"]] * B
    rows = sum(lens)
    # the keys once, the sampled value rows once, q, out and m*
    sampled = sum(min(case["S"] if "S" in case else max(1, n // 64), n) for n in lens) * H
    return {"bytes": 2.0 * D * (rows * KVH + min(sampled, rows * KVH) + 2 * B * H) + 4.0 * B * H,
            "flops": 2.0 * D * (rows * H + sampled)}


def tolerance(case):
    """santa_flash's two merges (per chunk, and the reference's per tile)
    differ by up to 4.2e-5 in bf16 and 8.1e-6 in f16 (an occasional last-bit
    rounding; the sampled rows are the same).  The attention is 3.7e-3 from
    its 64-bit value, the model's logits 1.3e-2 (step) and 2.0e-2 (prefill):
    the roundings of every bf16 activation on the way to them."""
    if case["kind"] in ("prefill", "step"):
        return {"rel": 3e-2}
    if case["kind"] == "attention":
        return {"rel": 1.2e-2}
    return {"rel": 5e-4 if case["dtype"] == "bf16" else 1e-4}


# -------------------------------------------------------------------- exact
def _exact_max(q, K):
    """max over rows of K [n, KVH, D] of q [H, D] . K / sqrt(D), per head, in float64."""
    H, KVH = q.shape[0], K.shape[1]
    out = []
    for kv in range(KVH):
        qs = q[kv * (H // KVH):(kv + 1) * (H // KVH)].double().t().contiguous() / math.sqrt(D)
        out.append((K[:, kv].double().contiguous() @ qs).amax(0))
    return torch.cat(out)


def _exact_causal(q, k, v):
    """q [P, H, D], k, v [P, KVH, D], float64 in and out."""
    P, H = q.shape[:2]
    G = H // k.shape[1]
    out = torch.empty(P, H, D, dtype=torch.float64, device=q.device)
    for h in range(H):
        kt, vh = k[:, h // G].t().contiguous(), v[:, h // G].contiguous()
        for c in range(0, P, 2048):
            n = min(P, c + 2048)
            s = (q[c:n, h].contiguous() @ kt[:, :n].contiguous()) / math.sqrt(D)
            at = torch.arange(n, device=q.device)
            s.masked_fill_(at[None, :] > at[c:n, None], -math.inf)
            out[c:n, h] = torch.softmax(s, -1) @ vh[:n]
    return out


def _exact_rope(x, pos, theta):
    """x [n, heads, D] rotated by position pos[n]."""
    inv = theta ** (-torch.arange(0, D, 2, dtype=torch.float64, device=x.device) / D)
    a = torch.cat([pos.double()[:, None] * inv] * 2, -1)[:, None]
    half = torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1)
    return x * a.cos() + half * a.sin()


def _exact_norm(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _exact_model(case, seed):
    st = prepare(case, seed)
    m, cache, s, B, P = st["model"], st["cache"], _shape(case), case["B"], case["P"]
    step = case["kind"] == "step"
    rows = 1 if step else P
    pos = torch.arange(P, P + 1, device="cuda") if step else torch.arange(P, device="cuda")
    h = m.embed[st["tokens"]].double().view(B * rows, s.hidden)
    ks, vs = [t.double() for t in cache.k], [t.double() for t in cache.v]

    def times(x, w):
        return x @ w.double().t()

    for i, w in enumerate(m.layers):
        qkv = times(_exact_norm(h, w["ln1"], s.rms_eps), w["wqkv"]).view(B, rows, -1, D)
        a = torch.empty(B, rows, s.heads, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            q = _exact_rope(qkv[b, :, :s.heads], pos, s.rope_theta)
            k = _exact_rope(qkv[b, :, s.heads:s.heads + s.kv_heads], pos, s.rope_theta)
            ks[i][b, pos], vs[i][b, pos] = k, qkv[b, :, s.heads + s.kv_heads:]
            if not step:
                a[b] = _exact_causal(q, k, vs[i][b, :P])
                continue
            for kv in range(s.kv_heads):
                g = slice(kv * (s.heads // s.kv_heads), (kv + 1) * (s.heads // s.kv_heads))
                p = torch.softmax(q[0, g] @ ks[i][b, :P + 1, kv].t().contiguous() / math.sqrt(D), -1)
                a[b, 0, g] = p @ vs[i][b, :P + 1, kv].contiguous()
        h = h + times(a.view(B * rows, s.heads * D), w["wo"])
        x = _exact_norm(h, w["ln2"], s.rms_eps)
        gate, up = times(x, w["wgu"]).chunk(2, -1)
        h = h + times(torch.nn.functional.silu(gate) * up, w["wd"])
    last = _exact_norm(h.view(B, rows, -1)[:, -1], m.norm, s.rms_eps)
    return {"logits": times(last, m.lm_head), "k": ks, "v": vs}


def exact(case, seed):
    """The maximum score of every head (santa_flash and santa_prop: their
    sampled output has no 64-bit value), the attention and the model in
    float64."""
    with torch.inference_mode():
        if case["kind"] in ("prefill", "step"):
            return _exact_model(case, seed)
        st = prepare(case, seed)
        q, K = st["q"], st.get("K")
        if case["kind"] == "attention":
            return {"out": torch.stack([_exact_causal(q[b].double(), st["k"][b].double(), st["v"][b].double())
                                        for b in range(case["B"])])}
        if q.dim() == 2:
            return {"out": None, "m_star": _exact_max(q, K)}
        lens = st["lens"] if isinstance(st["lens"], list) else [st["lens"]] * case["B"]
        if "table" in st:
            rows = K.view(-1, *K.shape[2:])
            seqs = []
            for b, n in enumerate(lens):
                at = torch.arange(n, device="cuda")
                seqs.append(rows[st["table"][b, at // case["page"]].long() * case["page"] + at % case["page"]])
        else:
            seqs = [K[b, :n] for b, n in enumerate(lens)]
        return {"out": None, "m_star": torch.stack([_exact_max(q[b], k) for b, k in enumerate(seqs)])}
