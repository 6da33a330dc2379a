"""The model-level decode runtime on the GPU (bf16, a small Llama shape with
head_dim 128 and 4 query heads per KV head).

* The exact float32 decode backend agrees with recomputing the prefix with
  the prefill (bf16 model: tolerance on the logits).
* santa_flash with a budget of many samples per row approaches exact
  attention: its teacher-forced logits stay close to the exact ones and agree
  on the top token; santa_prop runs through the same loop.

Every case prints its name before touching the GPU.
"""
from dataclasses import replace

import pytest
import torch
import torch.nn.functional as F

from santa_amd import attention_backends as ab
from santa_amd.runtime import ExactDecodeBackend, LlamaShape, NHDCache, RandomLlama, decode_deviation, greedy_decode

pytestmark = pytest.mark.gpu

SMALL = LlamaShape(hidden=512, intermediate=1024, heads=4, kv_heads=1, layers=2, vocab=1000)


def _setup(P=700, B=2, seed=11):
    dev = torch.device("cuda:0")
    model = RandomLlama(SMALL, seed=seed, std=0.05, device=dev)
    toks = torch.randint(0, SMALL.vocab, (B, P + 8), generator=torch.Generator().manual_seed(seed)).to(dev)
    cache = NHDCache(SMALL, B, P + 16, torch.bfloat16, dev)
    logits = model.prefill(toks[:, :P], cache, attn_chunk=128)
    return model, toks, cache, logits


def test_exact_decode_matches_recomputation():
    print("\n[case] runtime exact decode vs prefill recomputation, P=700 B=2", flush=True)
    model, toks, cache, logits = _setup()
    res = greedy_decode(model, logits, 700, cache, ExactDecodeBackend(), 6, forced=toks[:, 700:706])
    torch.cuda.synchronize()
    for j in range(6):
        ref = model.prefill(toks[:, :700 + j], NHDCache(SMALL, 2, 720, torch.bfloat16, toks.device), attn_chunk=128)
        err = (res["logits"][j] - ref).abs().max().item()
        scale = ref.abs().max().item()
        assert err <= 0.05 * scale, (j, err, scale)


@pytest.mark.parametrize("B,P,mlp_chunk", [(1, 1, 8192), (2, 97, 40), (1, 300, 128)])
def test_fused_prefill_matches_torch_expressions(B, P, mlp_chunk, monkeypatch):
    """The prefill on the library's kernels against the torch expressions: the
    same roundings up to the order of float32 sums, so logits and caches agree
    to a few bf16 units (2^-8 each) of their scale through two layers."""
    print(f"\n[case] fused prefill B={B} P={P} mlp_chunk={mlp_chunk}", flush=True)
    dev = torch.device("cuda:0")
    model = RandomLlama(SMALL, seed=7, std=0.05, device=dev)
    toks = torch.randint(0, SMALL.vocab, (B, P), generator=torch.Generator().manual_seed(P)).to(dev)
    fused, plain = (NHDCache(SMALL, B, P + 2, torch.bfloat16, dev) for _ in range(2))
    got = model.prefill(toks, fused, mlp_chunk=mlp_chunk, attn_chunk=64)
    monkeypatch.setattr(RandomLlama, "_fused_prefill_takes", lambda self, h, cache: False)
    want = model.prefill(toks, plain, mlp_chunk=mlp_chunk, attn_chunk=64)
    torch.cuda.synchronize()
    for a, b in [(got, want)] + list(zip(fused.k + fused.v, plain.k + plain.v)):
        a, b = a.float(), b.float()
        assert (a - b).abs().max() <= 8 * 2.0 ** -8 * b.abs().max(), ((a - b).abs().max(), b.abs().max())
        assert (a - b).norm() <= 2.0 ** -6 * b.norm()
    assert not fused.k[0][:, P:].any() and not fused.v[1][:, P:].any()


def test_model_without_layers():
    """Embedding, final norm and head: the prefill's logits are the step's."""
    print("\n[case] prefill and step of a model without layers", flush=True)
    dev, shape = torch.device("cuda:0"), replace(SMALL, layers=0)
    model = RandomLlama(shape, seed=7, std=0.05, device=dev)
    toks = torch.randint(0, shape.vocab, (2, 5), generator=torch.Generator().manual_seed(9)).to(dev)
    cache = NHDCache(shape, 2, 8, torch.bfloat16, dev)
    got = model.prefill(toks, cache)
    torch.cuda.synchronize()
    h = model.embed[toks[:, -1]].float()
    want = F.linear((h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + shape.rms_eps)).bfloat16().float(),
                    model.lm_head.float())
    assert torch.equal(got, model.decode_step(toks[:, -1], 5, cache, ExactDecodeBackend()))
    # the norm's sum in another order can move its rounding by one bf16 unit
    assert (got - want).abs().max() <= 2.0 ** -7 * want.abs().max()


def test_prefill_into_stacked_caches():
    """Caches that are one tensor over the layers, cut from a wider one (rows
    not packed): the same K and V in their places, nothing beside them."""
    print("\n[case] prefill into stacked caches", flush=True)
    dev = torch.device("cuda:0")
    model = RandomLlama(SMALL, seed=7, std=0.05, device=dev)
    toks = torch.randint(0, SMALL.vocab, (2, 33), generator=torch.Generator().manual_seed(10)).to(dev)
    plain, stacked = (NHDCache(SMALL, 2, 40, torch.bfloat16, dev) for _ in range(2))
    want = model.prefill(toks, plain)
    wide = [torch.zeros(SMALL.layers, 2, 40, 3, 128, device=dev, dtype=torch.bfloat16) for _ in range(2)]
    stacked.k, stacked.v = wide[0][:, :, :, 1:2], wide[1][:, :, :, 1:2]
    got = model.prefill(toks, stacked)
    torch.cuda.synchronize()
    for a, b in [(got, want)] + list(zip([*stacked.k, *stacked.v], plain.k + plain.v)):
        a, b = a.float(), b.float()
        assert (a - b).abs().max() <= 8 * 2.0 ** -8 * b.abs().max()  # the torch expressions' roundings, two layers
    assert not any(w[:, :, :, i].any() for w in wide for i in (0, 2))


def test_prefill_and_step_under_autocast():
    """Autocast to float16, torch's default on a GPU: the prefill is the torch
    expressions under the same autocast, and a step of more sequences than the
    few-row product takes stays the step without autocast (its products beside
    that kernel are torch's)."""
    print("\n[case] prefill and a step of nine sequences under autocast", flush=True)
    dev = torch.device("cuda:0")
    model = RandomLlama(SMALL, seed=7, std=0.05, device=dev)
    toks = torch.randint(0, SMALL.vocab, (9, 20), generator=torch.Generator().manual_seed(8)).to(dev)
    cast, want, plain = (NHDCache(SMALL, 9, 22, torch.bfloat16, dev) for _ in range(3))
    ref = model.prefill(toks, plain)
    with torch.autocast("cuda"):
        got = model.prefill(toks, cast)
        with pytest.MonkeyPatch.context() as mp:
            mp.setattr(RandomLlama, "_fused_prefill_takes", lambda self, h, cache: False)
            torch_path = model.prefill(toks, want)
    torch.cuda.synchronize()
    for a, b, c in [(got, torch_path, ref)] + list(zip(cast.k + cast.v, want.k + want.v, plain.k + plain.v)):
        assert torch.equal(a, b)
        a, c = a.float(), c.float()
        # float16 products keep three bits more than bf16's: a few bf16 units apart through two layers
        assert (a - c).abs().max() <= 8 * 2.0 ** -8 * c.abs().max()
    nxt = torch.argmax(ref, -1)
    other = plain.clone()
    step = model.decode_step(nxt, 20, plain, ExactDecodeBackend())
    with torch.autocast("cuda"):
        same = model.decode_step(nxt, 20, other, _NoAutocast())
    torch.cuda.synchronize()
    assert torch.equal(step, same) and all(torch.equal(a, b) for a, b in zip(plain.k + plain.v, other.k + other.v))


class _NoAutocast(ExactDecodeBackend):
    """The exact backend outside the step's autocast (its torch form would be cast)."""

    def decode(self, *args):
        with torch.autocast("cuda", enabled=False):
            return super().decode(*args)


def test_santa_backends_in_the_decode_loop():
    print("\n[case] runtime santa_flash (large S) and santa_prop vs exact, P=700 B=2", flush=True)
    model, toks, cache, logits = _setup()
    exact = greedy_decode(model, logits, 700, cache.clone(), ExactDecodeBackend(), 6)
    flash = ab.SantaFlashBackend(S=64 * 32 * 32, seed=1690, block_n=None)
    res = greedy_decode(model, logits, 700, cache.clone(), flash, 6, forced=exact["tokens"])
    torch.cuda.synchronize()
    assert flash.actual_mode == "batch"
    dev = decode_deviation(res["logits"], exact["logits"])
    scale = exact["logits"].abs().max().item()
    assert max(dev["max_abs"]) <= 0.1 * scale, (dev, scale)
    assert min(dev["top1_agree"]) == 1.0, dev
    prop = ab.SantaPropBackend(S=700, seed=1690, block_n=None)
    res_p = greedy_decode(model, logits, 700, cache.clone(), prop, 6, forced=exact["tokens"])
    torch.cuda.synchronize()
    assert prop.actual_mode == "batch" and torch.isfinite(res_p["logits"]).all()


def test_peaky_attention_agrees_with_exact_at_cfg4_shape():
    """The model-level loop at cfg4's attention shape (hidden 4096, 32q/8kv,
    d=128, B=4, 32768-token prompts, santa_flash S=256: T_c=129, S_per_tile=1)
    with two layers.  With the random model's nearly uniform attention over
    32k keys the S=256 estimate is noise; scaling the query projection (a
    trained model's peaky attention) makes the sampled decode agree with the
    exact one, and the agreement grows with the sharpness."""
    from santa_amd.runtime import LLAMA_3_1_8B, LlamaShape

    s = LLAMA_3_1_8B
    shape = LlamaShape(hidden=s.hidden, intermediate=s.intermediate, heads=s.heads, kv_heads=s.kv_heads, layers=2,
                       vocab=s.vocab)
    B, P, steps = 4, 32768, 6
    dev = torch.device("cuda:0")
    prompt = torch.randint(0, shape.vocab, (B, P), generator=torch.Generator().manual_seed(1690)).to(dev)
    stats = {}
    for scale in (1.0, 32.0):
        print(f"\n[case] cfg4 attention shape, 2 layers, B={B} P={P}, score_scale={scale}", flush=True)
        model = RandomLlama(shape, seed=1690, device=dev, score_scale=scale)
        cache = NHDCache(shape, B, P + steps, torch.bfloat16, dev)
        logits0 = model.prefill(prompt, cache)
        exact = greedy_decode(model, logits0, P, cache.clone(), ExactDecodeBackend(), steps)
        flash = ab.SantaFlashBackend(S=256, seed=1690, block_n=None)
        res = greedy_decode(model, logits0, P, cache, flash, steps, forced=exact["tokens"])
        torch.cuda.synchronize()
        assert flash.actual_mode == "batch"
        d = decode_deviation(res["logits"], exact["logits"])
        stats[scale] = (sum(d["mean_rel"]) / steps, sum(d["top1_agree"]) / steps)
        del model, cache
        torch.cuda.empty_cache()
    print(stats, flush=True)
    assert stats[32.0][0] <= 0.1 and stats[32.0][1] >= 0.8, stats
    assert stats[32.0][0] < 0.2 * stats[1.0][0], stats
