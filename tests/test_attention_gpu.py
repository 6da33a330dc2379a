"""The runtime's exact attention kernels against the same attention in plain
PyTorch float32.

Tolerance of the causal kernel: probabilities and output are rounded to the
16-bit type and the sums are float32.  Rounding to a p-bit significand is off by
at most half an ulp, 2^-p of the value (p = 8 in bf16, 11 in f16).  So an
element is off by at most 2^-p of itself plus the rounding of the
probabilities, which an output of |v| <= vmax scales to 2^-p vmax;
the float32 score sums over 128 products of magnitude <= 25 add
128 x 2^-24 x 25 = 2e-4 relative to every probability.

Every case prints its name before touching the GPU.
"""
import math

import pytest
import torch

from santa_amd.runtime import ExactDecodeBackend, causal_attention

pytestmark = pytest.mark.gpu


def _ref(q, k, v):
    """float32 causal attention, head by head."""
    B, P, H, D = q.shape
    G = H // k.shape[2]
    out = torch.empty(B, P, H, D, device=q.device)
    mask = torch.arange(P, device=q.device)[None, :] > torch.arange(P, device=q.device)[:, None]
    for b in range(B):
        for h in range(H):
            s = (q[b, :, h].float().contiguous() @ k[b, :, h // G].float().t().contiguous()) / math.sqrt(D)
            out[b, :, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[b, :, h // G].float().contiguous()
    return out


def _check(out, ref, v, dtype):
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    vmax = v.float().abs().max().item()
    bound = eps * ref.abs() + (eps + 2e-4) * vmax
    err = (out.float() - ref).abs()
    assert torch.isfinite(out).all() and (err <= bound).all(), (err / bound).max().item()


# position counts around the 32-row units and 64-key tiles; group sizes that
# fill a workgroup's waves, leave some idle and split over position blocks
@pytest.mark.parametrize("B,P,H,KVH,dtype", [
    (1, 1, 4, 1, torch.bfloat16), (1, 31, 8, 8, torch.bfloat16), (2, 32, 4, 2, torch.float16),
    (1, 33, 7, 1, torch.bfloat16), (1, 64, 16, 2, torch.bfloat16), (3, 65, 6, 2, torch.float16),
    (1, 127, 5, 1, torch.bfloat16), (2, 128, 8, 2, torch.bfloat16), (1, 129, 32, 8, torch.float16),
    (1, 700, 12, 4, torch.bfloat16), (2, 1025, 8, 1, torch.bfloat16), (1, 2048, 9, 3, torch.float16),
])
def test_causal_attention(B, P, H, KVH, dtype):
    print(f"\n[case] causal attention B={B} P={P} H={H} KVH={KVH} {dtype}", flush=True)
    g = torch.Generator().manual_seed(P)
    q, k, v = (torch.randn(B, P, h, 128, generator=g).mul(1.5).to("cuda", dtype) for h in (H, KVH, KVH))
    _check(causal_attention(q, k, v), _ref(q, k, v), v, dtype)


def test_causal_attention_strided():
    """Slices of a fused projection and of a cache, and a q that has to be copied."""
    print("\n[case] causal attention on strided operands", flush=True)
    g = torch.Generator().manual_seed(3)
    B, P, H, KVH = 2, 150, 8, 2
    qkv = torch.randn(B, P, H + 2 * KVH, 128, generator=g).to("cuda", torch.bfloat16)
    q, k, v = qkv.split([H, KVH, KVH], dim=2)
    want = _ref(q, k, v)
    _check(causal_attention(q, k, v), want, v, torch.bfloat16)
    # the prompt's part of caches whose tails hold anything: a V row read past
    # the end would show (0 * NaN), a K row only where its score is not masked
    ck, cv = (torch.full((B, P + 9, KVH, 128), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ck[:, :P], cv[:, :P] = k, v
    _check(causal_attention(q, ck[:, :P], cv[:, :P]), want, v, torch.bfloat16)
    odd = torch.empty(B * P * H * 128 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(B, P, H, 128)
    odd.copy_(q)
    _check(causal_attention(odd, k, v), want, v, torch.bfloat16)
    _check(causal_attention(q.transpose(2, 3).contiguous().transpose(2, 3), k, v), want, v, torch.bfloat16)


def test_attention_size_one_dimensions():
    """Strides of size-1 dimensions that are no multiple of 8, which torch
    leaves as they are in a tensor that counts as contiguous: one KV head with
    head stride 1, a batch of one cut from wider rows, a single position; and
    one position repeated, whose infinite values must not reach the rows past
    the end."""
    print("\n[case] attention on size-1 dimensions of odd strides", flush=True)
    g = torch.Generator().manual_seed(6)
    P, bf = 70, torch.bfloat16
    one_head = torch.randn(1, P, 128, 1, generator=g).to("cuda", bf).transpose(2, 3)
    packed = torch.randn(2, P * 256 + 4, generator=g).to("cuda", bf)[:, :P * 256].view(2, P, 2, 128)[:1]
    for k in (one_head, packed, packed[:, :1]):
        n, KVH = k.shape[1:3]
        q = torch.randn(1, n, 4 * KVH, 128, generator=g).to("cuda", bf)
        _check(causal_attention(q, k, k), _ref(q, k, k), k, bf)
        _check_decode(ExactDecodeBackend().decode(q[:, -1], k, k, n), _ref_decode(q[:, -1], k, k, n), k, bf)
    same = torch.randn(1, 1, 1, 128, generator=g).to("cuda", bf)
    same[..., 7] = math.inf
    k, v = torch.zeros(1, 9, 1, 128, device="cuda", dtype=bf), same.expand(1, 9, 1, 128)
    assert torch.equal(ExactDecodeBackend().decode(k[:, 0], k, v, 9)[0, 0].isinf(), same[0, 0, 0].isinf())


def test_causal_attention_large_scores():
    """Scores of several hundred, growing with the position: the running
    maximum moves in every tile and the early sums are rescaled to nothing."""
    print("\n[case] causal attention, large growing scores", flush=True)
    P = 300
    g = torch.Generator().manual_seed(4)
    q = torch.ones(1, P, 4, 128)
    k = torch.randn(1, P, 1, 128, generator=g) * 0.1 + torch.arange(P).view(1, P, 1, 1) * 0.25
    v = torch.randn(1, P, 1, 128, generator=g)
    q, k, v = (t.to("cuda", torch.bfloat16) for t in (q, k, v))
    out, ref = causal_attention(q, k, v), _ref(q, k, v)
    # scores up to 850 carry 128 x 2^-24 x 850 = 6.5e-3 of absolute rounding
    assert ((out.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + (2.0 ** -8 + 1.3e-2) * v.float().abs().max()).all()


def test_attention_minus_infinite_scores():
    """Keys masked through K, more of them than a tile, a step and a chunk
    hold, before the first one that counts: they weigh nothing, and a query
    with no other key is NaN, as in torch's softmax."""
    print("\n[case] attention, the first 100 keys at -inf", flush=True)
    g = torch.Generator().manual_seed(7)
    P, n, bf = 300, 100, torch.bfloat16
    q, k, v = (torch.randn(1, P, h, 128, generator=g) for h in (4, 1, 1))
    q[..., 5], k[:, :n, :, 5] = 1.0, -math.inf
    q, k, v = (t.to("cuda", bf) for t in (q, k, v))
    out = causal_attention(q, k, v)
    assert out[:, :n].isnan().all()
    _check(out[:, n:], _ref(q, k, v)[:, n:], v, bf)
    for L in (n + 1, P):
        _check_decode(ExactDecodeBackend().decode(q[:, -1], k, v, L), _ref_decode(q[:, -1], k, v, L), v, bf)
    assert ExactDecodeBackend().decode(q[:, -1], k, v, n).isnan().all()


def test_attention_huge_scores():
    """Scores of 1e12 to 1e16 (finite in float32), 1e13 and more apart: every
    query attends to its best key alone."""
    print("\n[case] attention, scores up to 1e16", flush=True)
    g = torch.Generator().manual_seed(8)
    P, bf = 300, torch.bfloat16
    # float32 products of integers below 2^8 and 2^20 sum to the same value for equal keys only
    level = torch.randperm(P, generator=g).float() + 1.0
    q = torch.full((1, P, 4, 128), 2.0 ** 20)
    k = (level * 2.0 ** 18).view(1, P, 1, 1).expand(1, P, 1, 128).contiguous()
    v = torch.randn(1, P, 1, 128, generator=g)
    q, k, v = (t.to("cuda", bf) for t in (q, k, v))
    best = torch.cummax(k[0, :, 0, 0].float(), 0)
    keep = (k[0, :, 0, 0][None, :] == best.values[:, None]).sum(1)  # bf16 rounds some levels together
    out = causal_attention(q, k, v)
    _check(out, _ref(q, k, v), v, bf)
    one = keep == 1
    assert one.sum() > 0 and torch.equal(out[0, one], v[0, best.indices[one]].expand(-1, 4, 128))
    for L in (40, 65, P):
        _check_decode(ExactDecodeBackend().decode(q[:, -1], k, v, L), _ref_decode(q[:, -1], k, v, L), v, bf)


def test_attention_keeps_autograd():
    """With gradients asked for of tensors the kernels would take, the torch
    expressions run: the outputs are differentiable.  The causal attention's
    backward is not run in bf16 (its batched products would have transposed
    right operands); the same expressions differentiate in float32."""
    print("\n[case] attention under autograd", flush=True)
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(1, 40, h, 128, generator=g).to("cuda", torch.bfloat16).requires_grad_() for h in (4, 1, 1))
    with torch.no_grad():
        kernel = causal_attention(q, k, v)
    out = causal_attention(q, k, v)
    assert out.grad_fn is not None and kernel.grad_fn is None
    # the kernel's tolerance for both, and the torch path's scores rounded to bf16: |q . k| < 64 here,
    # so off by 64 x 2^-9 before the scale of 128^-1/2
    eps, vmax = 2.0 ** -8, v.detach().float().abs().max()
    assert ((out - kernel).float().abs() <= 2 * (2 * eps + 2e-4 + 64 * 2.0 ** -9 / math.sqrt(128)) * vmax).all()
    causal_attention(q.float(), k.float(), v.float()).sum().backward()
    assert all(t.grad is not None and torch.isfinite(t.grad).all() for t in (q, k, v))

    leaves = [t.detach().clone().requires_grad_() for t in (q[:, -1], k, v)]
    w = torch.randn(1, 4, 128, generator=g).to("cuda", torch.bfloat16)
    dec = ExactDecodeBackend().decode(*leaves, 33)
    assert dec.grad_fn is not None
    (dec * w).float().sum().backward()
    d = [t.detach().double().cpu().requires_grad_() for t in leaves]
    p = torch.softmax(torch.einsum("hd,ld->hl", d[0][0], d[1][0, :33, 0]) / math.sqrt(128), -1)
    ((p @ d[2][0, :33, 0]) * w[0].double().cpu()).sum().backward()
    for got, want in zip(leaves, d):
        # the gradient in bf16 of a bf16 output: one rounding of each, float32 between
        assert (got.grad.double().cpu() - want.grad).norm() <= 2.0 ** -7 * want.grad.norm()


def test_attention_many_short_sequences():
    """More workgroups than one launch holds threads for (2^32): one position
    each, so the output is v."""
    B = (1 << 24) + 3
    print(f"\n[case] attention of {B} sequences of one position", flush=True)
    q, k, v = (torch.randn(B, 1, 1, 128, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    assert torch.equal(causal_attention(q, k, v), v)
    assert torch.equal(ExactDecodeBackend().decode(q[:, 0], k, v, 1), v[:, 0])


def test_attention_on_a_stream_of_its_own():
    """The kernels run on the current stream, behind what that stream wrote."""
    print("\n[case] attention on a side stream", flush=True)
    g = torch.Generator().manual_seed(10)
    q, k, v = (torch.randn(2, 200, h, 128, generator=g).to("cuda", torch.bfloat16) for h in (8, 2, 2))
    want, wantd = causal_attention(q, k, v), ExactDecodeBackend().decode(q[:, -1], k, v, 200)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        x = torch.randn(4096, 4096, device="cuda")
        for _ in range(8):  # work in front, so that a launch elsewhere would come too early
            x = x @ x * 1e-2
        k2 = torch.zeros_like(k) + x[:1, :1].to(k.dtype).nan_to_num(0.0) * 0 + k
        got, gotd = causal_attention(q, k2, v), ExactDecodeBackend().decode(q[:, -1], k2, v, 200)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want) and torch.equal(gotd, wantd)


def _ref_decode(q, k, v, L):
    """float64 decode attention, head by head."""
    B, H, D = q.shape
    G = H // k.shape[2]
    out = torch.empty(B, H, D, device=q.device, dtype=torch.float64)
    for b in range(B):
        for h in range(H):
            s = k[b, :L, h // G].double().contiguous() @ q[b, h].double() / math.sqrt(D)
            out[b, h] = torch.softmax(s, 0) @ v[b, :L, h // G].double().contiguous()
    return out


def _check_decode(out, ref, v, dtype):
    # the output's own rounding (2^-p, as above), and float32 throughout: scores of magnitude
    # <= 25 over 128 products carry 2e-4 relative into every probability
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = eps * ref.abs() + 2e-4 * v.double().abs().max()
    err = (out.double() - ref).abs()
    assert torch.isfinite(out).all() and (err <= bound).all(), (err / bound).max().item()


# lengths around the 32-position steps and 64-position chunks, one chunk and
# many; every group-size form, idle head slots, two head groups, item counts
# that do not fill a workgroup
@pytest.mark.parametrize("B,L,H,KVH,dtype", [
    (1, 1, 8, 2, torch.bfloat16), (2, 31, 4, 4, torch.float16), (1, 32, 2, 1, torch.bfloat16),
    (3, 33, 6, 2, torch.bfloat16), (1, 63, 8, 1, torch.float16), (1, 64, 32, 8, torch.bfloat16),
    (2, 65, 10, 2, torch.bfloat16), (1, 97, 16, 1, torch.bfloat16), (1, 700, 24, 2, torch.float16),
    (1, 20000, 4, 1, torch.bfloat16), (5, 2049, 7, 1, torch.bfloat16), (8, 3000, 32, 8, torch.float16),
    (1, 40001, 4, 4, torch.bfloat16),
])
def test_exact_decode(B, L, H, KVH, dtype):
    print(f"\n[case] exact decode B={B} L={L} H={H} KVH={KVH} {dtype}", flush=True)
    g = torch.Generator().manual_seed(L)
    q = torch.randn(B, H, 128, generator=g).mul(1.5).to("cuda", dtype)
    k, v = (torch.randn(B, L + 5, KVH, 128, generator=g).to("cuda", dtype) for _ in range(2))
    k[:, L:] = float("nan")  # past the valid length: never read into the result
    v[:, L:] = float("nan")
    _check_decode(ExactDecodeBackend().decode(q, k, v, L), _ref_decode(q, k, v, L), v[:, :L], dtype)


def test_exact_decode_growing_scores_and_strides():
    """Scores growing with the position (the maximum moves every step) over
    caches that are slices of one tensor."""
    print("\n[case] exact decode, growing scores, strided caches", flush=True)
    g = torch.Generator().manual_seed(5)
    L = 500
    kv = torch.randn(2, L, 4, 128, generator=g)
    kv[:, :, :2] = 0.1 * kv[:, :, :2] + torch.arange(L).view(1, L, 1, 1) * 0.02
    kv = kv.to("cuda", torch.bfloat16)
    k, v = kv[:, :, :2], kv[:, :, 2:]
    q = torch.ones(2, 8, 128, device="cuda", dtype=torch.bfloat16)
    ref = _ref_decode(q, k, v, L)
    out = ExactDecodeBackend().decode(q, k, v, L)
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-3 * v.double().abs().max()).all()
