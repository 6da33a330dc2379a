"""The runtime's exact attention kernels against the same attention in plain
PyTorch float32.

Tolerance of the causal kernel: probabilities and output are rounded to the
16-bit type (relative 2^-9 in bf16, 2^-12 in f16) and the sums are float32, so
an element is off by at most half an ulp of itself plus the rounding of the
probabilities, which an output of |v| <= vmax scales to 2^-9 vmax (2^-12);
the float32 score sums over 128 products of magnitude <= 25 add
128 x 2^-24 x 25 = 2e-4 relative to every probability.

Every case prints its name before touching the GPU.
"""
import math

import pytest
import torch

from santa_amd.runtime import causal_attention

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
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
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
    cache = torch.full((B, P + 9, KVH, 128), float("nan"), device="cuda", dtype=torch.bfloat16)
    cache[:, :P] = k
    _check(causal_attention(q, cache[:, :P], v), want, v, torch.bfloat16)
    odd = torch.empty(B * P * H * 128 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(B, P, H, 128)
    odd.copy_(q)
    _check(causal_attention(odd, k, v), want, v, torch.bfloat16)
    _check(causal_attention(q.transpose(2, 3).contiguous().transpose(2, 3), k, v), want, v, torch.bfloat16)


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
    assert ((out.float() - ref).abs() <= 2.0 ** -9 * ref.abs() + (2.0 ** -9 + 1.3e-2) * v.float().abs().max()).all()


def test_causal_attention_keeps_autograd():
    """With gradients asked for, the torch expressions run and differentiate."""
    print("\n[case] causal attention under autograd", flush=True)
    q, k, v = (torch.randn(1, 40, h, 128, device="cuda", dtype=torch.bfloat16, requires_grad=True) for h in (4, 1, 1))
    causal_attention(q.float(), k.float(), v.float()).sum().backward()
    assert all(t.grad is not None and torch.isfinite(t.grad).all() for t in (q, k, v))
