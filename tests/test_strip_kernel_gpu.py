"""The block_n 32 / 64 strip kernel (several tiles of one sequence per wave)
against the reference-structured per-tile kernel, which is bit-exact to the
oracle (tests/test_flash_gpu.py): m* and vrows equal, the output to the bf16
tolerance, for uniform, ragged and paged calls; and against the oracle.

Chunks are single waves' (any length) or workgroups' (four tiles and more);
lengths leave partial tiles, strips and chunks, and budgets run from none over
one sample per tile to more samples than rows.

Every case prints its name before touching the GPU.
"""
import numpy as np
import pytest
import torch

from helpers import SEED, bits16, flash_oracle_sequence, gen_qkv, h16_to_f32, seeded_lens, tol_check

pytestmark = pytest.mark.gpu


def _mod():
    import santa_flash_batch_cuda as m

    return m


def _same(a, b, is_bf16, what):
    for x, y, n in zip(a[1:], b[1:], ("m_star", "vrows")):
        np.testing.assert_array_equal(x.cpu().numpy(), y.cpu().numpy(), err_msg=f"{what} {n}")
    ok, mabs, mrel = tol_check(h16_to_f32(bits16(a[0]), is_bf16), h16_to_f32(bits16(b[0]), is_bf16))
    assert ok, (what, mabs, mrel)


@pytest.mark.parametrize("B,H,KVH,L,S,block_n,dtype", [
    # chunks of single waves: one tile (B = 3), three and more, partial strips
    (16, 32, 8, 1500, 256, 32, torch.bfloat16), (3, 64, 8, 1501, 256, 32, torch.bfloat16),
    (16, 32, 8, 3001, 512, 64, torch.bfloat16), (12, 64, 8, 2990, 100, 64, torch.float16),
    (24, 32, 8, 700, 47, 32, torch.float16), (16, 64, 8, 1472, 4000, 32, torch.bfloat16),
    (32, 32, 8, 1025, 5000, 64, torch.bfloat16), (16, 32, 8, 1409, 0, 32, torch.bfloat16),
    (3, 32, 8, 20001, 256, 32, torch.bfloat16), (2, 64, 8, 20010, 700, 64, torch.bfloat16),
    # chunks of workgroups: 5, 6 and 16 tiles over four waves
    (6, 32, 8, 1499, 256, 32, torch.bfloat16), (8, 32, 8, 2881, 512, 64, torch.float16),
    (40, 16, 4, 1501, 256, 32, torch.bfloat16), (30, 32, 4, 1100, 300, 32, torch.float16),
])
def test_uniform(B, H, KVH, L, S, block_n, dtype):
    m = _mod()
    print(f"\n[case] strips uniform B={B} H={H} KVH={KVH} L={L} S={S} block_n={block_n} {dtype}", flush=True)
    q, K, V = gen_qkv(B, H, KVH, L + 3, seed=SEED + L, dtype=dtype, lowrank=0.5)
    q, K, V = q.cuda(), K.cuda(), V.cuda()
    assert "strip" in m._tile_pass_kernel(B, H, KVH, -(-L // block_n), block_n)
    a = m.decode_systematic_batched(q, K, V, S, seed=SEED, block_n=block_n, want_vrows=True, valid_len=L)
    r = m._decode_reference_order(q, K, V, S, seed=SEED, block_n=block_n, want_vrows=True, valid_len=L)
    torch.cuda.synchronize()
    _same(a, r, dtype == torch.bfloat16, "uniform")
    if S == 0:
        assert not a[0].any()


@pytest.mark.parametrize("B,H,KVH,lo,hi,S,block_n", [
    (24, 32, 8, 1, 1500, 256, 0), (20, 64, 8, 300, 3000, 512, 0), (70, 32, 8, 200, 1000, 64, 32),
    (3, 64, 8, 200, 1500, 256, 0), (40, 16, 4, 200, 1500, 256, 0)])
def test_ragged_and_paged(B, H, KVH, lo, hi, S, block_n):
    """Every sequence against the reference-structured call on its length, the
    paged call bit for bit the ragged one, and two sequences against the oracle."""
    m = _mod()
    lens = seeded_lens(B, lo, hi, SEED + B)
    bn = block_n or (32 if max(lens) <= 1536 else 64)
    print(f"\n[case] strips ragged and paged B={B} H={H} KVH={KVH} lens {lo}..{hi} S={S} block_n={bn}", flush=True)
    qc, Kc, Vc = gen_qkv(B, H, KVH, max(lens), seed=SEED + B, lowrank=0.5)
    q, K, V = qc.cuda(), Kc.cuda(), Vc.cuda()
    a = m.decode_systematic_batched(q, K, V, S, seed=SEED, block_n=bn, want_vrows=True, valid_len=lens)
    torch.cuda.synchronize()
    for b in range(0, B, 5):
        r = m._decode_reference_order(q, K, V, S, seed=SEED, block_n=bn, want_vrows=True, valid_len=lens[b])
        torch.cuda.synchronize()
        _same([x[b] for x in a], [x[b] for x in r], True, f"b={b} len={lens[b]}")
    for b in (0, B - 1):
        exp = flash_oracle_sequence(qc, Kc, Vc, b, lens[b], S, bn)
        np.testing.assert_array_equal(a[1][b].cpu().numpy().view(np.uint32), exp["m_star"][0].view(np.uint32))
        np.testing.assert_array_equal(a[2][b].cpu().numpy(), exp["vrows"][0])
    page = 16
    used = [-(-l // page) for l in lens]
    order = torch.randperm(sum(used) + 2, generator=torch.Generator().manual_seed(SEED))
    table = torch.zeros(B, max(used), dtype=torch.int32)
    kp, vp = (torch.full((len(order), page, KVH, 128), float("nan"), device="cuda", dtype=torch.bfloat16)
              for _ in range(2))
    at = 0
    for b, n in enumerate(used):
        ids = order[at:at + n]
        at += n
        table[b, :n] = ids.int()
        for src, dst in ((K, kp), (V, vp)):
            rows = torch.full((n * page, KVH, 128), float("nan"), device="cuda", dtype=torch.bfloat16)
            rows[:lens[b]] = src[b, :lens[b]]
            dst[ids.cuda()] = rows.view(n, page, KVH, 128)
    p = m.decode_systematic_paged(q, kp, vp, table.cuda(), lens, S, seed=SEED, block_n=bn, want_vrows=True)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits16(a[0]), bits16(p[0]))
    for x, y in zip(a[1:], p[1:]):
        np.testing.assert_array_equal(x.cpu().numpy(), y.cpu().numpy())
