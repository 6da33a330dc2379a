"""Which calls of the runtime go to the library's kernels, and how they are
launched, on the CPU: the library is replaced by a recorder, so nothing here
needs a GPU.
"""
import contextlib
import ctypes

import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.flop_counter import FlopCounterMode

from santa_amd import runtime
from santa_amd.runtime import LlamaShape, NHDCache, _FusedOps, _plain

BF = torch.bfloat16


class _Recorder:
    """A library whose functions only note their arguments and the device that is current."""

    def __init__(self, current):
        self.current, self.calls = current, []

    def __getattr__(self, name):
        def fn(*args):
            self.calls.append((name, self.current[-1], args))
            return 0

        return fn


@pytest.fixture
def recorder(monkeypatch):
    current = ["another device"]

    @contextlib.contextmanager
    def device(d):
        current.append(d)
        yield
        current.pop()

    class stream:
        cuda_stream = 0  # a device's default stream: the current device's null stream to the runtime

    rec = _Recorder(current)
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)  # a CPU tensor's get_device() is -1
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: stream)
    monkeypatch.setattr(_FusedOps, "_lib", rec)
    return rec


def _ops():
    x, w = torch.ones(2, 64, dtype=BF), torch.ones(48, 64, dtype=BF)
    qkv, cs = torch.ones(1, 2, 64, dtype=BF), torch.ones(2, 16, dtype=BF)
    cache = NHDCache(LlamaShape(hidden=32, intermediate=8, heads=2, kv_heads=1, layers=1, vocab=8), 1, 4, BF, "cpu")
    kv = torch.ones(1, 4, 1, 128, dtype=BF)
    q = torch.ones(1, 4, 2, 128, dtype=BF)
    return {
        "add_rms_norm": lambda: _FusedOps.add_rms_norm(x, x.clone(), x[0], 1e-5),
        "rope_table": lambda: _FusedOps.rope_table(3, 16, 1e4, x),
        "rope_write": lambda: _FusedOps.rope_write(qkv[0, :1], cs[0], cs[0], cache, 0, 1, 2, 1, 16),
        "rope_write_rows": lambda: _FusedOps.rope_write_rows(qkv, cs, cs, cache.k[0], cache.v[0], 2, 1, 16),
        "linear": lambda: _FusedOps.linear(x, w),
        "linear_f32": lambda: _FusedOps.logits(x, w),
        "linear_rope": lambda: _FusedOps.linear_rope(x[:1], torch.ones(64, 64, dtype=BF), cs[0], cs[0], cache, 0, 1, 2,
                                                     1, 16),
        "argmax": lambda: _FusedOps.argmax(x.float()),
        "silu_mul": lambda: _FusedOps.silu_mul(x),
        "causal_attention": lambda: _FusedOps.causal_attention(q, kv, kv),
        "exact_decode": lambda: _FusedOps.exact_decode(q[:, 0], kv, kv, 3),
    }


@pytest.mark.parametrize("op", sorted(_ops()))
def test_launches_on_the_tensors_device(op, recorder):
    """Every kernel is launched with its tensors' device current: a default
    stream is 0, which the runtime takes as the current device's."""
    _ops()[op]()
    launches = [c for c in recorder.calls if not c[0].endswith("workspace_size")]
    assert [c[0] for c in launches] == ["santa_rt_" + op]
    assert launches[0][1] == torch.device("cpu")


def _operands():
    """(name, k of shape [B, P, heads, 128]): layouts the kernels cannot address
    as they are, or only because a stride belongs to a dimension of size 1."""
    one_head = torch.randn(1, 5, 128, 1, dtype=BF).transpose(2, 3)  # head stride 1
    packed = torch.randn(3, 5 * 2 * 128 + 4, dtype=BF)[:, :5 * 2 * 128].view(3, 5, 2, 128)[:1]  # batch stride 1284
    row = torch.randn(2, 3, 2 * 128 + 4, dtype=BF)[..., :256].view(2, 3, 2, 128)[:1, :1]  # 780, 260
    far = torch.randn(128, dtype=BF).as_strided((1, 1, 1, 128), (3, 1 << 25, 5, 1))  # a position stride above the limit
    swapped = torch.randn(2, 5, 128, 2, dtype=BF).transpose(2, 3)  # last dimension not contiguous
    ragged = torch.randn(2, 5 * 2 * 128 + 4, dtype=BF)[:, :5 * 2 * 128].view(2, 5, 2, 128)  # batch stride 1284, B 2
    odd = torch.randn(5 * 2 * 128 + 1, dtype=BF)[1:].view(1, 5, 2, 128)  # 2 bytes off
    expanded = torch.randn(1, 5, 1, 128, dtype=BF).expand(2, 5, 3, 128)
    same = torch.randn(2, 1, 3, 128, dtype=BF).expand(2, 5, 3, 128)  # one position for all
    return {"one head": one_head, "packed batch of one": packed, "single row": row, "far position": far,
            "swapped": swapped, "ragged batch": ragged, "odd address": odd, "expanded": expanded,
            "same positions": same}


def _rows(ptr, shape, strides):
    """The 256-byte rows [B, P, heads] of a 16-bit tensor at ptr."""
    return [ctypes.string_at(ptr + 2 * (b * strides[0] + p * strides[1] + h * strides[2]), 256)
            for b in range(shape[0]) for p in range(shape[1]) for h in range(shape[2])]


@pytest.mark.parametrize("name", sorted(_operands()))
def test_attention_operands_fit_the_kernels(name, recorder):
    """Whatever the layout, the strides and the address passed on are ones the
    kernels take (multiples of 8 elements, positions at least a row apart and
    below 2^24, 16-byte aligned) and lead to the same values."""
    k = _operands()[name]
    B, P, KVH, D = k.shape
    q = torch.randn(B, P, 2 * KVH, D, dtype=BF)
    dense = torch.empty(k.shape, dtype=BF).copy_(k)
    want = _rows(dense.data_ptr(), k.shape, (P * KVH * D, KVH * D, D))

    def check(ptr, strides):
        assert ptr % 16 == 0 and all(s >= 0 and s % 8 == 0 for s in strides) and 128 <= strides[1] < 1 << 24
        assert _rows(ptr, k.shape, strides) == want
        return 0

    recorder.santa_rt_causal_attention = lambda *a: check(a[1], a[10][3:6]) or check(a[2], a[10][6:9])
    recorder.santa_rt_exact_decode = lambda *a: check(a[1], a[10][:3]) or check(a[2], a[10][3:6])
    _FusedOps.causal_attention(q, k, k)
    _FusedOps.exact_decode(q[:, 0], k, k, P)


@contextlib.contextmanager
def _autocast(dtype):
    """torch.autocast("cuda", dtype) without a GPU, where it switches itself off."""
    kept = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    torch.set_autocast_enabled("cuda", True)
    torch.set_autocast_dtype("cuda", dtype)
    try:
        yield
    finally:
        torch.set_autocast_enabled("cuda", kept[0])
        torch.set_autocast_dtype("cuda", kept[1])


def test_autocast_to_another_type_is_not_plain():
    """Under autocast the torch products change type; a kernel's operands would not."""
    t = torch.ones(2, dtype=BF)
    assert _plain(t)
    with _autocast(torch.float16):
        assert not _plain(t) and _plain(t.half()) and not _plain(t.half(), t)
    with _autocast(BF):
        assert _plain(t) and not _plain(t.half())


@pytest.mark.parametrize("op", ["add_rms_norm", "rope_write", "rope_write_rows", "silu_mul"])
def test_kernels_refuse_another_type(op, recorder):
    """float16 bits are never read as bf16."""
    x, cs = torch.ones(2, 64, dtype=BF), torch.ones(2, 16, dtype=BF)
    cache = NHDCache(LlamaShape(hidden=32, intermediate=8, heads=2, kv_heads=1, layers=1, vocab=8), 1, 4, BF, "cpu")
    with pytest.raises(AssertionError):
        if op == "add_rms_norm":
            _FusedOps.add_rms_norm(x, x.half(), x[0], 1e-5)
        elif op == "rope_write":
            _FusedOps.rope_write(x[:1].half(), cs[0], cs[0], cache, 0, 1, 2, 1, 16)
        elif op == "rope_write_rows":
            _FusedOps.rope_write_rows(x[None].half(), cs, cs, cache.k[0], cache.v[0], 2, 1, 16)
        else:
            _FusedOps.silu_mul(x.half())
    assert not recorder.calls


def test_only_ordinary_calls_are_plain():
    """What a kernel behind raw pointers would drop or hide: gradients, tangents,
    transforms, and operations recorded by a dispatch mode."""
    t = torch.ones(2, 3, dtype=BF)
    leaf = t.clone().requires_grad_()
    assert _plain(t) and not _plain(t, leaf)
    with torch.no_grad():
        assert _plain(leaf)
    with fwAD.dual_level():
        dual = fwAD.make_dual(t, t)
        assert _plain(t) and not _plain(dual)
    seen = []
    torch.vmap(lambda x: seen.append(_plain(x)) or x)(t)
    torch.func.jvp(lambda x: seen.append(_plain(x)) or x, (t,), (t,))
    make_fx(lambda x: seen.append(_plain(x)) or x * 2)(t)  # records what is run on ordinary tensors
    with FakeTensorMode():
        seen.append(_plain(torch.empty(2, dtype=BF)))
    with FlopCounterMode(display=False):
        seen.append(_plain(t))
    assert seen == [False] * 5 and _plain(t)
